// Native check that slot_voxel and axis_slots (pyvr_amd/csrc/hvr_rules.h) are
// inverses: every slot axis_slots names for a voxel holds that voxel by
// slot_voxel, and every slot of texels 0 .. s + 1 is named once.
#include <stdio.h>

#include <vector>

#include "hvr_rules.h"

using namespace hvr;

int main()
{
    for (int lb = 2; lb <= 4; ++lb)
        for (int s = 1; s <= 150; ++s) {
            const uint32_t nb = bricks_along(s, lb), B = 1u << lb, E = B + 1u;
            std::vector<int> named((size_t)nb * E, 0);
            for (int c = 0; c < s; ++c) {
                uint32_t br[4], lo[4];
                const int n = axis_slots(c, s, lb, nb, br, lo);
                for (int k = 0; k < n; ++k) {
                    const uint32_t X = br[k] * B + lo[k];
                    ++named[br[k] * E + lo[k]];
                    if (X > (uint32_t)s + 1u || slot_voxel(X, s) != c) {
                        fprintf(stderr, "FAIL s=%d lb=%d voxel %d texel %u\n", s, lb, c, X);
                        return 1;
                    }
                }
            }
            for (uint32_t b = 0; b < nb; ++b)
                for (uint32_t l = 0; l <= B; ++l)
                    if (named[b * E + l] != (b * B + l <= (uint32_t)s + 1u ? 1 : 0)) {
                        fprintf(stderr, "FAIL s=%d lb=%d slot (%u, %u) named %d times\n", s, lb, b, l, named[b * E + l]);
                        return 1;
                    }
        }
    printf("slots ok\n");
    return 0;
}
