// Native check of the groups an upload is split into (upload_group,
// source_begin, source_end and slot_extent in pyvr_amd/csrc/hvr_rules.h): over
// axes of 1 to 300 voxels, brick edges 4 to 16 and staging bounds from less than a
// row to more than the field, every group's source holds the voxel of each of
// its bricks' slots, fits the bytes the rule names, and those fit the bound
// unless the group is one row of bricks.  Exit status 0 on success.
#include <stdint.h>
#include <stdio.h>

#include <algorithm>

#include "hvr_rules.h"

using namespace hvr;

static uint64_t g_state = 0x2545f4914f6cdd1dull;
static uint64_t rnd()
{
    g_state ^= g_state << 13;
    g_state ^= g_state >> 7;
    g_state ^= g_state << 17;
    return g_state >> 11;
}

#define CHECK(cond)                                                                                          \
    do {                                                                                                     \
        if (!(cond)) {                                                                                       \
            fprintf(stderr, "FAIL %s: s1=%d s2=%d lb=%d row=%llu max=%llu layers=%u rows=%u bytes=%llu\n", #cond, s1, s2, \
                    lb, (unsigned long long)row, (unsigned long long)max, g.layers, g.rows, (unsigned long long)g.bytes); \
            return 1;                                                                                        \
        }                                                                                                    \
    } while (0)

int main()
{
    long long split = 0, several = 0, over = 0;
    for (int it = 0; it < 40000; ++it) {
        const int lb = 2 + (int)(rnd() % 3), s1 = 1 + (int)(rnd() % (it % 2 ? 300 : 40)), s2 = 1 + (int)(rnd() % (it % 3 ? 300 : 40));
        const uint64_t row = 4 * (1 + rnd() % 500), whole = row * (uint64_t)s1 * (uint64_t)s2;
        const uint64_t max = 1 + rnd() % (whole + whole / 4 + 1) / (1 + rnd() % 64);
        const UploadGroup g = upload_group(row, s1, s2, lb, max);
        const uint32_t nby = bricks_along(s1, lb), nbz = bricks_along(s2, lb), B = 1u << lb;
        CHECK(g.layers >= 1 && g.rows >= 1 && g.layers <= nbz && g.rows <= nby);
        CHECK(g.layers == 1 || g.rows == nby);
        CHECK(g.bytes <= max || (g.layers == 1 && g.rows == 1));
        split += g.rows < nby;
        several += g.layers > 1 && g.layers < nbz;
        over += g.bytes > max;
        for (int axis = 0; axis < 2; ++axis) {
            const int s = axis ? s2 : s1;
            const uint32_t nb = axis ? nbz : nby, step = axis ? g.layers : g.rows;
            for (uint32_t b = 0; b < nb; b += step) {
                const int lo = source_begin(b, lb, s), hi = source_end(b, step, lb, s);
                CHECK(lo >= 0 && lo < hi && hi <= s);
                CHECK((uint64_t)(hi - lo) <= slot_extent(step, lb, s));
                for (uint64_t X = (uint64_t)b * B; X <= (uint64_t)std::min(nb, b + step) * B; ++X)
                    if (X <= (uint64_t)s + 1) CHECK(slot_voxel((uint32_t)X, s) >= lo && slot_voxel((uint32_t)X, s) < hi);
            }
        }
        CHECK(g.bytes == slot_extent(g.layers, lb, s2) * slot_extent(g.rows, lb, s1) * row);
    }
    if (split < 1000 || several < 1000 || over < 100) {
        fprintf(stderr, "FAIL: %lld split, %lld of several layers, %lld above the bound\n", split, several, over);
        return 1;
    }
    // 2048^2 planes of normals: below 256 MiB in bricks of 16, and whole for 512^2
    const UploadGroup large = upload_group(2048 * 12, 2048, 64, 4, 256ull << 20), small = upload_group(512 * 12, 512, 512, 3, 256ull << 20);
    if (large.layers != 1 || large.bytes > 256ull << 20 || large.rows < 32 || small.rows != 65 || small.layers != 10) {
        fprintf(stderr, "FAIL: %u x %u, %u x %u\n", large.layers, large.rows, small.layers, small.rows);
        return 1;
    }
    printf("groups ok\n");
    return 0;
}
