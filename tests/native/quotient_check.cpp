// Native check that quotients by a shared reciprocal (reciprocal_quotient in
// pyvr_amd/csrc/hvr_rules.h) are correctly rounded: every divisor mantissa,
// every approximation of its reciprocal within an ulp, and as numerators a
// power of two and two random mantissas, against the processor's division.
// Scaling by powers of two changes nothing between the normal numbers' ends.
// Exit status 0 on success.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include "hvr_rules.h"

using namespace hvr;

static float from_bits(uint32_t b)
{
    float f;
    memcpy(&f, &b, 4);
    return f;
}

int main()
{
    uint64_t state = 0x9e3779b97f4a7c15ull;
    long long checked = 0, refused = 0;
    for (uint32_t m = 0; m < (1u << 23); ++m) {
        const float d = from_bits(0x3f800000u | m);
        if (!reciprocal_divides(0x3f800000u | m)) {
            ++refused;
            continue;
        }
        state ^= state << 13;
        state ^= state >> 7;
        state ^= state << 17;
        const float g[3] = {1.f, from_bits(0x3f800000u | ((uint32_t)state & 0x7fffffu)),
                            from_bits(0x3f800000u | ((uint32_t)(state >> 32) & 0x7fffffu))};
        const double exact = 1.0 / (double)d;   // in (0.5, 1], where floats lie 2^-24 apart
        const float near = (float)exact;
        const float seeds[3] = {nextafterf(near, 0.f), near, nextafterf(near, 2.f)};
        for (float y0 : seeds) {
            if (fabs((double)y0 - exact) > 0x1p-24) continue;
            const float y = refine_reciprocal(d, y0);
            for (float n : g) {
                if (reciprocal_quotient(n, d, y) != n / d) {
                    fprintf(stderr, "FAIL: %a / %a from the seed %a: %a, not %a\n", n, d, y0,
                            reciprocal_quotient(n, d, y), n / d);
                    return 1;
                }
                ++checked;
            }
        }
    }
    if (refused > 1 || checked < 3ll * 2 * ((1 << 23) - 1)) {
        fprintf(stderr, "FAIL: %lld checked, %lld refused\n", checked, refused);
        return 1;
    }
    printf("quotients ok\n");
    return 0;
}
