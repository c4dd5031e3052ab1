// Native check of the clearance leap (leap_rate and leap_steps in
// pyvr_amd/csrc/hvr_rules.h): rays walked in float32 as the march walks them,
// over boxes far from and around the origin, brick edges 8 and 16, volumes of
// 1 to 4096 texels per axis and steps from a thousandth of a texel to several
// bricks.  From every sample, the samples up to leap_steps further on must lie
// within d - 1 bricks of the sample's brick along every axis.  Exit status 0
// on success.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>

#include <algorithm>
#include <vector>

#include "hvr_rules.h"

using namespace hvr;

static uint64_t g_state = 0x9e3779b97f4a7c15ull;
static double urand()
{
    g_state ^= g_state << 13;
    g_state ^= g_state >> 7;
    g_state ^= g_state << 17;
    return (double)(g_state >> 11) * 0x1p-53;
}

int main()
{
    long long leaps = 0, far = 0;
    for (int it = 0; it < 30000; ++it) {
        const int lb = urand() < 0.5 ? 3 : 4;
        float bmin[3], bmax[3], ext[3], k[3], ds[3], p[3], s[3];
        double dir[3], len = 0;
        const double at = urand() < 0.5 ? 0.0 : exp(urand() * 14.0);   // distance of the box from the origin
        for (int a = 0; a < 3; ++a) {
            const double w = exp(urand() * 4.0 - 1.0);
            bmin[a] = (float)((urand() < 0.5 ? -at : at) - w * urand());
            bmax[a] = (float)(bmin[a] + w);
            ext[a] = bmax[a] - bmin[a];
            if (!(ext[a] >= 1e-20f)) ext[a] = 1.f, bmax[a] = bmin[a] + 1.f;
            k[a] = (float)(floor(exp(urand() * 8.3)) / (double)ext[a]);
            dir[a] = urand() < 0.1 ? 0.0 : 2 * urand() - 1;
            len += dir[a] * dir[a];
        }
        if (!(len > 0)) continue;
        const float step = (float)(ext[0] * exp(urand() * -7.0));
        float rate = 0.f;
        for (int a = 0; a < 3; ++a) {
            ds[a] = (float)(dir[a] / sqrt(len)) * step;
            rate = std::max(rate, leap_rate(ds[a], k[a], std::max(fabsf(bmin[a]), fabsf(bmax[a]))));
            // walked along the step's direction, as the march does
            s[a] = ds[a] < 0.f ? -1.f : 1.f;
            p[a] = s[a] * (bmin[a] + ext[a] * (float)urand());
        }
        const float inv = 1.f / rate;
        const int d = 1 + (int)(urand() * kMaxClearance), n = std::min(leap_steps(d, lb, inv), 2000);
        int first[3] = {0, 0, 0};
        for (int i = 0; i <= n; ++i) {
            for (int a = 0; a < 3; ++a) {
                const float w = fabsf(p[a] + -(s[a] * bmin[a]));
                if (!(w <= ext[a] * 1.5f)) goto done;   // past the box: nothing is sampled
                const int b = (int)((uint32_t)fmaf(w, k[a], 0.5f) >> lb);
                if (i == 0) first[a] = b;
                else if (abs(b - first[a]) > d - 1) {
                    fprintf(stderr, "FAIL: axis %d, clearance %d, step %d of %d reached brick %d from %d (k %g ds %g at %g)\n",
                            a, d, i, n, b, first[a], k[a], ds[a], bmin[a]);
                    return 1;
                }
                far += i > 0 && abs(b - first[a]) == d - 1 && d > 1;
            }
            for (int a = 0; a < 3; ++a) p[a] = p[a] + s[a] * ds[a];
        }
    done:
        leaps += n > 0;
    }
    // the rule is not vacuous, and no leap leaves a brick without clearance
    if (leaps < 5000 || far < 5000 || leap_steps(1, 4, 0.01f) != 0 || leap_steps(3, 3, NAN) != 0 ||
        leap_steps(5, 4, INFINITY) != 65536) {
        fprintf(stderr, "FAIL: %lld leaps, %lld at the edge\n", leaps, far);
        return 1;
    }
    printf("leaps ok\n");
    return 0;
}
