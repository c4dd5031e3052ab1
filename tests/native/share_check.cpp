// Native check of the sharing search (pyvr_amd/csrc/hvr_share.h): things with
// distinct hashes are never compared, equal ones once each, ones whose hashes
// collide are told apart; the hash takes every float and the length.  Exit
// status 0 on success.
#include <stdio.h>

#include <vector>

#include "hvr_share.h"

using namespace hvr;

#define CHECK(cond)                                                     \
    do {                                                                \
        if (!(cond)) {                                                  \
            fprintf(stderr, "FAIL %s:%d: %s\n", __FILE__, __LINE__, #cond); \
            return 1;                                                   \
        }                                                               \
    } while (0)

int main()
{
    const int n = 20000;
    long long compared = 0;
    {   // 20,000 LUTs of 8 entries, each its own: no comparison, where a walk over those met before takes 2 * 10^8
        ShareTable t(n);
        std::vector<float> lut(32, 0.5f);
        for (int k = 0; k < n; ++k) {
            lut[k % 32] = 0.5f + (float)(k + 1) / (2 * n);
            CHECK(t.find_or_add(float_hash(lut.data(), lut.size()), k, [&](int) { return ++compared, false; }) == -1);
            lut[k % 32] = 0.5f;
        }
        CHECK(compared == 0);
    }
    {   // all equal: one comparison each, with the first
        ShareTable t(n);
        for (int k = 0; k < n; ++k)
            CHECK(t.find_or_add(42, k, [&](int v) { return ++compared, v == 0; }) == (k ? 0 : -1));
        CHECK(compared == n - 1);
    }
    {   // one hash for all of 16 kinds
        ShareTable t(160);
        for (int k = 0; k < 160; ++k) {
            const int got = t.find_or_add(7, k, [&](int v) { return v % 16 == k % 16; });
            CHECK(got == (k < 16 ? -1 : k % 16));
        }
    }
    for (size_t len : {size_t(0), size_t(1), size_t(7), size_t(8), size_t(9), size_t(1024), size_t(8191)}) {
        std::vector<float> f(len + 1, 0.25f);
        const uint64_t h = float_hash(f.data(), len);
        CHECK(h != float_hash(f.data(), len + 1));
        for (size_t k = 0; k < len; ++k) {
            f[k] = 0.5f;
            CHECK(h != float_hash(f.data(), len));
            f[k] = 0.25f;
        }
        CHECK(h == float_hash(f.data(), len));
    }
    printf("share ok\n");
    return 0;
}
