// hvr_share.h -- which requests of a batch share a volume and a LUT.  Plain
// C++17 (no HIP), so that a native test driver can run it
// (tests/native/share_check.cpp).
#pragma once

#include <stddef.h>
#include <stdint.h>
#include <string.h>

#include <vector>

namespace hvr {

// Hash of n floats by their bits: four FNV-1a chains over pairs, a quarter of
// the pairs each, so that the multiplications overlap (one chain over the
// single words of a 256-entry LUT took 0.7 us, a fifth of hvr_batch_add).
inline uint64_t float_hash(const float *f, size_t n)
{
    constexpr uint64_t kPrime = 0x100000001b3ull;
    uint64_t h[4] = {0xcbf29ce484222325ull, 0x84222325cbf29ce4ull, 0x9ce484222325cbf2ull, 0x2325cbf29ce48422ull};
    size_t k = 0;
    for (; k + 8 <= n; k += 8)
        for (int c = 0; c < 4; ++c) {
            uint64_t w;
            memcpy(&w, f + k + 2 * c, 8);
            h[c] = (h[c] ^ w) * kPrime;
        }
    for (; k < n; ++k) {
        uint32_t w;
        memcpy(&w, f + k, 4);
        h[0] = (h[0] ^ w) * kPrime;
    }
    uint64_t all = n;
    for (uint64_t c : h) all = (all ^ c ^ c >> 32) * kPrime;
    return all;
}

// The first of equal things among up to n, found by their hashes (open
// addressing, at most half full).
class ShareTable {
public:
    explicit ShareTable(size_t n)
    {
        size_t cap = 16;
        while (cap < 2 * n) cap *= 2;
        slots_.assign(cap, Slot{0, -1});
    }
    // The value added before with this hash for which `equal(value)` holds, or -1
    // after adding `value` (>= 0).
    template <typename Equal>
    int find_or_add(uint64_t hash, int value, Equal equal)
    {
        const size_t mask = slots_.size() - 1;
        for (size_t at = (size_t)(hash ^ hash >> 32) & mask;; at = (at + 1) & mask) {
            Slot &s = slots_[at];
            if (s.value < 0) {
                s = Slot{hash, value};
                return -1;
            }
            if (s.hash == hash && equal(s.value)) return s.value;
        }
    }

private:
    struct Slot {
        uint64_t hash;
        int value;
    };
    std::vector<Slot> slots_;
};

}  // namespace hvr
