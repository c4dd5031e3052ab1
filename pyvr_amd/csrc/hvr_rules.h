// hvr_rules.h -- the texel-layout and transparency rules of libhipvr as
// plain C++17 (no HIP headers): constexpr functions, which HIP compiles for
// both the host and the device, so the kernels (hvr_device.h), the host side
// (hipvr.hip) and a native test driver built with AddressSanitizer and
// UndefinedBehaviorSanitizer (tests/native/rules_check.cpp) run the same
// code.
#pragma once

#include <stdint.h>

namespace hvr {

// Bricks along an axis of GL size s with 2^lb interior texels per brick: the
// extended texture holds s + 2 texels (the edge copies), X in [0, s + 1].
constexpr uint32_t bricks_along(int s, int lb) { return ((uint32_t)s >> lb) + 1u; }

// The layout seen from the voxels, for checking slot_voxel (which the build
// kernel fills every slot by) against it.
// Slots along one axis that hold texel coordinate c of a texture of size s
// stored in nb bricks: (brick, local) pairs; returns how many (1..4).  In
// extended coordinates the texel sits at X = c + 1, and also at X = 0 when
// c = 0 and at X = s + 1 when c = s - 1 (the CLAMP_TO_EDGE copies).  Each X
// lives in brick X >> lb at local X & (B - 1), and, when it is the first
// texel of a brick, in the previous brick's apron at local B.  A position
// whose own brick would be brick nb (X = s + 1 with s + 1 a multiple of B)
// is only ever read through the apron of brick nb - 1.
constexpr int axis_slots(int c, int s, int lb, uint32_t nb, uint32_t br[4], uint32_t lo[4])
{
    const uint32_t B = 1u << lb, M = B - 1u;
    int n = 0;
    uint32_t X[3] = {(uint32_t)c + 1u, 0u, 0u};
    int nx = 1;
    if (c == 0) X[nx++] = 0u;
    if (c == s - 1) X[nx++] = (uint32_t)s + 1u;
    for (int k = 0; k < nx; ++k) {
        if ((X[k] >> lb) < nb) {
            br[n] = X[k] >> lb;
            lo[n] = X[k] & M;
            ++n;
        }
        if ((X[k] & M) == 0u && X[k] > 0u) {  // apron copy in the previous brick
            br[n] = (X[k] >> lb) - 1u;
            lo[n] = B;
            ++n;
        }
    }
    return n;
}

// The voxel that texel X of an axis (extended coordinates) holds, X <= s + 1:
// the inverse of axis_slots, which names the slots of a voxel.
constexpr int slot_voxel(uint32_t X, int s)
{
    const int c = (int)X - 1;
    return c < 0 ? 0 : c < s ? c : s - 1;
}

// The bricks that one group of an upload builds: `layers` brick layers of
// `rows` brick rows each, whose source -- the planes and rows that the bricks'
// slots hold, one more of either than their own -- takes `bytes` of staging.
// Whole planes while one layer's fit `max`, else rows of one layer; a single
// row of bricks may take more than `max`.
struct UploadGroup {
    uint32_t layers, rows;
    uint64_t bytes;
};
constexpr uint64_t slot_extent(uint64_t bricks, int lb, int s)
{
    const uint64_t n = (bricks << lb) + 1u;
    return n < (uint64_t)s ? n : (uint64_t)s;
}
constexpr UploadGroup upload_group(uint64_t row_bytes, int s1, int s2, int lb, uint64_t max)
{
    UploadGroup g = {1, 1, 0};
    const uint32_t nby = bricks_along(s1, lb), nbz = bricks_along(s2, lb);
    const uint64_t plane = row_bytes * (uint64_t)s1, planes = max / plane, depth = slot_extent(1, lb, s2);
    if (planes >= depth) {
        g.rows = nby;
        if (planes >= (uint64_t)s2) g.layers = nbz;
        else g.layers = (uint32_t)((planes - 1) >> lb);   // at least 1: planes >= 2^lb + 1
        g.bytes = slot_extent(g.layers, lb, s2) * plane;
    } else {
        const uint64_t lines = max / (row_bytes * depth);
        if (lines >= (uint64_t)s1) g.rows = nby;
        else if (lines > (1u << lb)) g.rows = (uint32_t)((lines - 1) >> lb);
        g.bytes = depth * slot_extent(g.rows, lb, s1) * row_bytes;
    }
    return g;
}
// The source indices along an axis of size s for bricks [b, b + n): texel X
// holds voxel X - 1, the edge texels the edge voxels.
constexpr int source_begin(uint32_t b, int lb, int s)
{
    const int64_t at = ((int64_t)b << lb) - 1;
    return at < 0 ? 0 : at < s ? (int)at : s - 1;
}
constexpr int source_end(uint32_t b, uint32_t n, int lb, int s)
{
    const int64_t at = ((int64_t)b + n) << lb;
    return at < s ? (int)at : s;
}

// Whether a brick whose density range is [lo, hi] can only ever sample LUT
// entries that are exactly transparent.  A sample of density rho reads
// u = clamp(rho*N - 1/2, 0, N-1) and weights entry floor(u) by 1 - frac(u)
// and entry floor(u) + 1 by frac(u), so the entries with non-zero weight over
// densities in [lo, hi] are floor(u(lo)) .. ceil(u(hi)); the range is widened
// by a margin for the rounding of the interpolated density (a few ulps of
// the largest tap).  `nz` holds the prefix counts (N + 1 values) of entries
// that are not exactly transparent.  Ranges of bricks holding a NaN are
// (-inf, +inf).  The clamps follow IEEE maxNum/minNum (fmaxf/fminf); the
// clamped values are non-negative, so truncation is floor.
constexpr bool brick_clear_range(float lo, float hi, const int *nz, int n)
{
    const float fn = (float)n, fn1 = (float)(n - 1);
    const float alo = lo < 0.f ? -lo : lo, ahi = hi < 0.f ? -hi : hi;
    const float m = (alo > ahi ? alo : ahi) * fn * 1e-5f + 1e-3f;
    float ulo = lo * fn - 0.5f - m;
    float uhi = hi * fn - 0.5f + m;
    ulo = ulo > 0.f ? (ulo < fn1 ? ulo : fn1) : 0.f;
    uhi = uhi > 0.f ? (uhi < fn1 ? uhi : fn1) : 0.f;
    const int i0 = (int)ulo;
    const int t1 = (int)uhi;
    const int i1 = (float)t1 < uhi ? t1 + 1 : t1;
    return nz[i1 + 1] - nz[i0] == 0;
}

// Clearance of a brick: 0 when it is not transparent for the LUT, else
// r + 1 for the largest r <= kMaxClearance - 1 such that every brick within r
// bricks of it along every axis is transparent (bricks outside the volume
// count as transparent: a ray that gets there has left the box).
//
// From a sample in a brick of clearance d, a ray stays among transparent
// bricks for as many further steps as it needs to move (d - 1) bricks of B
// texels along any axis.  `leap_rate` bounds its motion per step along one
// axis, in texels: the step ds times the texels per unit k, plus the rounding
// of the position (at most half an ulp of the larger bound in magnitude, `m`,
// taken doubled).  With `inv` = 1 / the largest rate of the three axes,
// leap_steps is floor(((d - 1) B - 1) inv), the 1 covering the rounding of the
// texel coordinates at both ends (below 2^-21 of at most 2^20 texels).
constexpr int kMaxClearance = 5;
constexpr float leap_rate(float ds, float k, float m) { return ((ds < 0.f ? -ds : ds) + m * 0x1p-23f) * k * 1.000001f; }
constexpr int leap_steps(int d, int lb, float inv)
{
    const float n = (float)(((d - 1) << lb) - 1) * inv;
    return n > 0.f ? (n < 65536.f ? (int)n : 65536) : 0;   // 0 for a NaN
}

// Prefix counts (n + 1 values) of LUT entries that are not exactly
// transparent.  The march reads entry i as v[i] + a*(v[i+1] - v[i]) with a
// in [0, 1), so entry i yields alpha 0 and a finite colour for every a (the
// reach of a > 0 into entry i+1 is accounted for by the brick rule) only
// when its alpha is 0 and the colours of it and of its successor, and the
// successor's alpha, are bounded (|x| <= 1e38 also excludes NaN and
// overflow of the difference: 0 * inf is NaN).
constexpr bool lut_bounded(float x) { return (x < 0.f ? -x : x) <= 1e38f; }

constexpr void lut_prefix_counts(const float *src, int cnt, int *nz)
{
    nz[0] = 0;
    for (int i = 0; i < cnt; ++i) {
        const float *e = src + 4 * i, *f = i + 1 < cnt ? e + 4 : e;
        const bool clear = e[3] == 0.f && lut_bounded(e[0]) && lut_bounded(e[1]) && lut_bounded(e[2]) &&
                           lut_bounded(f[0]) && lut_bounded(f[1]) && lut_bounded(f[2]) && lut_bounded(f[3]);
        nz[i + 1] = nz[i] + (clear ? 0 : 1);
    }
}

// Cost-ordered dispatch of a frame's ray blocks.  A frame ends when
// its longest waves do; dispatched in row order, long blocks that start
// late (after the first round of resident blocks) set the frame's end.
// k_order_blocks gives each block a cost key, the largest iteration bound of
// three of its rays, and files the block under a key bucket; the march then
// takes the blocks of the largest keys first.  Buckets split [0, max_steps] evenly,
// bucket 0 holding the largest keys.
constexpr int kOrderBuckets = 16;
constexpr int order_bucket(int key, int max_steps)
{
    if (key <= 0 || max_steps <= 0) return kOrderBuckets - 1;
    const long long k = (long long)key * kOrderBuckets / ((long long)max_steps + 1);
    return kOrderBuckets - 1 - (int)(k < kOrderBuckets - 1 ? k : kOrderBuckets - 1);
}

// Dispatch position b of a cost-ordered frame -> logical block (row-major,
// `ntx` blocks per row).  The first `head` positions (the blocks of the
// first multiple-of-8 block rows) are dealt to 8 classes in turn: class
// b & 7 holds block rows class, class + 8, ... (blocks are dispatched
// round-robin over the 8 XCDs, so one class runs on one XCD and its L2 sees
// whole rows), and within a class the blocks are taken bucket by bucket
// from `slots` (`cap` entries per class and bucket, cap = the class's
// block count) in the numbers `cnt` holds (kOrderBuckets per class).
// Later positions keep the row-major order.  Returns b itself when the
// counts do not cover the position (never with counts ray setup wrote).
template <typename U>
constexpr int ordered_block(int b, int head, const U *cnt, const U *slots, int cap)
{
    if (b >= head) return b;
    const int x = b & 7;
    uint32_t j = (uint32_t)(b >> 3);
    for (int k = 0; k < kOrderBuckets; ++k) {
        const uint32_t c = (uint32_t)cnt[x * kOrderBuckets + k];
        if (j < c)
            return j < (uint32_t)cap ? (int)slots[(uint64_t)(x * kOrderBuckets + k) * (uint64_t)cap + j] : b;
        j -= c;
    }
    return b;
}

// Lanes per ray of a single frame's march: with fewer rays than keep the device
// busy, a frame takes as long as its longest rays, whose samples follow one
// another; marched by 2 or 4 adjacent lanes, which take successive samples and
// composite them in order, a ray ends in as many fewer iterations, for more
// instructions a sample (14-18 % with 2 lanes, about 35 % with 4).  `resident`:
// the rays the device marches at once with one lane each (524,288 on 256
// compute units).
//
// Where transparent bricks are stepped over, rays differ in length and the
// lines lie far out.  Measured (us, 1 / 2 / 4 lanes; cameras averaged): 64^2 of
// a 256^3 volume 338 / 177 / 100, 362^2 of it 268 / 166 / 116, 512^2 79 / 63 /
// 66, 1024^2 504 / 452 / 480 and 366 / 331 / 409, 1280^2 601 / 635 / 720, 2048^2
// 1237 / 1491 / 1780; 692 steps (`steps`: the largest iteration bound the rays
// can have), 2 / 4 lanes: 640^2 299 254 / 221 206 / 252 234, 720^2 326 303 / 250
// 240 / 285 276 (FP32+FP32x3 256^3 / FP16+FP16x3 320^3 / UNORM8+SNORM8x3 224^3).
//
// Where none are, rays of a filled volume are about equally long and the device
// stays busy to the end, while those that end in dense matter or cross thin noise
// still differ.  Long rays gain from lanes as long as a sample waits for its
// texels: 16-byte ones, which take the L1 several passes, and volumes well above
// the L2s (`bytes` in all); few steps leave little to share out; texels below 4
// bytes, whose loads cost more than what is done with them, gain throughout.  A
// volume filled with thin fog, us by 1 / 2 / 4 lanes in row order at 0.15, 0.3, 0.5,
// 0.75 and 1.5 of the resident rays:
//   FP32+FP32x3 256^3, 692 steps     411 266 219  447 425 350  679 544 504  728 695 715  1258 1162 1330
//   FP16+FP16x3 256^3, 692 steps     275 189 149  285 263 244  368 363 361  450 476 499  796 815 916
//   UNORM8+SNORM8x3 224^3, 692       292 212 166  333 308 285  437 424 403  524 563 576  922 972 1069
//   FP16+SNORM8x3 96^3, 2000         854 753 625  1078 1115 1079  1484 1617 1618  1870 2191 2313  3451 3809 4320
//   FP16+FP16x3 448^3, 346           280 232 211  267 319 280  331 331 325  342 375 382  479 511 570
//   FP32+FP32x3 256^3, 100           107 110 94  111 134 142  176 169 191  189 216 269  321 341 504
//   UNORM8+SNORM8x3 224^3, 100       73 58 49  85 81 79  108 111 108  136 146 150  232 248 276
//   FP32 256^3, 692                  253 158 115  253 199 190  295 269 278  368 348 380  601 588 695
//   UNORM8 224^3, 346                123 111 79  155 175 129  259 231 182  295 296 249  491 490 448
// 448 random frames without skipping (the workloads' ranges of volumes, presets
// and sizes) take 0.64 times as long by these lines as by one lane in plain row or
// cost order, two of them more than 4.5 % longer and the worst 12 %; 1992 of
// volumes filled with fog 0.84 times, 77 of them more than 4.5 % longer and the
// worst 20 %.  With 4 lanes out to 3/8 and 2 out to 3/4 of the resident rays for
// few steps and small texels, too, the fog's worst took 37 % longer.
constexpr int march_lanes(long long rays, long long resident, bool skipping, double steps, int texel,
                          unsigned long long bytes)
{
    if (skipping) return 8 * rays <= (steps < 512.0 ? 3 : 7) * resident ? 4 : 4 * rays <= 9 * resident ? 2 : 1;
    if (texel < 4) return 4 * rays <= 3 * resident ? 4 : 1;
    if (steps < 256.0) return 16 * rays <= 5 * resident ? 4 : 16 * rays <= 9 * resident ? 2 : 1;
    if (8 * rays <= (steps < 512.0 ? 3 : 4) * resident) return 4;
    return 4 * rays <= (texel >= 16 || bytes >= 128ull << 20 ? 6 : 3) * resident ? 2 : 1;
}

// Lanes per ray of a class of a batch, whose kernel takes transparent bricks
// into account whether there are any or not (how many there are is not known
// when it is launched) and fetches its tiles itself, the costliest first.
// `steps`: of a mean ray.  500 random batches of one to four requests take 0.76
// times as long by these lines as by one lane; over twelve volumes, mostly
// empty, partly empty and filled, by steps: 50 1.01, 100 0.95, 346 0.84, 692 0.76,
// 2000 0.63.  From the resident rays on, mostly empty volumes still gain by 2
// lanes and filled ones lose (1.25 times, 692 steps, the time of one lane before
// over that by 1 and by 2: 1.16, 1.24 and 1.00, 1.00; 2 times, 346 steps: 1.15, 1.11
// and 0.99, 0.91).  One rule for all steps, 4 lanes out to 3/8 and 2 out to 9/4 of
// the resident rays, took 7 % longer at 50 steps than one lane and cost 872 of
// those 6432 batches more than 10 %; these lines cost 141.
constexpr int batch_lanes(long long rays, long long resident, double steps)
{
    if (steps < 64.0) return 10 * rays <= resident ? 4 : 4 * rays <= resident ? 2 : 1;
    if (steps < 256.0) return 4 * rays <= resident ? 4 : 4 * rays <= 3 * resident ? 2 : 1;
    if (8 * rays <= 3 * resident) return 4;
    return 4 * rays <= (steps < 512.0 ? 5 : steps < 1024.0 ? 7 : 9) * resident ? 2 : 1;
}

// Dispatch order of the blocks kept in rows: consecutive blocks of a class
// (ordered_block) go to its 32 compute units in turn, so the number of blocks
// per row, modulo 32, is how far a column of the image, which is dense or empty
// as a whole more often than not, moves from row to row.  Where that keeps it
// on a few units (0 or 1, up to 4 backwards, or 16), row r of a class is rotated
// by r times this, which moves a column by 13 units a row (512^2, 2 lanes: 232
// -> 187 us, 184 -> 149; 496^2 306 -> 248, 171 -> 147; 480^2 270 -> 251; 528^2
// 183 -> 165; 256^2, 4 lanes: 106 -> 98).  Other widths spread by themselves:
// rotating them gained nothing (640^2, 672^2 +1..7 %), and above the resident
// rays the blocks that start late even things out either way.
constexpr int row_rotation(int ntx)
{
    const int n = ntx & 31;
    return ntx >= 16 && (n <= 1 || n == 16 || n >= 28) ? ((ntx - 13) & 31) % ntx : 0;
}

// Whether HVR_ORDER_AUTO orders a frame by cost: with more blocks than the
// march keeps resident (8 of 256 threads per unit) blocks start late, and
// that sets the frame's end, unless the rays' `steps` are few.  Where bricks are
// stepped over, a frame of more than 2.25 times the resident rays loses more to
// marching all dense blocks at once than it gains (us in row order / ordered:
// 1024^2, 1 lane, 346 steps 394 / 364, 446 / 422; 2 lanes, 692 steps 529 / 495; 2
// lanes, 100 steps 159 / 178; 1536^2 767 / 771; 2048^2, 100 steps 452 / 516).
// Where none are, it does not (three times the resident rays of a filled volume,
// 692 steps: 4 % longer in row order, 2000 steps 5 to 9 %).
constexpr bool order_auto(long long blocks, long long rays, long long resident, bool skipping, int lanes, double steps)
{
    return blocks * 256 > resident && steps >= 256.0 * lanes && (!skipping || 4 * rays <= 9 * resident);
}

// Correctly rounded quotients g / d of several g by one reciprocal (Markstein,
// IBM J. Res. Dev. 34, 1990): an approximation within an ulp of 1 / d, refined
// once, is 1 / d correctly rounded unless the mantissa of d is all ones (its
// reciprocal lies next to the middle of two floats); with it the first
// product's exact residual makes the quotient faithful and the second one's
// rounds it, as long as no residual is lost below the normal numbers.
constexpr bool reciprocal_divides(uint32_t d_bits) { return (d_bits & 0x7fffffu) != 0x7fffffu; }
template <typename F>   // F: float (clang takes no constexpr function of __builtin_fmaf that is no template)
constexpr F refine_reciprocal(F d, F y)
{
    return __builtin_fmaf(__builtin_fmaf(-d, y, 1.f), y, y);
}
template <typename F>
constexpr F reciprocal_quotient(F g, F d, F y)
{
    F q = g * y;
    q = __builtin_fmaf(__builtin_fmaf(-d, q, g), y, q);
    return __builtin_fmaf(__builtin_fmaf(-d, q, g), y, q);
}

// Inverse of a 4x4 matrix (row-major, m[4*r + c]) by Gauss-Jordan
// elimination with partial pivoting.  Returns false when singular.
constexpr bool inverse4(const double *m, double *inv)
{
    double a[4][8] = {};
    for (int r = 0; r < 4; ++r)
        for (int c = 0; c < 8; ++c) a[r][c] = c < 4 ? m[4 * r + c] : (c - 4 == r ? 1.0 : 0.0);
    for (int col = 0; col < 4; ++col) {
        int piv = col;
        for (int r = col + 1; r < 4; ++r) {
            const double x = a[r][col] < 0 ? -a[r][col] : a[r][col];
            const double y = a[piv][col] < 0 ? -a[piv][col] : a[piv][col];
            if (x > y) piv = r;
        }
        if (a[piv][col] == 0.0) return false;
        if (piv != col)
            for (int c = 0; c < 8; ++c) {
                const double t = a[col][c];
                a[col][c] = a[piv][c];
                a[piv][c] = t;
            }
        const double d = a[col][col];
        for (int c = 0; c < 8; ++c) a[col][c] /= d;
        for (int r = 0; r < 4; ++r) {
            if (r == col) continue;
            const double f = a[r][col];
            if (f != 0.0)
                for (int c = 0; c < 8; ++c) a[r][c] -= f * a[col][c];
        }
    }
    for (int r = 0; r < 4; ++r)
        for (int c = 0; c < 4; ++c) inv[4 * r + c] = a[r][c + 4];
    return true;
}

}  // namespace hvr
