// hvr_device.h -- device code of libhipvr: texel formats, GL-style sampling,
// ray setup and cost ordering, the march-and-composite kernels, the kernels that
// build volumes and their transparency flags, and the batch kernels (gfx950,
// wave64).
//
// Semantics follow the reference fragment shader pyvr/shaders/volume.frag.glsl
// and the GL state of pyvr/moderngl_renderer/manager.py (paths relative to the
// reference repository); each block names the lines it implements.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hvr_rules.h"

namespace hvr {

// ---------------------------------------------------------------------------
// Texel formats.  A volume stores one texel per voxel; a texel holds the
// scalar field, the normal field, or both (interleaved so that one load per
// trilinear tap returns everything a sample needs).
//   S_*  scalar only         N_*  normals only        C_*  both
// Decoding yields (nx, ny, nz, rho).  For scalar-only texels the normal part
// reads (rho, 0, 0), which is what a 3-channel GL sampler returns from a
// 1-channel texture; for normal-only texels rho reads nx (the .r channel).
// In the fast paths SNORM8 normals stay raw integers (the normal is
// normalised afterwards, so the 1/127 scale cancels) and UNORM8 scalars are
// scaled by 1/255 after interpolation (filtering is linear).  FP16 scalars
// and normals are interpolated straight from their halves (v_fma_mix_f32:
// float32 accumulation of exactly converted halves), with no conversion
// instructions.
enum TexFmt : int {
    TF_NONE = 0,
    TF_S_F32 = 1,      // float                                    4 B
    TF_S_F16 = 2,      // half                                     2 B
    TF_S_U8 = 3,       // unorm8                                   1 B
    TF_N_F32 = 4,      // float4 (nx, ny, nz, 0)                  16 B
    TF_N_SN8 = 5,      // u32 nx | ny<<8 | nz<<16                  4 B
    TF_C_F32_F32 = 6,  // float4 (nx, ny, nz, rho)                16 B
    TF_C_F16_F32 = 7,  // float4 (nx, ny, nz, bits: half rho)     16 B
    TF_C_U8_F32 = 8,   // float4 (nx, ny, nz, bits: u8 rho)       16 B
    TF_C_F32_SN8 = 9,  // u32x2 (float rho, sn8 xyz)               8 B
    TF_C_F16_SN8 = 10, // u32x2 (half rho | half qx << 16, half qy | half qz << 16), q the
                       // SNORM8 integers in [-127, 127], exact as halves  8 B
    TF_C_U8_SN8 = 11,  // u32 sn8 xyz | u8 rho << 24               4 B
    TF_C_F16_F16 = 12, // u32x2 (half rho | half nx << 16, half ny | half nz << 16)  8 B
    TF_N_F16 = 13,     // u32x2 (half nx | half ny << 16, half nz)  8 B
    TF_COUNT = 14
};

__host__ __device__ constexpr int texel_bytes(int f)
{
    return f == TF_S_F32 ? 4 : f == TF_S_F16 ? 2 : f == TF_S_U8 ? 1
         : f == TF_N_F32 ? 16 : f == TF_N_SN8 ? 4
         : (f == TF_C_F32_F32 || f == TF_C_F16_F32 || f == TF_C_U8_F32) ? 16
         : (f == TF_C_F32_SN8 || f == TF_C_F16_SN8) ? 8 : f == TF_C_U8_SN8 ? 4
         : (f == TF_C_F16_F16 || f == TF_N_F16) ? 8 : 0;
}
__host__ __device__ constexpr bool fmt_has_scalar(int f)
{
    return f == TF_S_F32 || f == TF_S_F16 || f == TF_S_U8 || (f >= TF_C_F32_F32 && f <= TF_C_F16_F16);
}
__host__ __device__ constexpr bool fmt_has_normal(int f)
{
    return f == TF_N_F32 || f == TF_N_SN8 || f == TF_N_F16 || f >= TF_C_F32_F32;
}
__host__ __device__ constexpr bool fmt_sn8_normal(int f)
{
    return f == TF_N_SN8 || f == TF_C_F32_SN8 || f == TF_C_F16_SN8 || f == TF_C_U8_SN8;
}
__host__ __device__ constexpr bool fmt_u8_scalar(int f)
{
    return f == TF_S_U8 || f == TF_C_U8_F32 || f == TF_C_U8_SN8;
}

// ---------------------------------------------------------------------------
// Brick layout with apron.  A texture of GL size (s0, s1, s2) is addressed in
// extended coordinates X = x + 1 in [0, s+1] per axis, where X = 0 and
// X = s+1 hold copies of the edge texels (x = 0 and x = s-1): sampling the
// extended texture without clamping is exactly GL's CLAMP_TO_EDGE.  The
// extended texture is cut into bricks of B = 2^lb interior texels per axis,
// each stored with one more texel per axis (its neighbour's first), so a
// brick holds E^3 texels, E = B + 1, x fastest.  A trilinear footprint with
// lower corner X0 lies in brick X0 >> lb at local X0 & (B-1) .. +1: one base
// address per sample, the eight taps at fixed offsets.
struct TexDesc {
    const void *base;
    int s0, s1, s2;        // GL size
    float k0, k1, k2;      // s_axis / world extent of the axis it samples
    int lb;                // log2 of the brick interior edge
    uint32_t nbx, nby;     // bricks along x and y
    uint32_t brick_bytes;  // E^3 * texel bytes
    uint32_t nbytes32;     // allocation bytes when below 4 GiB with fewer than 2^24
                           // bricks (buffer-load path), else 0
    int fmt;
    int role;              // field a sampler reads: 0 scalar, 1 normal
};


// Loads and stores through pointers the compiler cannot place (fetched from
// descriptors in memory): they address device global memory, so issue
// global (not flat) instructions.
template <typename T>
__device__ __forceinline__ T ld_global(const T *p)
{
    return *(const __attribute__((address_space(1))) T *)p;
}
__device__ __forceinline__ float4 ld_global(const float4 *p)
{
    typedef float v4 __attribute__((ext_vector_type(4)));
    const v4 v = *(const __attribute__((address_space(1))) v4 *)p;
    return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ float2 ld_global(const float2 *p)
{
    typedef float v2 __attribute__((ext_vector_type(2)));
    const v2 v = *(const __attribute__((address_space(1))) v2 *)p;
    return make_float2(v.x, v.y);
}
template <typename T>
__device__ __forceinline__ void st_global(T *p, const T &v)
{
    *(__attribute__((address_space(1))) T *)p = v;
}
__device__ __forceinline__ void st_global(uchar4 *p, const uchar4 &v)
{
    const uint32_t w = (uint32_t)v.x | ((uint32_t)v.y << 8) | ((uint32_t)v.z << 16) | ((uint32_t)v.w << 24);
    *(__attribute__((address_space(1))) uint32_t *)p = w;
}

__device__ __forceinline__ float sn8f(uint32_t w, int sh) { return (float)(int8_t)((w >> sh) & 0xffu); }
// the half in the low 16 bits of w
__device__ __forceinline__ float h16f(uint32_t w) { return __half2float(__ushort_as_half((unsigned short)(w & 0xffffu))); }

// Decode the texel at byte address p to (nx, ny, nz, rho) (raw SNORM8/UNORM8).
template <int F>
__device__ __forceinline__ float4 fetch4(const char *p)
{
    if constexpr (F == TF_S_F32) {
        const float v = *(const float *)p;
        return make_float4(v, 0.f, 0.f, v);
    } else if constexpr (F == TF_S_F16) {
        const float v = __half2float(*(const __half *)p);
        return make_float4(v, 0.f, 0.f, v);
    } else if constexpr (F == TF_S_U8) {
        const float v = (float)*(const uint8_t *)p;
        return make_float4(v, 0.f, 0.f, v);
    } else if constexpr (F == TF_N_F32) {
        const float4 t = *(const float4 *)p;
        return make_float4(t.x, t.y, t.z, t.x);
    } else if constexpr (F == TF_N_SN8) {
        const uint32_t w = *(const uint32_t *)p;
        const float x = sn8f(w, 0);
        return make_float4(x, sn8f(w, 8), sn8f(w, 16), x);
    } else if constexpr (F == TF_C_F32_F32) {
        return *(const float4 *)p;
    } else if constexpr (F == TF_C_F16_F32) {
        const float4 t = *(const float4 *)p;
        const __half h = __ushort_as_half((unsigned short)(__float_as_uint(t.w) & 0xffffu));
        return make_float4(t.x, t.y, t.z, __half2float(h));
    } else if constexpr (F == TF_C_U8_F32) {
        const float4 t = *(const float4 *)p;
        return make_float4(t.x, t.y, t.z, (float)(__float_as_uint(t.w) & 0xffu));
    } else if constexpr (F == TF_C_F32_SN8) {
        const uint2 t = *(const uint2 *)p;
        return make_float4(sn8f(t.y, 0), sn8f(t.y, 8), sn8f(t.y, 16), __uint_as_float(t.x));
    } else if constexpr (F == TF_C_U8_SN8) {
        const uint32_t w = *(const uint32_t *)p;
        return make_float4(sn8f(w, 0), sn8f(w, 8), sn8f(w, 16), (float)(w >> 24));
    } else if constexpr (F == TF_C_F16_F16 || F == TF_C_F16_SN8) {
        const uint2 t = *(const uint2 *)p;
        return make_float4(h16f(t.x >> 16), h16f(t.y), h16f(t.y >> 16), h16f(t.x));
    } else if constexpr (F == TF_N_F16) {
        const uint2 t = *(const uint2 *)p;
        const float x = h16f(t.x);
        return make_float4(x, h16f(t.x >> 16), h16f(t.y), x);
    } else {
        return make_float4(0.f, 0.f, 0.f, 0.f);
    }
}

// Scalar-only decode (avoids interpolating unused channels).
template <int F>
__device__ __forceinline__ float fetch1(const char *p)
{
    if constexpr (F == TF_S_F32) return *(const float *)p;
    else if constexpr (F == TF_S_F16) return __half2float(*(const __half *)p);
    else if constexpr (F == TF_S_U8) return (float)*(const uint8_t *)p;
    else return fetch4<F>(p).w;
}

// Runtime-format decode with exact GL scaling (generic path).
__device__ __forceinline__ float4 fetch_any(int fmt, const char *p)
{
    float4 t;
    switch (fmt) {
    case TF_S_F32: t = fetch4<TF_S_F32>(p); break;
    case TF_S_F16: t = fetch4<TF_S_F16>(p); break;
    case TF_S_U8: t = fetch4<TF_S_U8>(p); break;
    case TF_N_F32: t = fetch4<TF_N_F32>(p); break;
    case TF_N_SN8: t = fetch4<TF_N_SN8>(p); break;
    case TF_C_F32_F32: t = fetch4<TF_C_F32_F32>(p); break;
    case TF_C_F16_F32: t = fetch4<TF_C_F16_F32>(p); break;
    case TF_C_U8_F32: t = fetch4<TF_C_U8_F32>(p); break;
    case TF_C_F32_SN8: t = fetch4<TF_C_F32_SN8>(p); break;
    case TF_C_F16_SN8: t = fetch4<TF_C_F16_SN8>(p); break;
    case TF_C_U8_SN8: t = fetch4<TF_C_U8_SN8>(p); break;
    case TF_C_F16_F16: t = fetch4<TF_C_F16_F16>(p); break;
    case TF_N_F16: t = fetch4<TF_N_F16>(p); break;
    default: return make_float4(0.f, 0.f, 0.f, 0.f);
    }
    const float k127 = 1.0f / 127.0f, k255 = 1.0f / 255.0f;
    if (fmt_sn8_normal(fmt)) {
        t.x = fmaxf(t.x * k127, -1.f);
        t.y = fmaxf(t.y * k127, -1.f);
        t.z = fmaxf(t.z * k127, -1.f);
        if (fmt == TF_N_SN8) t.w = t.x;
    }
    if (fmt_u8_scalar(fmt)) {
        t.w *= k255;
        if (fmt == TF_S_U8) t.x = t.w;
    }
    return t;
}

// ---------------------------------------------------------------------------
// Trilinear sampling (GL_LINEAR, CLAMP_TO_EDGE, no mipmaps;
// manager.py:95-101, 123-129).  Per axis the GL rule is u = c*size - 1/2,
// taps floor(u), floor(u)+1 (clamped), weight frac(u).  With the extended
// coordinates of the brick layout the lower tap is X0 = floor(c*size + 1/2)
// in [0, size] and no clamp is needed.  (w0, w1, w2) is the position in
// world units from the box minimum along the axes sampled by texture x, y, z
// (world z, y, x: the shader's swizzle, volume.frag.glsl:90).
struct Footprint {
    const char *p;    // byte address of the lower-corner texel (global-load path)
    uint32_t off;     // its byte offset in the allocation (buffer-load path)
    float u, v, w;    // extended texel coordinates along texture x, y, z (>= 0 in
                      // the box; the weights are their fractional parts)
    uint32_t X, Y, Z; // the lower-corner texel (floor of u, v, w)
    uint32_t brick;   // brick holding the whole footprint
};

// A footprint in two steps: the coordinates and the brick (all that the
// transparent-brick test needs), then the texel address (what the loads
// need), so that samples in transparent bricks skip the second.
template <int LB, bool BUF>
__device__ __forceinline__ Footprint footprint_brick(const TexDesc &t, float w0, float w1, float w2)
{
    // u, v, w >= 0 for in-box positions (and the 0 the callers pass for
    // others), so truncation is floor
    Footprint f;
    f.u = fmaf(w0, t.k0, 0.5f);
    f.v = fmaf(w1, t.k1, 0.5f);
    f.w = fmaf(w2, t.k2, 0.5f);
    f.X = (uint32_t)f.u;
    f.Y = (uint32_t)f.v;
    f.Z = (uint32_t)f.w;
    if constexpr (BUF) {
        // The buffer path is only used with nbricks < 2^24 (and the
        // allocation below 4 GiB): every partial brick index and
        // brick_bytes (<= 17^3 * 16) fit 24 bits and the byte offset 32, so
        // single-pass 24-bit multiplies are exact.
        f.brick = __umul24(__umul24(f.Z >> LB, t.nby) + (f.Y >> LB), t.nbx) + (f.X >> LB);
    } else {
        f.brick = ((f.Z >> LB) * t.nby + (f.Y >> LB)) * t.nbx + (f.X >> LB);
    }
    f.p = nullptr;
    f.off = 0;
    return f;
}

template <int T, int LB, bool BUF>
__device__ __forceinline__ void footprint_addr(const TexDesc &t, Footprint &f)
{
    constexpr uint32_t M = (1u << LB) - 1u, E = (1u << LB) + 1u;
    const uint32_t local = ((f.Z & M) * E + (f.Y & M)) * E + (f.X & M);
    if constexpr (BUF)
        f.off = __umul24(f.brick, t.brick_bytes) + local * (uint32_t)T;   // < nbytes32 < 2^32
    else
        f.p = (const char *)t.base + (uint64_t)f.brick * t.brick_bytes + (uint64_t)(local * (uint32_t)T);
}


// Where the march reads texels from: a buffer resource (base and size in
// scalar registers, 32-bit per-lane offsets, reads past the allocation
// return 0) for allocations below 4 GiB, else a 64-bit base pointer.
template <bool BUF>
struct Src;
template <>
struct Src<true> {
    __amdgpu_buffer_rsrc_t r;
    __device__ explicit Src(const TexDesc &t)
        : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(t.base), (short)0, (int)t.nbytes32,
                                              0x00020000)) {}
};
template <>
struct Src<false> {
    __device__ explicit Src(const TexDesc &) {}
};

typedef uint32_t hvr_u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t hvr_u32x4 __attribute__((ext_vector_type(4)));

// NB dwords at byte offset o from the footprint's lower corner (o a
// compile-time constant; the buffer path folds it into the instruction).
template <int NB, bool BUF>
__device__ __forceinline__ void load_words(const Src<BUF> &s, const Footprint &f, uint32_t o, uint32_t *w)
{
    if constexpr (BUF) {
        if constexpr (NB == 1) {
            w[0] = __builtin_amdgcn_raw_buffer_load_b32(s.r, f.off + o, 0, 0);
        } else if constexpr (NB == 2) {
            const hvr_u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(s.r, f.off + o, 0, 0);
            w[0] = v.x; w[1] = v.y;
        } else {
#pragma unroll
            for (int q = 0; q < NB / 4; ++q) {
                const hvr_u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(s.r, f.off + o + 16u * q, 0, 0);
                w[4 * q] = v.x; w[4 * q + 1] = v.y; w[4 * q + 2] = v.z; w[4 * q + 3] = v.w;
            }
        }
    } else {
        // texels are 4-byte aligned: load with that alignment
        typedef hvr_u32x2 u2a __attribute__((aligned(4)));
        typedef hvr_u32x4 u4a __attribute__((aligned(4)));
        const char *p = f.p + o;
        if constexpr (NB == 1) {
            w[0] = *(const uint32_t *)p;
        } else if constexpr (NB == 2) {
            const hvr_u32x2 v = *(const u2a *)p;
            w[0] = v.x; w[1] = v.y;
        } else {
#pragma unroll
            for (int q = 0; q < NB / 4; ++q) {
                const hvr_u32x4 v = *(const u4a *)(p + 16 * q);
                w[4 * q] = v.x; w[4 * q + 1] = v.y; w[4 * q + 2] = v.z; w[4 * q + 3] = v.w;
            }
        }
    }
}

// Decode one texel held in dwords w[0 .. T/4-1] (formats of 4 bytes and
// more) to (nx, ny, nz, rho), raw SNORM8/UNORM8 integers as fetch4 gives.
template <int F>
__device__ __forceinline__ float4 decode_words(const uint32_t *w)
{
    if constexpr (F == TF_S_F32) {
        const float v = __uint_as_float(w[0]);
        return make_float4(v, 0.f, 0.f, v);
    } else if constexpr (F == TF_N_F32) {
        const float x = __uint_as_float(w[0]);
        return make_float4(x, __uint_as_float(w[1]), __uint_as_float(w[2]), x);
    } else if constexpr (F == TF_N_SN8) {
        const float x = sn8f(w[0], 0);
        return make_float4(x, sn8f(w[0], 8), sn8f(w[0], 16), x);
    } else if constexpr (F == TF_C_F32_F32) {
        return make_float4(__uint_as_float(w[0]), __uint_as_float(w[1]), __uint_as_float(w[2]),
                           __uint_as_float(w[3]));
    } else if constexpr (F == TF_C_F16_F32) {
        return make_float4(__uint_as_float(w[0]), __uint_as_float(w[1]), __uint_as_float(w[2]),
                           __half2float(__ushort_as_half((unsigned short)(w[3] & 0xffffu))));
    } else if constexpr (F == TF_C_U8_F32) {
        return make_float4(__uint_as_float(w[0]), __uint_as_float(w[1]), __uint_as_float(w[2]),
                           (float)(w[3] & 0xffu));
    } else if constexpr (F == TF_C_F32_SN8) {
        return make_float4(sn8f(w[1], 0), sn8f(w[1], 8), sn8f(w[1], 16), __uint_as_float(w[0]));
    } else if constexpr (F == TF_C_U8_SN8) {
        return make_float4(sn8f(w[0], 0), sn8f(w[0], 8), sn8f(w[0], 16), (float)(w[0] >> 24));
    } else if constexpr (F == TF_C_F16_F16 || F == TF_C_F16_SN8) {
        return make_float4(h16f(w[0] >> 16), h16f(w[1]), h16f(w[1] >> 16), h16f(w[0]));
    } else if constexpr (F == TF_N_F16) {
        const float x = h16f(w[0]);
        return make_float4(x, h16f(w[0] >> 16), h16f(w[1]), x);
    } else {
        return make_float4(0.f, 0.f, 0.f, 0.f);
    }
}

// Scalar (raw, as decode_words' w) and normal of a combined-format texel.
template <int F>
__device__ __forceinline__ float decode_scalar(const uint32_t *w)
{
    if constexpr (F == TF_C_F32_F32) return __uint_as_float(w[3]);
    else if constexpr (F == TF_C_F16_F32) return __half2float(__ushort_as_half((unsigned short)(w[3] & 0xffffu)));
    else if constexpr (F == TF_C_U8_F32) return (float)(w[3] & 0xffu);
    else if constexpr (F == TF_C_F32_SN8) return __uint_as_float(w[0]);
    else if constexpr (F == TF_C_U8_SN8) return (float)(w[0] >> 24);
    else if constexpr (F == TF_C_F16_F16 || F == TF_C_F16_SN8) return h16f(w[0]);
    else return 0.f;
}
template <int F>
__device__ __forceinline__ float3 decode_normal(const uint32_t *w)
{
    if constexpr (F == TF_C_F32_F32 || F == TF_C_F16_F32 || F == TF_C_U8_F32)
        return make_float3(__uint_as_float(w[0]), __uint_as_float(w[1]), __uint_as_float(w[2]));
    else if constexpr (F == TF_C_F32_SN8)
        return make_float3(sn8f(w[1], 0), sn8f(w[1], 8), sn8f(w[1], 16));
    else if constexpr (F == TF_C_U8_SN8)
        return make_float3(sn8f(w[0], 0), sn8f(w[0], 8), sn8f(w[0], 16));
    else if constexpr (F == TF_C_F16_F16 || F == TF_C_F16_SN8)
        return make_float3(h16f(w[0] >> 16), h16f(w[1]), h16f(w[1] >> 16));
    else return make_float3(0.f, 0.f, 0.f);
}

// The raw dwords of a footprint's eight texels of a combined format (4
// bytes and more): pair k = taps 2k, 2k+1 (y = k & 1, z = k >> 1).
template <int F, int LB, bool BUF>
__device__ __forceinline__ void load_pairs(const Src<BUF> &s, const Footprint &f, uint32_t raw[4][texel_bytes(F) / 2])
{
    constexpr int T = texel_bytes(F);
    constexpr uint32_t E = (1u << LB) + 1u;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        load_words<T / 2, BUF>(s, f, ((uint32_t)(k & 1) * E + (uint32_t)(k >> 1) * E * E) * (uint32_t)T, raw[k]);
}

// Trilinear scalar of a combined-format footprint from its raw pairs.
template <int F>
__device__ __forceinline__ float interp_scalar(const uint32_t (*raw)[texel_bytes(F) / 2], const float w[8])
{
    constexpr int H = texel_bytes(F) / 4;
    // an fma from 0 (not a product) lets a half operand fold into v_fma_mix
    float r = fmaf(w[0], decode_scalar<F>(raw[0]), 0.f);
#pragma unroll
    for (int k = 1; k < 8; ++k) r = fmaf(w[k], decode_scalar<F>(raw[k >> 1] + (k & 1) * H), r);
    return r;
}
template <int F>
__device__ __forceinline__ float3 interp_normal(const uint32_t (*raw)[texel_bytes(F) / 2], const float w[8])
{
    constexpr int H = texel_bytes(F) / 4;
    const float3 t0 = decode_normal<F>(raw[0]);
    float n0 = fmaf(w[0], t0.x, 0.f), n1 = fmaf(w[0], t0.y, 0.f), n2 = fmaf(w[0], t0.z, 0.f);
#pragma unroll
    for (int k = 1; k < 8; ++k) {
        const float3 t = decode_normal<F>(raw[k >> 1] + (k & 1) * H);
        n0 = fmaf(w[k], t.x, n0);
        n1 = fmaf(w[k], t.y, n1);
        n2 = fmaf(w[k], t.z, n2);
    }
    return make_float3(n0, n1, n2);
}

// The eight taps of a footprint, x fastest: tap i at (i&1, (i>>1)&1, i>>2).
// Formats of 4 bytes and more load each x-adjacent pair with one load of
// 2T bytes (texels are dword aligned); 1- and 2-byte formats load per tap.
template <int F, int LB, bool BUF>
__device__ __forceinline__ void load_taps(const Src<BUF> &s, const Footprint &f, float4 t[8])
{
    constexpr int T = texel_bytes(F);
    constexpr uint32_t E = (1u << LB) + 1u;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t o = ((uint32_t)(k & 1) * E + (uint32_t)(k >> 1) * E * E) * (uint32_t)T;
        if constexpr (T >= 4) {
            uint32_t w[T / 2];
            load_words<T / 2, BUF>(s, f, o, w);
            t[2 * k] = decode_words<F>(w);
            t[2 * k + 1] = decode_words<F>(w + T / 4);
        } else {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                float v;
                if constexpr (BUF) {
                    if constexpr (T == 2)
                        v = __half2float(__ushort_as_half(
                            __builtin_amdgcn_raw_buffer_load_b16(s.r, f.off + o + 2u * j, 0, 0)));
                    else
                        v = (float)__builtin_amdgcn_raw_buffer_load_b8(s.r, f.off + o + (uint32_t)j, 0, 0);
                } else {
                    v = fetch1<F>(f.p + o + T * j);
                }
                t[2 * k + j] = make_float4(v, 0.f, 0.f, v);
            }
        }
    }
}

// The eight trilinear weights, x fastest: w[i] for tap (i&1, (i>>1)&1, i>>2).
__device__ __forceinline__ void tri_weights(float a, float b, float g, float w[8])
{
    const float a1 = 1.f - a, b1 = 1.f - b, g1 = 1.f - g;
    const float w00 = b1 * g1, w10 = b * g1, w01 = b1 * g, w11 = b * g;
    w[0] = a1 * w00; w[1] = a * w00;
    w[2] = a1 * w10; w[3] = a * w10;
    w[4] = a1 * w01; w[5] = a * w01;
    w[6] = a1 * w11; w[7] = a * w11;
}

// Weights of a footprint: frac(u) = u - floor(u), exact for u >= 0 (the
// box); v_fract_f32 computes it in one instruction.
__device__ __forceinline__ void fp_weights(const Footprint &f, float w[8])
{
    tri_weights(__builtin_amdgcn_fractf(f.u), __builtin_amdgcn_fractf(f.v), __builtin_amdgcn_fractf(f.w), w);
}

template <int F, int LB, bool BUF>
__device__ __forceinline__ float sample1(const Src<BUF> &s, const Footprint &f)
{
    float w[8];
    float4 t[8];
    load_taps<F, LB, BUF>(s, f, t);
    fp_weights(f, w);
    float r = w[0] * t[0].w;
#pragma unroll
    for (int k = 1; k < 8; ++k) r = fmaf(w[k], t[k].w, r);
    return r;
}

// Generic path: runtime format and brick size.
__device__ __forceinline__ float4 sample_any(const TexDesc &t, float w0, float w1, float w2)
{
    const float u = fmaf(w0, t.k0, 0.5f), v = fmaf(w1, t.k1, 0.5f), w = fmaf(w2, t.k2, 0.5f);
    const float fu = floorf(u), fv = floorf(v), fw = floorf(w);
    const uint32_t X = (uint32_t)(int)fu, Y = (uint32_t)(int)fv, Z = (uint32_t)(int)fw;
    const int lb = t.lb;
    const uint32_t M = (1u << lb) - 1u, E = (1u << lb) + 1u, T = (uint32_t)texel_bytes(t.fmt);
    const uint32_t brick = ((Z >> lb) * t.nby + (Y >> lb)) * t.nbx + (X >> lb);
    const uint32_t local = ((Z & M) * E + (Y & M)) * E + (X & M);
    const char *p = (const char *)t.base + (uint64_t)brick * t.brick_bytes + (uint64_t)local * T;
    float wt[8];
    tri_weights(u - fu, v - fv, w - fw, wt);
    float4 r = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int k = 0; k < 8; ++k) {
        const uint32_t off = ((k & 1) + ((k >> 1) & 1) * E + (k >> 2) * E * E) * T;
        const float4 c = fetch_any(t.fmt, p + off);
        r.x = fmaf(wt[k], c.x, r.x);
        r.y = fmaf(wt[k], c.y, r.y);
        r.z = fmaf(wt[k], c.z, r.z);
        r.w = fmaf(wt[k], c.w, r.w);
    }
    return r;
}

// ---------------------------------------------------------------------------
// Per-frame constants (uniforms after host-side FP64 preparation).
struct FrameConst {
    float prow[8];    // rows 0-1 of inverse(P_gl)          (volume.frag.glsl:50)
    float rot[9];     // 3x3 block of inverse(V_gl)         (volume.frag.glsl:52)
    float o[3];       // camera_pos
    float bmin[3], bmax[3], ext[3];   // ext = bmax - bmin in float (:26)
    float step;       // step_size
    float alpha_k;    // log2(e) * step_size / reference_step_size  (:101)
    float ka, kd;     // ambient_light, diffuse_light       (:110)
    float L[3];       // normalize(light_target - light_position) (:107)
    float tau;        // early-termination alpha            (:87)
    float fW, fH;
    int W, H;
    int max_steps;
    int ok;           // 0: camera unset or singular matrices -> every pixel 0
    int L_ok;         // 0: zero-length light vector -> diffuse term 0
    uint32_t clear[4];  // framebuffer clear colour (8-bit per channel)
    int blend;          // 1: SRC_ALPHA, ONE_MINUS_SRC_ALPHA over the clear colour
    int count_shaded;   // counting instances: count only samples that load texels
    uint8_t *touched;   // counting instances: set to 1 for every brick a sample loads from (or null)
};

// One ray per pixel, produced by the setup kernel.
struct __align__(16) RayRec {
    float p0x, p0y, p0z;  // first sample position (entry point or camera)
    int nlim;             // iterations to run (0: the ray misses the box)
    float dsx, dsy, dsz;  // ray_dir * step_size
    int pad;
};

// Ray setup (volume.vert.glsl:8; volume.frag.glsl:47-68, 71-82), run inline
// by the march kernels (once per ray) and by the block-ordering pass.
// Pixel (px, py), py = 0 the bottom row.  Positions use separately rounded
// products and sums (no fused multiply-add), as the shader states them.
__device__ __forceinline__ RayRec ray_setup(const FrameConst &fc, int px, int py)
{
    RayRec r;
    r.p0x = r.p0y = r.p0z = 0.f;
    r.dsx = r.dsy = r.dsz = 0.f;
    r.nlim = 0;
    r.pad = 0;
    if (fc.ok) {
        // A1: pixel centre -> NDC
        const float ux = ((float)px + 0.5f) / fc.fW, uy = ((float)py + 0.5f) / fc.fH;
        const float nx = ux * 2.f - 1.f, ny = uy * 2.f - 1.f;
        // A2: eye direction: inverse(P) * (ndc, -1, 1), then (x, y, -1, 0)
        const float ex = fc.prow[0] * nx + fc.prow[1] * ny - fc.prow[2] + fc.prow[3];
        const float ey = fc.prow[4] * nx + fc.prow[5] * ny - fc.prow[6] + fc.prow[7];
        // A3: world direction
        const float w0 = fc.rot[0] * ex + fc.rot[1] * ey - fc.rot[2];
        const float w1 = fc.rot[3] * ex + fc.rot[4] * ey - fc.rot[5];
        const float w2 = fc.rot[6] * ex + fc.rot[7] * ey - fc.rot[8];
        const float wn = 1.0f / sqrtf(w0 * w0 + w1 * w1 + w2 * w2);
        const float d[3] = {w0 * wn, w1 * wn, w2 * wn};
        // A4: slab test
        float tn = -INFINITY, tf = INFINITY;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float inv = 1.0f / d[k];
            const float t0 = (fc.bmin[k] - fc.o[k]) * inv, t1 = (fc.bmax[k] - fc.o[k]) * inv;
            float lo = fminf(t0, t1), hi = fmaxf(t0, t1);
            if (t0 != t0 || t1 != t1) { lo = -INFINITY; hi = INFINITY; }
            tn = fmaxf(tn, lo);
            tf = fminf(tf, hi);
        }
        if (tn <= tf && tf > 0.f) {
            tn = fmaxf(tn, 0.f);
            // A5: entry point and step vector
            r.p0x = __fadd_rn(fc.o[0], __fmul_rn(d[0], tn));
            r.p0y = __fadd_rn(fc.o[1], __fmul_rn(d[1], tn));
            r.p0z = __fadd_rn(fc.o[2], __fmul_rn(d[2], tn));
            r.dsx = __fmul_rn(d[0], fc.step);
            r.dsy = __fmul_rn(d[1], fc.step);
            r.dsz = __fmul_rn(d[2], fc.step);
            // Iterations: every in-box sample lies within 1.0625*(tf-tn)/step
            // + 16 steps of the entry point (margin for FP32 stepping drift);
            // later iterations of the shader's loop are out-of-box no-ops.
            const float span = (tf - tn) / fc.step * 1.0625f + 16.f;
            r.nlim = span < (float)fc.max_steps ? (int)span : fc.max_steps;
        }
    }
    return r;
}

// K1 -- the dispatch order of a cost-ordered frame: `order`, the logical block
// of each dispatch position of the first `head_rows` block rows (a multiple of
// 8; 2^lbw x 2^lbh pixels each, ntx per row).  One thread block per dispatch
// class (block row mod 8) files the class's `cap` blocks under the largest
// iteration bound of three rays of each (two corners and the middle) in
// kOrderBuckets lists, counted in LDS, and reads them back in order
// (ordered_block).  Ray setup bounds it; every pixel's ray, and one atomic on
// global memory per block, took twice as long (4096 blocks 12.6 us, 8192 22).
static constexpr int kOrderThreads = 1024;
static __global__ void __launch_bounds__(kOrderThreads)
k_order_blocks(const FrameConst fc, uint32_t *order, uint32_t *slots, int ntx, int head_rows, int cap, int lbw,
               int lbh)
{
    __shared__ uint32_t s_cnt[8 * kOrderBuckets];   // of this class only
    const int cls = blockIdx.x;
    if (threadIdx.x < 8 * kOrderBuckets) s_cnt[threadIdx.x] = 0u;
    __syncthreads();
    for (int k = threadIdx.x; k < cap; k += kOrderThreads) {
        const int tx = k % ntx, ty = (k / ntx) * 8 + cls;
        int key = 0;
        for (int c = 0; c < 3; ++c) {
            const int x = min((tx << lbw) + (((1 << lbw) - 1) * c >> 1), fc.W - 1),
                      y = min((ty << lbh) + (((1 << lbh) - 1) * c >> 1), fc.H - 1);
            key = max(key, ray_setup(fc, x, y).nlim);
        }
        const int q = cls * kOrderBuckets + order_bucket(key, fc.max_steps);
        slots[(uint64_t)q * (uint64_t)cap + atomicAdd(&s_cnt[q], 1u)] = (uint32_t)(ty * ntx + tx);
    }
    __syncthreads();   // the slots of this class were written by this block
    for (int k = threadIdx.x; k < cap; k += kOrderThreads) {
        const int b = k * 8 + cls;
        order[b] = (uint32_t)ordered_block(b, head_rows * ntx, s_cnt, slots, cap);
    }
}

// Stored RGBA8 (manager.py:29-31, 212-220): the source colour is clamped
// and converted to 8 bits (Cq, Aq), then blended with (SRC_ALPHA,
// ONE_MINUS_SRC_ALPHA) over the 8-bit clear colour D in fixed point:
// out = round((S*Aq + D*(255 - Aq)) / 255) per channel.  With the
// reference's clear colour 0 this is rgb = Cq*Aq/255, a = Aq*Aq/255.
__device__ __forceinline__ uint32_t unorm8(float x)
{
    x = fminf(fmaxf(x, 0.f), 1.f);  // NaN -> 0
    return (uint32_t)floorf(fmaf(x, 255.f, 0.5f));
}
__device__ __forceinline__ uchar4 blend_store(const FrameConst &fc, float c0, float c1, float c2, float a)
{
    const uint32_t aq = unorm8(a);
    const uint32_t q0 = unorm8(c0), q1 = unorm8(c1), q2 = unorm8(c2);
    if (!fc.blend) return make_uchar4((unsigned char)q0, (unsigned char)q1, (unsigned char)q2, (unsigned char)aq);
    const uint32_t ia = 255u - aq;
    return make_uchar4((unsigned char)((q0 * aq + fc.clear[0] * ia + 127u) / 255u),
                       (unsigned char)((q1 * aq + fc.clear[1] * ia + 127u) / 255u),
                       (unsigned char)((q2 * aq + fc.clear[2] * ia + 127u) / 255u),
                       (unsigned char)((aq * aq + fc.clear[3] * ia + 127u) / 255u));
}

// How the normal sampler is served in a march kernel instance.
enum NormalMode : int {
    NM_SAME = 0,   // normals interleaved in the scalar volume's texels
    NM_ALIAS = 1,  // the scalar volume read as (rho, 0, 0)
    NM_ZERO = 2,   // unbound: normal = 0 -> diffuse term 0
    NM_ANY = 3     // generic: scalar and normal from any volumes/formats
};

// LUT lookup at (rho, 0.5) with u = rho*N - 1/2, clamp to edge
// (manager.py:163-181; volume.frag.glsl:96).  `lut` holds, per entry i, the
// pair (entry i, entry i+1 - entry i) (difference 0 after the last), so that
// clamping u to [0, N-1] gives both edge cases and one fma per channel.  The
// clamp is one v_med3_f32 (which maps a NaN to min(0, N-1) = 0, as
// fminf(fmaxf(NaN, 0), N-1) does), so u >= 0: truncation is floor and
// v_fract_f32 gives u - floor(u) exactly.
__device__ __forceinline__ float4 lut_sample(const float4 *lut, float fn1, float fn, float rho)
{
    const float u = __builtin_amdgcn_fmed3f(fmaf(rho, fn, -0.5f), 0.f, fn1);
    const float a = __builtin_amdgcn_fractf(u);
    const int i = (int)u;
    const float4 v = lut[2 * i], d = lut[2 * i + 1];
    return make_float4(fmaf(a, d.x, v.x), fmaf(a, d.y, v.y), fmaf(a, d.z, v.z), fmaf(a, d.w, v.w));
}

static constexpr int kLutLdsMax = 2048;  // entries; 2 x 16 B each in LDS

// Clamp-to-edge LUT lookup from global memory (generic path).
__device__ __forceinline__ float4 lut_global(const float4 *__restrict__ lut, int n, float fn1, float fn, float rho)
{
    const float u = fminf(fmaxf(fmaf(rho, fn, -0.5f), 0.f), fn1);
    const float fu = floorf(u);
    const int i0 = (int)fu, i1 = min(i0 + 1, n - 1);
    const float a = u - fu;
    const float4 v0 = lut[i0], v1 = lut[i1];
    return make_float4(fmaf(a, v1.x - v0.x, v0.x), fmaf(a, v1.y - v0.y, v0.y), fmaf(a, v1.z - v0.z, v0.z),
                       fmaf(a, v1.w - v0.w, v0.w));
}

// One sample's contribution (volume.frag.glsl:96-115): Beer-Lambert opacity
// correction 1 - exp(-alpha*step/ref), ambient + Lambert with the zero-vector
// rule (a normal of zero or subnormal length has no direction and gives no
// diffuse light), front-to-back composite.
__device__ __forceinline__ float lambert(const FrameConst &fc, float n0, float n1, float n2)
{
    // v_rsq_f32 without the subnormal-input rescaling of rsqrtf: the result
    // is only used for nn >= FLT_MIN, where the two agree
    const float nn = fmaf(n0, n0, fmaf(n1, n1, n2 * n2));
    const float dt = fmaf(n0, fc.L[0], fmaf(n1, fc.L[1], n2 * fc.L[2])) * __builtin_amdgcn_rsqf(nn);
    return (fc.L_ok && nn >= 1.17549435e-38f) ? fmaxf(dt, 0.f) : 0.f;
}

// The composite with the light factor lam = ka + kd * diffuse given.
__device__ __forceinline__ void composite_lam(const FrameConst &fc, const float4 &q, float lam, float &C0,
                                              float &C1, float &C2, float &A)
{
    const float a = 1.f - __builtin_amdgcn_exp2f(-(q.w * fc.alpha_k));
    const float ta = (1.f - A) * a;
    const float tl = ta * lam;
    C0 = fmaf(tl, q.x, C0);
    C1 = fmaf(tl, q.y, C1);
    C2 = fmaf(tl, q.z, C2);
    A = A + ta;
}

__device__ __forceinline__ void composite_diff(const FrameConst &fc, const float4 &q, float diff, float &C0,
                                               float &C1, float &C2, float &A)
{
    // v_exp_f32 without the subnormal-result rescaling of exp2f: when
    // exp2(-x) is subnormal, 1 - exp2(-x) rounds to 1 either way
    const float a = 1.f - __builtin_amdgcn_exp2f(-(q.w * fc.alpha_k));
    const float lam = fmaf(fc.kd, diff, fc.ka);
    const float ta = (1.f - A) * a;
    const float tl = ta * lam;
    C0 = fmaf(tl, q.x, C0);
    C1 = fmaf(tl, q.y, C1);
    C2 = fmaf(tl, q.z, C2);
    A = A + ta;
}

template <int NM>
__device__ __forceinline__ void composite(const FrameConst &fc, const float4 &q, float n0, float n1, float n2,
                                          float &C0, float &C1, float &C2, float &A)
{
    composite_diff(fc, q, NM != NM_ZERO ? lambert(fc, n0, n1, n2) : 0.f, C0, C1, C2, A);
}

// K2 -- march and composite (volume.frag.glsl:84-121), P adjacent lanes per
// ray (march_lanes; one in most large frames).  A block of 4 waves covers
// 16x16, 16x8 or 8x8 pixels; each wave64 an 8x8, 8x4 or 4x4 tile.  Blocks
// are dispatched round-robin over the 8 XCDs (block b on XCD (b + c) mod 8,
// c varying from launch to launch), and each XCD runs its blocks in order.
// The block -> tile mapping deals block rows to the XCDs in turn
// (XCD of b & 7 takes rows b & 7, 8 + (b & 7), ...): the work per row varies
// strongly over the image (where the rays cross dense matter), so
// contiguous bands per XCD left some XCDs idle for half the frame, while
// interleaved rows give every XCD an even share, and its L2 still sees whole
// rows; within a row the start is rotated (row_rotation) to spread the
// columns over the XCD's compute units.  Rows past the last multiple of 8
// keep the plain order.  With `order` (a cost-ordered frame,
// k_order_blocks), each XCD's class of rows is taken in decreasing order of
// its blocks' iteration bounds instead, so that the long blocks start in the
// first round of resident blocks rather than after it.  A wave runs
// while any of its rays is live; a ray stops at its iteration bound
// (max_steps at most), when its alpha reaches tau, or when it leaves the box.
//
// What bounds it: in frames of more rays than stay resident, VALU issue (about
// 100 instructions a shaded sample) and, for 16-byte texels, the L1; in smaller
// ones the chain of one ray's samples (about 1000 cycles each for a wave
// alone on its SIMD, 500 of them VALU), which lanes shorten.
//
// In-box test (:88-92): fl((p - bmin)/ext) lies in [0, 1] exactly when
// fl(p - bmin) lies in [0, ext] (for ext > 0 the quotient of a larger
// difference rounds above 1), so the test needs no division.  The in-box
// samples of a ray are one contiguous run (each coordinate moves
// monotonically), so the loop skips the leading outside samples (the entry
// point may round outside) and ends at the first outside sample after them.
//
// Transparent bricks (SKIP instances): `skip[brick]`, the brick's clearance
// (hvr_rules.h), is not 0 when every LUT
// entry that a density of the brick can weight is transparent (alpha 0 and
// a finite colour).  Such a sample contributes exactly nothing
// (C += (1-A)*lambda*rgb*0, A += (1-A)*0; lambda is finite because the
// Lambert term is 0 or max(dot, 0) with fmaxf dropping a NaN), so it is
// counted and stepped over without loading texels.  Where every ray of the
// wave is in a brick of clearance 2 and more, the wave walks on as far as the
// least of them allows without looking at flags or the box (the positions are
// the same additions; a sample past the box ends the ray as before): 5
// instructions a step instead of 26.  Letting each ray leap by itself spread
// the rays of a wave over different depths, and the texels they then no
// longer shared cost more than the leaps gained (512^3 batch 7.77 -> 8.2 ms;
// the whole wave 7.77 -> 7.44).
__device__ __forceinline__ bool inbox(const FrameConst &fc, float wx, float wy, float wz)
{
    return (wz >= 0.f) & (wz <= fc.ext[2]) & (wy >= 0.f) & (wy <= fc.ext[1]) & (wx >= 0.f) & (wx <= fc.ext[0]);
}

// 1 / the texels a ray may move per step along any axis (leap_rate), rays
// walking texture x, y, z along world z, y, x.
__device__ __forceinline__ float leap_inverse(const FrameConst &fc, const TexDesc &t, const RayRec &r)
{
    const float x = leap_rate(r.dsx, t.k2, fmaxf(fabsf(fc.bmin[0]), fabsf(fc.bmax[0]))),
                y = leap_rate(r.dsy, t.k1, fmaxf(fabsf(fc.bmin[1]), fabsf(fc.bmax[1]))),
                z = leap_rate(r.dsz, t.k0, fmaxf(fabsf(fc.bmin[2]), fabsf(fc.bmax[2])));
    return 1.f / fmaxf(fmaxf(x, y), z);
}

// Exchange inside groups of P adjacent lanes (P = 2 or 4) with quad_perm: the
// value of the group's lane K, its first lane's, and whether any lane's is not 0.
template <int P, int K>
__device__ __forceinline__ int group_lane(int v)
{
    constexpr int perm = P == 4 ? K * 0x55 : (K | K << 2 | (K + 2) << 4 | (K + 2) << 6);
    return __builtin_amdgcn_mov_dpp(v, perm, 0xf, 0xf, true);
}
template <int P, int K>
__device__ __forceinline__ float group_lane(float v)
{
    return __int_as_float(group_lane<P, K>(__float_as_int(v)));
}
template <int P>
__device__ __forceinline__ int group_first(int v)
{
    return group_lane<P, 0>(v);
}
template <int P>
__device__ __forceinline__ bool group_any(int v)
{
    v |= __builtin_amdgcn_mov_dpp(v, 0xb1, 0xf, 0xf, true);             // [1, 0, 3, 2]
    if constexpr (P == 4) v |= __builtin_amdgcn_mov_dpp(v, 0x4e, 0xf, 0xf, true);   // [2, 3, 0, 1]
    return v != 0;
}
// The group's samples in order, lane 0's first: what composite_diff adds for
// each, in every lane.  A lane without a sample (`now` false) has a, lam and q
// zero, which changes nothing while the alphas are finite.  Terms of the
// fused multiply-adds are read from the other lanes by the add itself.
template <int P, int K>
__device__ __forceinline__ void add_color(float tl, float q0, float q1, float q2, float &C0, float &C1, float &C2)
{
    // s_nop: a lane's q may have been written by the instruction before.  & : the
    // first colours are written while q1, q2 and tl are still to be read, so none
    // of those may share an accumulator's register, also where both hold the same
    // value.
#define HVR_FMAC3(QP)                                                           \
    asm volatile("s_nop 1\n\tv_fmac_f32_dpp %0, %3, %6 " QP " row_mask:0xf bank_mask:0xf\n\t" \
        "v_fmac_f32_dpp %1, %4, %6 " QP " row_mask:0xf bank_mask:0xf\n\t"               \
        "v_fmac_f32_dpp %2, %5, %6 " QP " row_mask:0xf bank_mask:0xf"                   \
        : "+&v"(C0), "+&v"(C1), "+&v"(C2)                                           \
        : "v"(q0), "v"(q1), "v"(q2), "v"(tl))
    if constexpr (P == 2 && K == 0) HVR_FMAC3("quad_perm:[0,0,2,2]");
    else if constexpr (P == 2) HVR_FMAC3("quad_perm:[1,1,3,3]");
    else if constexpr (K == 0) HVR_FMAC3("quad_perm:[0,0,0,0]");
    else if constexpr (K == 1) HVR_FMAC3("quad_perm:[1,1,1,1]");
    else if constexpr (K == 2) HVR_FMAC3("quad_perm:[2,2,2,2]");
    else HVR_FMAC3("quad_perm:[3,3,3,3]");
#undef HVR_FMAC3
}
template <int P, int K>
__device__ __forceinline__ void group_alpha(float a, float lam, float A, float (&tl)[P], float (&al)[P])
{
    const float ta = (1.f - A) * group_lane<P, K>(a);
    tl[K] = ta * group_lane<P, K>(lam);
    al[K] = A + ta;
    if constexpr (K + 1 < P) group_alpha<P, K + 1>(a, lam, al[K], tl, al);
}
template <int P, int K>
__device__ __forceinline__ void group_color(const float (&tl)[P], float q0, float q1, float q2, float &C0, float &C1,
                                            float &C2)
{
    add_color<P, K>(tl[K], q0, q1, q2, C0, C1, C2);
    if constexpr (K + 1 < P) group_color<P, K + 1>(tl, q0, q1, q2, C0, C1, C2);
}
// The same with each sample taken only while alpha is below its lane's tau
// (-infinity in a lane without a sample).
template <int P, int K>
__device__ __forceinline__ void group_select(float tau, float a, float lam, float q0, float q1, float q2, float &C0,
                                             float &C1, float &C2, float &A)
{
    const float ta = (1.f - A) * group_lane<P, K>(a);
    const float tl = ta * group_lane<P, K>(lam);
    const float c0 = fmaf(tl, group_lane<P, K>(q0), C0), c1 = fmaf(tl, group_lane<P, K>(q1), C1),
                c2 = fmaf(tl, group_lane<P, K>(q2), C2), al = A + ta;
    const bool take = A < group_lane<P, K>(tau);
    C0 = take ? c0 : C0;
    C1 = take ? c1 : C1;
    C2 = take ? c2 : C2;
    A = take ? al : A;
    if constexpr (K + 1 < P) group_select<P, K + 1>(tau, a, lam, q0, q1, q2, C0, C1, C2, A);
}
template <int P>
__device__ __forceinline__ void composite_group(float tau, bool now, float a, float lam, float q0, float q1, float q2,
                                                float &C0, float &C1, float &C2, float &A)
{
    float tl[P], al[P];
    group_alpha<P, 0>(a, lam, A, tl, al);
    // every ray of the wave still below tau before its last sample, with
    // finite alphas: no sample is dropped
    bool plain = true;
#pragma unroll
    for (int k = 0; k + 1 < P; ++k) plain &= fabsf(al[k]) < tau;
    if (__ballot(!plain) == 0) {
        group_color<P, 0>(tl, q0, q1, q2, C0, C1, C2);
        A = al[P - 1];
    } else {
        group_select<P, 0>(now ? tau : -INFINITY, a, lam, q0, q1, q2, C0, C1, C2, A);
    }
}

// The march of one ray (volume.frag.glsl:84-121) from its setup record:
// accumulated colour (C0, C1, C2), alpha A, and the number of composited
// samples ns (COUNT).  s_lut: the LUT with its differences in LDS (lut_sample).
// GATE: interpolate and light the normal only for samples of non-zero
// alpha (fewer instructions where the march is instruction-bound; the
// result is identical either way).
template <int SF, int NM, int LB, bool COUNT, bool SKIP, bool BUF, bool GATE = false, int P = 1>
__device__ __forceinline__ void march_ray(const FrameConst &fc, const TexDesc &ts, const TexDesc &tn,
                                          const float4 *__restrict__ lut_g, int lut_n, const float4 *s_lut,
                                          const RayRec &r, const uint8_t *__restrict__ skip,
                                          float &C0, float &C1, float &C2, float &A, uint32_t &ns)
{
    float x = r.p0x, y = r.p0y, z = r.p0z;
    const float fn = (float)lut_n, fn1 = (float)(lut_n - 1);
    constexpr float u8k = fmt_u8_scalar(SF) ? 1.0f / 255.0f : 1.0f;
    constexpr int T = texel_bytes(SF);
    const int nlim = r.nlim;
    int i = 0;
    // leading samples outside the box
    for (; i < nlim; ++i) {
        if (inbox(fc, x - fc.bmin[0], y - fc.bmin[1], z - fc.bmin[2])) break;
        x = __fadd_rn(x, r.dsx);
        y = __fadd_rn(y, r.dsy);
        z = __fadd_rn(z, r.dsz);
    }
    if constexpr (NM == NM_ANY || SF == TF_NONE) {
        // the in-box run, generic texture access
        for (; i < nlim; ++i) {
            if (!(A < fc.tau)) break;
            const float wx = x - fc.bmin[0], wy = y - fc.bmin[1], wz = z - fc.bmin[2];
            if (!inbox(fc, wx, wy, wz)) break;
            if constexpr (COUNT) ++ns;
            // texture x <- world z (size s0), y <- world y (s1), z <- world x (s2)
            float rho = 0.f, n0 = 0.f, n1 = 0.f, n2 = 0.f;
            if constexpr (NM == NM_ANY) {
                if (ts.base) {
                    const float4 t = sample_any(ts, wz, wy, wx);
                    rho = ts.role == 0 ? t.w : t.x;
                }
                if (tn.base) {
                    const float4 t = sample_any(tn, wz, wy, wx);
                    if (tn.role == 1) { n0 = t.x; n1 = t.y; n2 = t.z; }
                    else n0 = t.w;
                }
            }
            const float4 q = NM == NM_ANY ? lut_global(lut_g, lut_n, fn1, fn, rho)
                                          : lut_sample(s_lut, fn1, fn, rho);
            composite<NM>(fc, q, n0, n1, n2, C0, C1, C2, A);
            x = __fadd_rn(x, r.dsx);
            y = __fadd_rn(y, r.dsy);
            z = __fadd_rn(z, r.dsz);
        }
    } else {
        const Src<BUF> src(ts);
        // one sample's contribution from its footprint (coordinates and
        // brick; the address is completed here)
        auto shade = [&](const Footprint &fb) {
            Footprint f = fb;
            footprint_addr<T, LB, BUF>(ts, f);
            if constexpr (COUNT) {
                if (fc.touched) fc.touched[f.brick] = 1;   // the bricks the frame reads
            }
            if constexpr (NM == NM_SAME) {
                constexpr int T = texel_bytes(SF);
                uint32_t raw[4][T / 2];
                load_pairs<SF, LB, BUF>(src, f, raw);
                float w[8];
                fp_weights(f, w);
                const float rho = interp_scalar<SF>(raw, w) * u8k;
                if constexpr (GATE) {
                    // Normals only for a non-zero alpha: with alpha 0 the
                    // sample adds (1-A)*0*lambda = 0 for any finite lambda
                    // (the Lambert term is 0 or fmaxf(dot, 0)), so skipping
                    // the normal changes nothing; the texel loads are shared.
                    const float4 q = lut_sample(s_lut, fn1, fn, rho);
                    float lam = fc.ka;   // fma(kd, 0, ka) = ka exactly (kd finite)
                    if (q.w != 0.f) {
                        const float3 n = interp_normal<SF>(raw, w);
                        lam = fmaf(fc.kd, lambert(fc, n.x, n.y, n.z), fc.ka);
                    }
                    composite_lam(fc, q, lam, C0, C1, C2, A);
                } else {
                    const float3 n = interp_normal<SF>(raw, w);
                    const float4 q = lut_sample(s_lut, fn1, fn, rho);
                    composite_diff(fc, q, lambert(fc, n.x, n.y, n.z), C0, C1, C2, A);
                }
            } else {
                const float rho = sample1<SF, LB, BUF>(src, f) * u8k;
                const float4 q = lut_sample(s_lut, fn1, fn, rho);
                composite<NM>(fc, q, NM == NM_ALIAS ? rho : 0.f, 0.f, 0.f, C0, C1, C2, A);
            }
        };
        // The in-box run tests one bound per axis.  Per axis, with s = -1
        // where the step is negative (else +1), the run walks q = s*p by
        // s*ds >= 0 and forms a = fl(q - s*bmin): round-to-nearest commutes
        // with negation, so q is exactly s times the shader's position and
        // a = s*fl(p - bmin).  fl is monotonic, so a never decreases; the
        // run starts at a sample that passed the two-sided test, so a's
        // lower bound stays met and only a <= (s > 0 ? ext : 0) is tested.
        // In the box, p - bmin >= 0, so the footprint takes |a| (a free
        // source modifier) as fl(p - bmin).
        const float sx = r.dsx < 0.f ? -1.f : 1.f, sy = r.dsy < 0.f ? -1.f : 1.f,
                    sz = r.dsz < 0.f ? -1.f : 1.f;
        x *= sx;
        y *= sy;
        z *= sz;
        const float dqx = sx * r.dsx, dqy = sy * r.dsy, dqz = sz * r.dsz;
        const float bqx = -(sx * fc.bmin[0]), bqy = -(sy * fc.bmin[1]), bqz = -(sz * fc.bmin[2]);
        const float lx = sx > 0.f ? fc.ext[0] : 0.f, ly = sy > 0.f ? fc.ext[1] : 0.f,
                    lz = sz > 0.f ? fc.ext[2] : 0.f;
        if constexpr (P > 1) {
            // P adjacent lanes march one ray: lane j holds samples j, P + j, ...
            // of the in-box run (each position the sum of the same additions
            // as a single lane's), every lane the ray's colour.  Lanes of a
            // group leave the loop together.
            static_assert(!COUNT && !GATE && (P == 2 || P == 4), "");
            const int j = (int)threadIdx.x & (P - 1);
            auto advance = [&](int n) {
#pragma unroll
                for (int k = 0; k < n; ++k) {
                    x = __fadd_rn(x, dqx);
                    y = __fadd_rn(y, dqy);
                    z = __fadd_rn(z, dqz);
                }
            };
            for (int k = 1; k < P; ++k)
                if (j >= k) advance(1);
            i += j;
            float ax = __fadd_rn(x, bqx), ay = __fadd_rn(y, bqy), az = __fadd_rn(z, bqz);
            bool in = i < nlim && (az <= lz) & (ay <= ly) & (ax <= lx);
            Footprint fa = footprint_brick<LB, BUF>(ts, in ? fabsf(az) : 0.f, in ? fabsf(ay) : 0.f,
                                                    in ? fabsf(ax) : 0.f),
                      fb;
            uint32_t flag = SKIP ? ld_global(skip + fa.brick) : 0u;
            bool live = group_first<P>((int)in) != 0;
            const float inv = SKIP ? leap_inverse(fc, ts, r) : 0.f;
            auto step = [&](const Footprint &f, Footprint &g) {
                if constexpr (SKIP) {
                    if (__ballot(in && flag < 2) == 0) {
                        int n = in ? leap_steps((int)flag, LB, inv) : 1 << 20;   // the group's first lane is in
                        while (__ballot(n < 4) == 0) {
                            advance(4);
                            i += 4;
                            n -= 4;
                        }
                    }
                }
                const bool now = SKIP ? in && flag == 0 : in;
                i += P;
                advance(P);
                ax = __fadd_rn(x, bqx);
                ay = __fadd_rn(y, bqy);
                az = __fadd_rn(z, bqz);
                in = i < nlim && (az <= lz) & (ay <= ly) & (ax <= lx);
                g = footprint_brick<LB, BUF>(ts, fabsf(az), fabsf(ay), fabsf(ax));
                if (SKIP && in && g.brick != f.brick) flag = ld_global(skip + g.brick);
                if (group_any<P>((int)now)) {
                    float a = 0.f, lam = 0.f, q0 = 0.f, q1 = 0.f, q2 = 0.f;
                    if (now) {
                        Footprint h = f;
                        footprint_addr<T, LB, BUF>(ts, h);
                        float4 q;
                        float diff = 0.f;
                        if constexpr (NM == NM_SAME) {
                            uint32_t raw[4][T / 2];
                            load_pairs<SF, LB, BUF>(src, h, raw);
                            float w[8];
                            fp_weights(h, w);
                            const float rho = interp_scalar<SF>(raw, w) * u8k;
                            const float3 n = interp_normal<SF>(raw, w);
                            q = lut_sample(s_lut, fn1, fn, rho);
                            diff = lambert(fc, n.x, n.y, n.z);
                        } else {
                            const float rho = sample1<SF, LB, BUF>(src, h) * u8k;
                            q = lut_sample(s_lut, fn1, fn, rho);
                            if constexpr (NM == NM_ALIAS) diff = lambert(fc, rho, 0.f, 0.f);
                        }
                        a = 1.f - __builtin_amdgcn_exp2f(-(q.w * fc.alpha_k));
                        lam = fmaf(fc.kd, diff, fc.ka);
                        q0 = q.x;
                        q1 = q.y;
                        q2 = q.z;
                    }
                    composite_group<P>(fc.tau, now, a, lam, q0, q1, q2, C0, C1, C2, A);
                }
                live = group_first<P>((int)in) != 0;
            };
            while (live && A < fc.tau) {
                step(fa, fb);
                if (!(live && A < fc.tau)) break;
                step(fb, fa);
            }
        } else if constexpr (!SKIP) {
            // the in-box run
            for (; i < nlim; ++i) {
                if (!(A < fc.tau)) break;
                const float ax = __fadd_rn(x, bqx), ay = __fadd_rn(y, bqy), az = __fadd_rn(z, bqz);
                if (!((az <= lz) & (ay <= ly) & (ax <= lx))) break;
                if constexpr (COUNT) ++ns;
                shade(footprint_brick<LB, BUF>(ts, fabsf(az), fabsf(ay), fabsf(ax)));
                x = __fadd_rn(x, dqx);
                y = __fadd_rn(y, dqy);
                z = __fadd_rn(z, dqz);
            }
        } else {
            // The in-box run with transparent bricks stepped over: a sample
            // in a transparent brick is counted without loading texels.  The
            // flag is loaded again only when the sample's brick changes (a
            // brick spans several steps), which saves most flag loads.  Each
            // iteration first advances to the next sample (its position, box
            // test and brick: none depends on the composite) and issues that
            // sample's flag load, then shades the current sample: the flag
            // load is in flight together with the current sample's texel
            // loads, so a wave waits for memory once per iteration, not
            // twice (some lane of a wave changes brick on most iterations).
            // A footprint outside the box is never used.
            float ax = __fadd_rn(x, bqx), ay = __fadd_rn(y, bqy), az = __fadd_rn(z, bqz);
            bool in = i < nlim && (az <= lz) & (ay <= ly) & (ax <= lx);
            // Unrolled by two, two footprints trading roles (no register
            // copies between iterations).  The flag held is always that
            // of the current sample's brick.
            Footprint fa = footprint_brick<LB, BUF>(ts, in ? fabsf(az) : 0.f, in ? fabsf(ay) : 0.f,
                                                    in ? fabsf(ax) : 0.f),
                      fb;
            uint32_t flag = ld_global(skip + fa.brick);
            bool clear = in && flag != 0;
            const float inv = leap_inverse(fc, ts, r);
            // one sample: f the current sample's footprint, g receives the next one's
            auto step = [&](const Footprint &f, Footprint &g) {
                if constexpr (!COUNT) {
                    if (__ballot(!(clear && flag > 1)) == 0) {
                        int n = leap_steps((int)flag, LB, inv);
                        while (__ballot(n < 4) == 0) {
#pragma unroll
                            for (int k = 0; k < 4; ++k) {
                                x = __fadd_rn(x, dqx);
                                y = __fadd_rn(y, dqy);
                                z = __fadd_rn(z, dqz);
                            }
                            i += 4;
                            n -= 4;
                        }
                    }
                }
                ++i;
                x = __fadd_rn(x, dqx);
                y = __fadd_rn(y, dqy);
                z = __fadd_rn(z, dqz);
                ax = __fadd_rn(x, bqx);
                ay = __fadd_rn(y, bqy);
                az = __fadd_rn(z, bqz);
                const bool in_next = i < nlim && (az <= lz) & (ay <= ly) & (ax <= lx);
                g = footprint_brick<LB, BUF>(ts, fabsf(az), fabsf(ay), fabsf(ax));
                if (in_next && g.brick != f.brick) flag = ld_global(skip + g.brick);
                if (!clear) shade(f);
                if constexpr (COUNT) ns += (fc.count_shaded && clear) ? 0u : 1u;
                in = in_next;
                clear = in && flag != 0;
            };
            while (in && A < fc.tau) {
                step(fa, fb);
                if (!(in && A < fc.tau)) break;
                step(fb, fa);
            }
        }
    }
}

// Load the LUT of n entries, each followed by its difference to the next
// entry (0 after the last), into LDS.
__device__ __forceinline__ void load_lut_lds(const float4 *__restrict__ lut_g, int n, float4 *s_lut)
{
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const float4 v = ld_global(lut_g + i);
        float4 d = make_float4(0.f, 0.f, 0.f, 0.f);
        if (i + 1 < n) {
            const float4 nx = ld_global(lut_g + i + 1);
            d = make_float4(nx.x - v.x, nx.y - v.y, nx.z - v.z, nx.w - v.w);
        }
        s_lut[2 * i] = v;
        s_lut[2 * i + 1] = d;
    }
}

// Pixels of a block of four waves with P lanes per ray, as log2: a wave covers
// 8x8, 8x4 or 4x4 pixels, a block 2x2 waves.
struct MarchTile {
    int lbw, lbh;
};
__host__ __device__ constexpr MarchTile march_tile(int P) { return MarchTile{P == 4 ? 3 : 4, P == 1 ? 4 : 3}; }

template <int SF, int NM, int LB, bool COUNT, bool SKIP, bool BUF, int P = 1>
__global__ void __launch_bounds__(256)
k_march(const FrameConst fc, const TexDesc ts, const TexDesc tn, const float4 *__restrict__ lut_g,
        int lut_n, uchar4 *__restrict__ out,
        uint32_t *__restrict__ counts, const uint8_t *__restrict__ skip, int ntx, int nblocks,
        const uint32_t *__restrict__ order, int rot)
{
    extern __shared__ float4 s_lut[];
    if constexpr (NM != NM_ANY) {
        load_lut_lds(lut_g, lut_n, s_lut);
        __syncthreads();
    }
    const int b = blockIdx.x;
    const int head = ((nblocks / ntx) >> 3 << 3) * ntx;   // blocks of the first multiple-of-8 rows
    int logical = b;
    if (order) {
        if (b < head) logical = (int)order[b];   // cost-ordered (k_order_blocks)
    } else if (b < head) {
        const int j = b >> 3;   // j-th block of its XCD
        const int row = j / ntx;
        logical = (row * 8 + (b & 7)) * ntx + (j + row * rot) % ntx;
    }
    const int tx = logical % ntx, ty = logical / ntx;
    constexpr MarchTile bt = march_tile(P);
    const int wv = threadIdx.x >> 6, ray = (threadIdx.x & 63) / P;
    const int px = (tx << bt.lbw) + ((wv & 1) << (bt.lbw - 1)) + (ray & ((1 << (bt.lbw - 1)) - 1));
    const int py = (ty << bt.lbh) + ((wv >> 1) << (bt.lbh - 1)) + (ray >> (bt.lbw - 1));
    if (px >= fc.W || py >= fc.H) return;
    const int pix = py * fc.W + px;
    const RayRec r = ray_setup(fc, px, py);

    float C0 = 0.f, C1 = 0.f, C2 = 0.f, A = 0.f;
    uint32_t ns = 0;
    march_ray<SF, NM, LB, COUNT, SKIP, BUF, false, P>(fc, ts, tn, lut_g, lut_n, s_lut, r, skip, C0, C1, C2, A, ns);
    if (P == 1 || threadIdx.x % P == 0) out[pix] = blend_store(fc, C0, C1, C2, A);
    if constexpr (COUNT) counts[pix] = ns;
}

// K5 -- transparent-brick flags for one LUT.  A sample of density rho reads
// u = clamp(rho*N - 1/2, 0, N-1) and weights entry floor(u) by 1 - frac(u)
// and entry floor(u) + 1 by frac(u), so the entries with non-zero weight
// over densities in [lo, hi] are floor(u(lo)) .. ceil(u(hi)); the range is
// widened by a margin for the rounding of the interpolated density.  `nz`
// is the prefix count (N + 1 values) of entries that are not exactly
// transparent (alpha != 0, or a non-finite colour).
__device__ __forceinline__ bool brick_clear(float2 r, const int *__restrict__ nz, int n)
{
    return brick_clear_range(r.x, r.y, nz, n);
}

// The clearance (hvr_rules.h) of a tile of 8x8x8 bricks, by one block of 1024
// threads.  Whether each brick of the tile and of the kMaxClearance - 1 = 4
// bricks around it is transparent (brick_clear) makes 16x16 rows of 16 bits;
// then one thread per row: the bricks whose every neighbour within r is in
// the set are e & e << 1 & e >> 1 of those for r - 1, and the same with the
// neighbour rows in y and z through LDS.  Bits past the ends of the rows read
// as not transparent, which reaches no brick of the tile in four steps.  The
// reads of the ranges and of the LUT's prefix counts bound it (each brick's
// range is read for 8 tiles, from L2), so a block has 16 waves to keep them in
// flight: 7.6 us for the 35937 bricks of a 256^3 volume, where one thread per
// brick, without clearances, took 9.3.  s: 512 words of LDS.  Returns the transparent bricks of the tile this
// thread's row holds.
static constexpr int kClearTile = 8, kClearThreads = 1024;
__device__ __forceinline__ int clearance_tile(const float2 *__restrict__ range, const int *__restrict__ nz, int n,
                                              int nbx, int nby, int nbz, int tile, uint8_t *__restrict__ flags,
                                              uint32_t *s)
{
    constexpr int H = kMaxClearance - 1, N = kClearTile + 2 * H;
    static_assert(N == 16, "16 rows of 16 bits per plane");
    const int ntx = (nbx + kClearTile - 1) / kClearTile, nty = (nby + kClearTile - 1) / kClearTile;
    const int x0 = tile % ntx * kClearTile - H, y0 = tile / ntx % nty * kClearTile - H,
              z0 = tile / ntx / nty * kClearTile - H;
    const int t = threadIdx.x, lane = t & 63;
#pragma unroll
    for (int row = t >> 4; row < N * N; row += kClearThreads / 16) {
        const int x = x0 + (t & 15), y = y0 + (row & 15), z = z0 + (row >> 4);
        bool clear = true;   // past the volume
        if (x >= 0 && x < nbx && y >= 0 && y < nby && z >= 0 && z < nbz)
            clear = brick_clear(ld_global(range + ((uint64_t)z * nby + y) * nbx + x), nz, n);
        const uint64_t m = __ballot(clear);
        if ((lane & 15) == 0) s[row] = (uint32_t)(m >> lane) & 0xffffu;
    }
    __syncthreads();
    const bool own = t < N * N;
    const int ry = t & 15, rz = t >> 4;
    uint32_t e = own ? s[t] : 0u, cnt = 0u;   // cnt: a nibble for each brick of the tile in this row
    const uint32_t first = e >> H & 0xffu;
    for (int r = 0;; ++r) {
        uint32_t b = e >> H & 0xffu;   // its bits to the low bits of the nibbles
        b = (b | b << 12) & 0x000f000fu;
        b = (b | b << 6) & 0x03030303u;
        b = (b | b << 3) & 0x11111111u;
        cnt += b;
        if (r == H) break;
        e = e & e << 1 & e >> 1;
        if (own) s[256 + t] = e;
        __syncthreads();
        if (own) {
            e &= (ry > 0 ? s[256 + t - 1] : 0u) & (ry < 15 ? s[256 + t + 1] : 0u);
            s[t] = e;
        }
        __syncthreads();
        if (own) e &= (rz > 0 ? s[t - 16] : 0u) & (rz < 15 ? s[t + 16] : 0u);
    }
    int clear = 0;
    const int y = y0 + ry, z = z0 + rz;
    if (own && ry >= H && ry < H + kClearTile && rz >= H && rz < H + kClearTile && y < nby && z < nbz) {
        uint8_t *f = flags + ((uint64_t)z * nby + y) * nbx + (x0 + H);
        const int w = min(kClearTile, nbx - (x0 + H));
        for (int k = 0; k < w; ++k) st_global(f + k, (uint8_t)(cnt >> 4 * k & 15u));
        clear = __popc(first & ((1u << w) - 1u));
    }
    __syncthreads();   // s may be filled again
    return clear;
}
__host__ __device__ constexpr uint32_t clearance_tiles(uint32_t nbx, uint32_t nby, uint32_t nbz)
{
    return ((nbx + kClearTile - 1) / kClearTile) * ((nby + kClearTile - 1) / kClearTile) *
           ((nbz + kClearTile - 1) / kClearTile);
}

// `n_clear` counts the transparent bricks; block 0 clears `next`, the counter
// of the next launch.
static __global__ void __launch_bounds__(kClearThreads)
k_brick_flags(const float2 *__restrict__ range, int nbx, int nby, int nbz, const int *__restrict__ nz, int n,
              uint8_t *__restrict__ flags, uint32_t *__restrict__ n_clear, uint32_t *__restrict__ next)
{
    __shared__ uint32_t s[512];
    if (blockIdx.x == 0 && threadIdx.x == 0) *next = 0u;
    int c = clearance_tile(range, nz, n, nbx, nby, nbz, blockIdx.x, flags, s);
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
    if ((threadIdx.x & 63) == 0 && c) atomicAdd(n_clear, (uint32_t)c);
}

// K3 -- build: a volume's bricks from float32 data in numpy C order (= GL texel
// order, x fastest).  Sources: the scalar field, the normal field (3 floats
// per voxel), or a scalar field that also gives the normals by its gradient.
__device__ __forceinline__ uint32_t enc_sn8(float v)
{
    v = fminf(fmaxf(v, -1.f), 1.f);  // NaN -> -1 .. kept finite
    const int q = (int)rintf(v * 127.f);
    return (uint32_t)(uint8_t)(int8_t)q;
}
__device__ __forceinline__ uint32_t enc_u8(float v)
{
    v = fminf(fmaxf(v, 0.f), 1.f);
    return (uint32_t)rintf(v * 255.f);
}
__device__ __forceinline__ uint32_t enc_h(float v) { return (uint32_t)__half_as_ushort(__float2half_rn(v)); }

// A texel as words (the low bytes of one word below 4 bytes): the scalar or
// the normal put in place, the rest kept.
template <int F>
__device__ __forceinline__ void put_scalar(uint32_t *w, float v)
{
    if constexpr (F == TF_S_F32 || F == TF_C_F32_SN8) w[0] = __float_as_uint(v);
    else if constexpr (F == TF_S_F16) w[0] = enc_h(v);
    else if constexpr (F == TF_S_U8) w[0] = enc_u8(v);
    else if constexpr (F == TF_C_F32_F32) w[3] = __float_as_uint(v);
    else if constexpr (F == TF_C_F16_F32) w[3] = enc_h(v);
    else if constexpr (F == TF_C_U8_F32) w[3] = enc_u8(v);
    else if constexpr (F == TF_C_U8_SN8) w[0] = (w[0] & 0xffffffu) | enc_u8(v) << 24;
    else if constexpr (F == TF_C_F16_F16 || F == TF_C_F16_SN8) w[0] = (w[0] & 0xffff0000u) | enc_h(v);
}
template <int F>
__device__ __forceinline__ void put_normal(uint32_t *w, float nx, float ny, float nz)
{
    if constexpr (F == TF_N_F32 || F == TF_C_F32_F32 || F == TF_C_F16_F32 || F == TF_C_U8_F32) {
        w[0] = __float_as_uint(nx);
        w[1] = __float_as_uint(ny);
        w[2] = __float_as_uint(nz);
    } else if constexpr (F == TF_N_SN8 || F == TF_C_F32_SN8 || F == TF_C_U8_SN8) {
        const uint32_t packed = enc_sn8(nx) | (enc_sn8(ny) << 8) | (enc_sn8(nz) << 16);
        if constexpr (F == TF_N_SN8) w[0] = packed;
        else if constexpr (F == TF_C_F32_SN8) w[1] = packed;
        else w[0] = (w[0] & 0xff000000u) | packed;
    } else if constexpr (F == TF_C_F16_SN8) {
        // the SNORM8 integers as halves (exact), which the march feeds
        // to v_fma_mix without a conversion per channel and tap
        const auto h = [](float v) { return (uint32_t)__half_as_ushort(__int2half_rn((int)(int8_t)enc_sn8(v))); };
        w[0] = (w[0] & 0xffffu) | h(nx) << 16;
        w[1] = h(ny) | h(nz) << 16;
    } else if constexpr (F == TF_C_F16_F16) {
        w[0] = (w[0] & 0xffffu) | enc_h(nx) << 16;
        w[1] = enc_h(ny) | enc_h(nz) << 16;
    } else if constexpr (F == TF_N_F16) {
        w[0] = enc_h(nx) | enc_h(ny) << 16;
        w[1] = enc_h(nz);
    }
}

// Normals of a device float32 field (numpy C order, shape (s0, s1, s2)),
// as compute_normal_volume (pyvr/datasets/synthetic.py:109-122) computes them from a float32 array: np.gradient along each numpy axis
// (central differences halved inside, one-sided at the two faces, unit
// spacing), the norm sqrt((gx^2 + gy^2) + gz^2) summed left to right as
// numpy does, plus float32(1e-8), and each component divided by it, in float32:
// sums, products and quotients correctly rounded, the square root within an
// ulp.  Every axis has at least 2 voxels.
// Voxel l of a field; with 32-bit indices (below 2^30) its byte offset has 32
// bits as well, beside a base the wave shares.
template <typename I>
__device__ __forceinline__ float field_at(const float *__restrict__ f, I l)
{
    return *(const float *)((const char *)f + (I)(l * 4));
}
template <typename I>
__device__ __forceinline__ float np_gradient(const float *__restrict__ f, I l, int i, int n, I st)
{
    // the voxel itself stands in for the neighbour past a face
    const float hi = field_at(f, i == n - 1 ? l : l + st), lo = field_at(f, i == 0 ? l : l - st), d = __fsub_rn(hi, lo);
    return i == 0 || i == n - 1 ? d : __fmul_rn(d, 0.5f);  // /2, exact
}
template <int F>
__device__ __forceinline__ void put_gradient(uint32_t *w, float gx, float gy, float gz)
{
    const float nn = __fadd_rn(
        __fsqrt_rn(__fadd_rn(__fadd_rn(__fmul_rn(gx, gx), __fmul_rn(gy, gy)), __fmul_rn(gz, gz))), 1e-8f);
    // The three quotients by one reciprocal (reciprocal_quotient), between
    // bounds that keep the residuals normal; v_rcp_f32 is within an ulp, and zeros
    // keep their sign by the fixup.  Other operands are divided one by one.
    // (g << 1) - 1 orders |g|, zero last.
    const auto key = [](float g) { return (__float_as_uint(g) << 1) - 1u; };
    const uint32_t least = min(min(key(gx), key(gy)), key(gz));
    if (least >= (__float_as_uint(0x1p-60f) << 1) - 1u && nn <= 0x1p60f && reciprocal_divides(__float_as_uint(nn))) {
        const float y = refine_reciprocal(nn, __builtin_amdgcn_rcpf(nn));
        const auto quotient = [&](float g) {
            return __builtin_amdgcn_div_fixupf(reciprocal_quotient(g, nn, y), nn, g);
        };
        put_normal<F>(w, quotient(gx), quotient(gy), quotient(gz));
    } else {
        put_normal<F>(w, __fdiv_rn(gx, nn), __fdiv_rn(gy, nn), __fdiv_rn(gz, nn));
    }
}

// l / d for l below 2^32: the quotient by double multiplication is off by one at most.
__device__ __forceinline__ uint32_t div_u32(uint32_t l, uint32_t d, double inv)
{
    uint32_t q = (uint32_t)((double)l * inv);
    if (q * d > l) --q;                  // q * d is below 2^32 + d
    else if (l - q * d >= d) ++q;
    return q;
}

struct BuildArgs {
    char *dst;
    int s0, s1, s2;            // GL size
    uint32_t nbx, nby;         // bricks
    uint32_t by0, rows, bz0;   // the launch's first brick row, its rows, its first brick layer
    uint64_t runs;             // groups of build_bricks bricks along x in the launch
    const float *scalar;       // the source, of one kind
    const float *normal;
    const float *field;
    uint64_t plane;            // voxels between the source's planes
    uint64_t first;            // index of the source's first voxel, counted in such planes
    double inv_n12, inv_s2;    // 1 / (s1 s2), 1 / s2
    int keep;                  // the texels hold the other part, which stays
    float2 *range;             // per-brick density range, where the scalar is written
};
constexpr int build_bricks(int lb) { return lb == 4 ? 1 : 4; }   // bricks along x per block: V waves each

// One wave per brick (all 4 of a block for 16^3 bricks, which are as many
// times fewer), build_bricks bricks along x per block: one per wave, since
// blocks of more leave most of the device idle in their last round (2,646
// blocks of four 16^3 bricks are 1.3 rounds of 8 per unit).  Every slot of a
// brick is written once, in order, from its voxel: texel X = c + 1 of an axis
// holds voxel c, X = 0 and X = s + 1 the edge voxels, and slots past those are
// 0.  In a brick clear of the volume's faces, where the numpy axes are the GL
// ones (s0 == s2), a slot is one offset beside seven wave-wide bases.
// Per-brick density range (for the transparent-brick flags): over all slots as
// stored, the apron included, so that it covers every footprint the brick
// serves; a NaN widens it to everything.  UNORM8 ranges are in decoded units
// (raw / 255).
// What bounds it, FP16+FP16x3 from a field: for 320^3 in 16^3 bricks (163 us)
// VALU issue, 72 % busy, and memory (392 MB out; 658 MB in, since each of the 8
// L2s fetches its bricks' surroundings, from the last cache for the most part).
// 512^3 in 8^3 bricks takes 1020 us, 1.5 times as long per voxel: 1.73 GB out
// and 1.85 GB in at 3.5 TB/s where 1.60 and 0.54 GB are what it cannot do
// without, VALU issue 51 % busy, a wave 17 us for the 12 rounds of its brick.  ONCE
// writes the texels past the caches, which leaves the field there; it is for
// field and texels together above the 256 MB of the last cache (the 320^3 217
// -> 160 us, FP32+FP32x3 256^3 154 -> 114, UNORM8+SNORM8x3 384^3 316 -> 224).
// Below, it gains nothing (FP16+FP16x3 192^3 54 / 54) and a march after it takes
// 5-8 us longer.  Writing whole texels in order, the range formed on the way,
// replaces a thread per voxel that scattered it to its up to eight slots, a
// clearing pass and a pass for the ranges: FP16+FP16x3 255x193x160 from a field
// 174 -> 81 us, 320^3 in 16^3 bricks 709 -> 160; FP32+FP32x3 192^3 in its two
// parts 236 -> 152.  A slab of the volume per XCD fetches the field once (78 MB)
// but was no faster on the whole (320^3 144, 384^3 298 -> 327).
template <int F, int LB, typename I, bool ONCE>
__global__ void __launch_bounds__(256)
k_build(const BuildArgs a)
{
    constexpr uint32_t B = 1u << LB, E = B + 1u, N = E * E * E, T = (uint32_t)texel_bytes(F), W = (T + 3) / 4;
    constexpr uint32_t G = (uint32_t)build_bricks(LB), V = LB == 4 ? 4 : 1;   // V: waves per brick
    __shared__ float s_range[3][4];
    const uint32_t ngx = (a.nbx + G - 1) / G, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const I plane = (I)a.plane, n12 = (I)a.s1 * (I)a.s2, first = (I)a.first;
    for (uint64_t run = blockIdx.x; run < a.runs; run += gridDim.x)
    for (uint32_t j = wave / V; j < G; j += 4 / V) {
        const uint32_t bx = (uint32_t)(run % ngx) * G + j, by = a.by0 + (uint32_t)(run / ngx % a.rows),
                       bz = a.bz0 + (uint32_t)(run / ngx / a.rows);
        if (bx >= a.nbx) break;
        const uint64_t brick = ((uint64_t)bz * a.nby + by) * a.nbx + bx;
        char *out = a.dst + brick * ((uint64_t)N * T);
        float lo = INFINITY, hi = -INFINITY;
        bool nan = false;
        const bool inside = fmt_has_normal(F) && a.field && a.s0 == a.s2 && bx && by && bz &&
                            (bx + 1) * B < (uint32_t)a.s0 && (by + 1) * B < (uint32_t)a.s1 &&
                            (bz + 1) * B < (uint32_t)a.s2;
        const auto put = [&](uint32_t k, const uint32_t *w) {
            char *p = out + k * T;
            if constexpr (T == 1) *(uint8_t *)p = (uint8_t)w[0];
            else if constexpr (T == 2) *(uint16_t *)p = (uint16_t)w[0];
            else if constexpr (ONCE) {
#pragma unroll
                for (uint32_t q = 0; q < W; ++q) __builtin_nontemporal_store(w[q], (uint32_t *)p + q);
            } else {
#pragma unroll
                for (uint32_t q = 0; q < W; ++q) ((uint32_t *)p)[q] = w[q];
            }
            if constexpr (fmt_has_scalar(F)) {
                float v;
                if constexpr (F == TF_S_F16) v = h16f(w[0]);
                else if constexpr (F == TF_S_U8) v = (float)w[0];
                else if constexpr (F == TF_S_F32) v = __uint_as_float(w[0]);
                else v = decode_scalar<F>(w);
                if constexpr (fmt_u8_scalar(F)) v *= 1.0f / 255.0f;
                nan |= v != v;
                lo = fminf(lo, v);
                hi = fmaxf(hi, v);
            }
        };
        const uint32_t k0 = wave % V * 64 + lane;
        if (fmt_has_normal(F) && inside) {
            // the voxel of slot 0, and from it those of the others
            const float *f0 = a.field + ((I)(bz * B - 1) * plane + (I)(by * B - 1) * (I)a.s0 + (I)(bx * B - 1));
            for (uint32_t k = k0; k < N; k += 64 * V) {
                const I r = (I)(k / (E * E)) * plane + (I)(k / E % E * (uint32_t)a.s0) + (I)(k % E);
                const auto slope = [&](I st) {
                    return __fmul_rn(__fsub_rn(field_at(f0 + st, r), field_at(f0 - st, r)), 0.5f);
                };
                uint32_t w[W] = {};
                put_scalar<F>(w, field_at(f0, r));
                put_gradient<F>(w, slope(n12), slope((I)a.s2), slope((I)1));
                put(k, w);
            }
        } else for (uint32_t k = k0; k < N; k += 64 * V) {
            const uint32_t X = bx * B + k % E, Y = by * B + k / E % E, Z = bz * B + k / (E * E);
            uint32_t w[W] = {};
            if (X <= (uint32_t)a.s0 + 1u && Y <= (uint32_t)a.s1 + 1u && Z <= (uint32_t)a.s2 + 1u) {
                const int x = slot_voxel(X, a.s0), y = slot_voxel(Y, a.s1), z = slot_voxel(Z, a.s2);
                const I l = (I)z * plane + (I)y * (I)a.s0 + (I)x;
                if (T >= 4 && a.keep) {
#pragma unroll
                    for (uint32_t q = 0; q < W; ++q) w[q] = ((const uint32_t *)(out + k * T))[q];
                }
                if (a.normal) {
                    const float *n = a.normal + 3 * (uint64_t)(l - first);
                    put_normal<F>(w, n[0], n[1], n[2]);
                } else if (a.scalar) {
                    put_scalar<F>(w, a.scalar[l - first]);
                } else {
                    put_scalar<F>(w, field_at(a.field, l));
                    if constexpr (fmt_has_normal(F)) {
                        // numpy coordinates of flat index l
                        int i0 = z, i1 = y, i2 = x;
                        if (a.s0 != a.s2) {
                            if constexpr (sizeof(I) == 4) {
                                i0 = (int)div_u32(l, n12, a.inv_n12);
                                const uint32_t r = l - (uint32_t)i0 * n12;
                                i1 = (int)div_u32(r, (uint32_t)a.s2, a.inv_s2);
                                i2 = (int)(r - (uint32_t)i1 * (uint32_t)a.s2);
                            } else {
                                i0 = (int)(l / n12);
                                const I r = l - (I)i0 * n12;
                                i1 = (int)(r / (I)a.s2);
                                i2 = (int)(r - (I)i1 * (I)a.s2);
                            }
                        }
                        const float gx = np_gradient(a.field, l, i0, a.s0, n12);
                        const float gy = np_gradient(a.field, l, i1, a.s1, (I)a.s2);
                        const float gz = np_gradient(a.field, l, i2, a.s2, (I)1);
                        put_gradient<F>(w, gx, gy, gz);
                    }
                }
            }
            put(k, w);
        }
        if (fmt_has_scalar(F) && a.range) {
            for (int off = 32; off > 0; off >>= 1) {
                lo = fminf(lo, __shfl_xor(lo, off, 64));
                hi = fmaxf(hi, __shfl_xor(hi, off, 64));
            }
            nan = __ballot(nan) != 0;
            if constexpr (V > 1) {   // every wave of the block is at this brick
                if (lane == 0) {
                    s_range[0][wave] = lo;
                    s_range[1][wave] = hi;
                    s_range[2][wave] = nan ? 1.f : 0.f;
                }
                __syncthreads();
                lo = fminf(fminf(s_range[0][0], s_range[0][1]), fminf(s_range[0][2], s_range[0][3]));
                hi = fmaxf(fmaxf(s_range[1][0], s_range[1][1]), fmaxf(s_range[1][2], s_range[1][3]));
                nan = s_range[2][0] + s_range[2][1] + s_range[2][2] + s_range[2][3] != 0.f;
                __syncthreads();
            }
            if (lane == 0 && wave % V == 0) a.range[brick] = nan ? make_float2(-INFINITY, INFINITY) : make_float2(lo, hi);
        }
    }
}

// Seeded Gaussian-blob field generated on the device (numpy C order): the
// family of pyvr_amd.datasets.blob_field -- axes linspace(-1, 1, s),
// amplitude * exp(-(axis - centre)^2 / (2 sigma^2)) per axis multiplied as
// amp * (fx * (fy * fz)) in double, summed over the blobs -- plus uniform
// noise in [-noise, noise] from a counter-based hash of (seed, voxel),
// clipped to [0, 1] and rounded to float32.
static constexpr int kMaxBlobs = 32;
struct BlobSpec {
    double c[3 * kMaxBlobs], s[kMaxBlobs], a[kMaxBlobs];
    double noise;
    uint64_t seed;
    int n;
};

__device__ __forceinline__ uint64_t splitmix64(uint64_t z)
{
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

__device__ __forceinline__ double np_linspace(int i, int n)
{
    if (n <= 1) return -1.0;
    if (i == n - 1) return 1.0;
    return (double)i * (2.0 / (double)(n - 1)) + -1.0;
}

// The blobs' factors exp(-(axis - centre)^2 / (2 sigma^2)) along each axis:
// for blob b, s0 of them at fac + b * (s0 + s1 + s2), then s1, then s2.
static __global__ void __launch_bounds__(256)
k_blob_factors(double *__restrict__ fac, int s0, int s1, int s2, const BlobSpec *__restrict__ spec)
{
    const int len = s0 + s1 + s2;
    for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < (int64_t)len * spec->n;
         t += (int64_t)gridDim.x * 256) {
        const int b = (int)(t / len), j = (int)(t % len);
        const int axis = j < s0 ? 0 : j < s0 + s1 ? 1 : 2;
        const int i = axis == 0 ? j : axis == 1 ? j - s0 : j - s0 - s1;
        const double k = 2.0 * spec->s[b] * spec->s[b];
        const double d = np_linspace(i, axis == 0 ? s0 : axis == 1 ? s1 : s2) - spec->c[3 * b + axis];
        fac[t] = exp(-(d * d) / k);
    }
}

// A wave takes 64 voxels along the last axis and kBlobRows rows of the middle
// one: the last axis' factor is a load per blob, the others' are scalar.
// With every factor computed at every voxel (three exponentials in double per
// blob) the kernel took 1058 us for 8 blobs at 320^3; these two take 110-120.
// VALU issue bounds it (88 % busy for 8 blobs at 512^3, 390 us: the noise's hash,
// an FP64 product and sum per blob); the field is written at 1.4 TB/s.
static constexpr int kBlobRows = 8;
static __global__ void __launch_bounds__(256)
k_blob_field(float *__restrict__ out, int s0, int s1, int s2, const BlobSpec *__restrict__ spec,
             const double *__restrict__ fac)
{
    const uint64_t nz = ((uint64_t)s2 + 63) / 64, ny = ((uint64_t)s1 + kBlobRows - 1) / kBlobRows, total = nz * ny * s0;
    const int len = s0 + s1 + s2, n = spec->n;
    const double noise = spec->noise;
    for (uint64_t t = (uint64_t)blockIdx.x * 4 + (uint64_t)(__builtin_amdgcn_readfirstlane((int)threadIdx.x) >> 6);
         t < total; t += (uint64_t)gridDim.x * 4) {
        const int i2 = (int)(t % nz) * 64 + (int)(threadIdx.x & 63), j1 = (int)(t / nz % ny) * kBlobRows,
                  i0 = (int)(t / nz / ny);
        const int c2 = min(i2, s2 - 1);
        double acc[kBlobRows] = {};
        for (int b = 0; b < n; ++b) {
            const double *f = fac + (int64_t)b * len;
            const double amp = spec->a[b], fx = f[i0], fz = f[s0 + s1 + c2];
#pragma unroll
            for (int r = 0; r < kBlobRows; ++r) acc[r] += amp * (fx * (f[s0 + min(j1 + r, s1 - 1)] * fz));
        }
        if (i2 >= s2) continue;
#pragma unroll
        for (int r = 0; r < kBlobRows; ++r) {
            if (j1 + r >= s1) break;
            const uint64_t l = ((uint64_t)i0 * s1 + (uint64_t)(j1 + r)) * s2 + (uint64_t)i2;
            double v = acc[r];
            if (noise > 0.0) {
                const uint64_t h = splitmix64(spec->seed ^ splitmix64(l));
                const double u = (double)(h >> 11) * 0x1p-53;  // [0, 1)
                v += (2.0 * u - 1.0) * noise;
            }
            out[l] = (float)fmin(fmax(v, 0.0), 1.0);
        }
    }
}

// ---------------------------------------------------------------------------
// Batched rendering: many requests (own volume, image size, camera, LUT) in
// one persistent launch per kernel instance.  The host groups requests by
// instance (storage format, normal mode, brick size) into classes and
// stages, for each class, a descriptor array ordered by decreasing cost;
// tiles of 256 pixels are numbered through the class's requests in that
// order.  Blocks take the next tile from an atomic counter until none is
// left, load the request's LUT into LDS when the request changes, and set
// up and march each pixel's ray exactly as the single-request kernels do.

struct ReqDesc {
    FrameConst fc;
    TexDesc ts;                    // scalar volume (also the normals: NM_SAME / NM_ALIAS)
    const float4 *lut;             // lut_n RGBA entries
    const int *nz;                 // lut_n + 1 prefix counts of non-transparent entries
    const float2 *range;           // per-brick density range of the volume
    uint8_t *flags;                // per-brick transparent flags for this LUT
    uchar4 *out;                   // W*H RGBA8, bottom row first
    uint32_t *counts;              // W*H composited-sample counts (counting runs)
    uint32_t nbz;                  // bricks along z
    uint32_t flag_end;             // one past this request's last tile of k_batch_flags
    int lut_n;
    int ntx;                       // tiles along x
    int tile_end;                  // one past this request's last tile in its class
};

// Per class: where its descriptors are in the staged block, and how many.
struct BatchClass {
    uint32_t desc_offset;          // bytes from the block start
    int nreq;
};

static constexpr int kBatchMaxClasses = 8;

// The staged block starts with this header, then the descriptors, LUTs and
// prefix counts.
struct BatchHeader {
    BatchClass cls[kBatchMaxClasses];
    int nclass;
    int nreq;                      // all requests (descriptors are contiguous)
    uint32_t all_offset;           // first descriptor of the first class
    int pad;
};

// Ray-tile shapes: a wave covers WX x WY pixels; a block is W waves (2, 4
// or 8; 4 by default), 2 across and W / 2 down, and takes one tile of
// (2 WX) x (W / 2 * WY) pixels at a time.  Fewer waves per block halve the
// tile and double the counter traffic; more lengthen the wait at the
// per-tile barrier.  The autotuner times them.
static constexpr int kBatchWaves = 4;

template <int TS>
struct TileShape;
template <>
struct TileShape<0> {
    static constexpr int WX = 8, WY = 8;
};
template <>
struct TileShape<1> {
    static constexpr int WX = 16, WY = 4;
};

// W: waves per block.  SKIP: step over transparent bricks (the flags of
// k_batch_flags).  GATE: interpolate and light normals only for samples of
// non-zero alpha.  Every variant gives the same image.  For texels of up
// to 8 bytes the launch bounds ask for 8 waves per SIMD (64 VGPRs): the
// compiler then keeps a few per-ray values in scratch outside the march
// loop rather than run 7 waves.  16-byte texels would spill inside the
// loop, so their kernels keep the registers they need.
// P lanes per ray (batch_lanes, by a class's rays; no gating): a wave covers
// 8x4 or 4x4 pixels then.
template <int SF, int NM, int LB, bool COUNT, int TS, bool BUF, int W = kBatchWaves, bool SKIP = true,
          bool GATE = true, int P = 1>
__global__ void __launch_bounds__(64 * W, texel_bytes(SF) > 8 ? 1 : 8)
k_batch(const char *__restrict__ block, int cls, uint32_t *__restrict__ counter)
{
    extern __shared__ float4 s_lut[];
    __shared__ int s_item[2];
    static_assert(P == 1 || TS == 0, "several lanes march square tiles");
    constexpr int WX = P == 4 ? 4 : TileShape<TS>::WX, WY = P == 1 ? TileShape<TS>::WY : 4, BX = 2 * WX, BY = W / 2 * WY;
    const BatchHeader *hdr = (const BatchHeader *)block;
    const int nreq = hdr->cls[cls].nreq;
    if (nreq <= 0) return;
    const ReqDesc *__restrict__ reqs = (const ReqDesc *)(block + hdr->cls[cls].desc_offset);
    const int total = reqs[nreq - 1].tile_end;
    // the wave's index in the block as a scalar, so that no per-thread value
    // but the lane index is needed after a ray's march (the pixel is formed
    // again there from scalars and the lane index)
    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x) >> 6, lane = threadIdx.x & 63;
    int cur = -1;
    for (;;) {
        if (threadIdx.x == 0) {
            const int t = (int)atomicAdd(counter, 1u);
            int q = 0;
            if (t < total) {
                int lo = 0, hi = nreq - 1;
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (reqs[mid].tile_end > t) hi = mid;
                    else lo = mid + 1;
                }
                q = lo;
            }
            s_item[0] = t;
            s_item[1] = q;
        }
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(s_item[0]);
        const int q = __builtin_amdgcn_readfirstlane(s_item[1]);
        if (t >= total) break;
        const ReqDesc &R = reqs[q];
        if (q != cur) {
            load_lut_lds(R.lut, R.lut_n, s_lut);
            __syncthreads();
            cur = q;
        }
        const int lt = t - (q ? reqs[q - 1].tile_end : 0);
        const int tx = lt % R.ntx, ty = lt / R.ntx;
        const int px = tx * BX + (wv & 1) * WX + lane / P % WX;
        const int py = ty * BY + (wv >> 1) * WY + lane / P / WX;
        if (px < R.fc.W && py < R.fc.H) {
            const RayRec r = ray_setup(R.fc, px, py);
            float C0 = 0.f, C1 = 0.f, C2 = 0.f, A = 0.f;
            uint32_t ns = 0;
            march_ray<SF, NM, LB, COUNT, SKIP, BUF, GATE && P == 1, P>(R.fc, R.ts, R.ts, R.lut, R.lut_n, s_lut, r,
                                                           R.flags, C0, C1, C2, A, ns);
            const int ln = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));   // = lane
            const int pix =
                (ty * BY + (wv >> 1) * WY + ln / P / WX) * R.fc.W + tx * BX + (wv & 1) * WX + ln / P % WX;
            if (P == 1 || ln % P == 0) st_global(R.out + pix, blend_store(R.fc, C0, C1, C2, A));
            if constexpr (COUNT) st_global(R.counts + pix, ns);
        }
        // every thread is done with this tile's LDS before the next fetch
        __syncthreads();
    }
}

// Clearances of every request of a batch for its own LUT: tiles are
// numbered through the requests (requests that share volume and LUT share
// one set of flags, and all but the first have no tiles).
static __global__ void __launch_bounds__(kClearThreads) k_batch_flags(const char *__restrict__ block)
{
    __shared__ uint32_t s[512];
    const BatchHeader *hdr = (const BatchHeader *)block;
    const ReqDesc *__restrict__ reqs = (const ReqDesc *)(block + hdr->all_offset);
    const int nreq = hdr->nreq;
    const uint32_t total = reqs[nreq - 1].flag_end;
    for (uint32_t t = blockIdx.x; t < total; t += gridDim.x) {
        int lo = 0, hi = nreq - 1;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (reqs[mid].flag_end > t) hi = mid;
            else lo = mid + 1;
        }
        const ReqDesc &R = reqs[lo];
        clearance_tile(R.range, R.nz, R.lut_n, (int)R.ts.nbx, (int)R.ts.nby, (int)R.nbz,
                       (int)(t - (lo ? reqs[lo - 1].flag_end : 0u)), R.flags, s);
    }
}

static __global__ void __launch_bounds__(64) k_fill_u32(uint32_t *__restrict__ p, int n, uint32_t v)
{
    for (int i = threadIdx.x; i < n; i += 64) p[i] = v;
}

// A one-request batch block written on the device from kernel arguments (so
// that a frame needs no host-to-device copy and no staging allocation): the
// header at the start of the block (where k_batch and k_batch_flags read
// it), the tile counter reset to 0, the prefix counts of the unbound LUT
// (0, 1), and the descriptor, at the offsets the host chose.
struct StageOffsets {
    uint32_t counter, unbound_nz, desc;
};

static __global__ void __launch_bounds__(64)
k_stage_request(char *__restrict__ blk, const StageOffsets off, const BatchHeader hdr, const ReqDesc desc)
{
    const int lane = threadIdx.x;
    if (lane == 0) {
        *(uint32_t *)(blk + off.counter) = 0u;
        ((int *)(blk + off.unbound_nz))[0] = 0;
        ((int *)(blk + off.unbound_nz))[1] = 1;
    }
    static_assert(sizeof(BatchHeader) % 4 == 0 && sizeof(ReqDesc) % 4 == 0, "dword copies");
    const uint32_t *h = (const uint32_t *)&hdr, *d = (const uint32_t *)&desc;
    uint32_t *hh = (uint32_t *)blk, *dd = (uint32_t *)(blk + off.desc);
    for (int i = lane; i < (int)(sizeof(BatchHeader) / 4); i += 64) hh[i] = h[i];
    for (int i = lane; i < (int)(sizeof(ReqDesc) / 4); i += 64) dd[i] = d[i];
}

// Decoded texels of a volume in numpy C order (texel (x, y, z) at flat
// x + s0*(y + s1*z)), z-planes z0 .. z0 + nz - 1: the scalar as the march
// reads it (UNORM8 times 1/255) and the normal as stored (SNORM8 as its
// integer, FP16 as float).  Either output may be null.
template <int F>
__global__ void __launch_bounds__(256)
k_download(const char *__restrict__ texels, int s0, int s1, int lb, uint32_t nbx, uint32_t nby, uint32_t brick_bytes,
           int z0, uint64_t nvox, float *__restrict__ scalar, float *__restrict__ normal)
{
    const uint64_t l = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (l >= nvox) return;
    const uint64_t plane = (uint64_t)s0 * (uint64_t)s1;
    const uint32_t z = (uint32_t)(l / plane) + (uint32_t)z0;
    const uint64_t rem = l % plane;
    const uint32_t y = (uint32_t)(rem / (uint64_t)s0), x = (uint32_t)(rem % (uint64_t)s0);
    // the texel's own slot in the extended (apron) coordinates X = x + 1
    const uint32_t X = x + 1u, Y = y + 1u, Z = z + 1u, M = (1u << lb) - 1u, E = (1u << lb) + 1u;
    const uint64_t brick = ((uint64_t)(Z >> lb) * nby + (Y >> lb)) * nbx + (X >> lb);
    const uint32_t local = ((Z & M) * E + (Y & M)) * E + (X & M);
    const float4 t = fetch4<F>(texels + brick * brick_bytes + (uint64_t)local * (uint32_t)texel_bytes(F));
    if (scalar) scalar[l] = fmt_u8_scalar(F) ? t.w * (1.0f / 255.0f) : t.w;
    if (normal) {
        normal[3 * l] = t.x;
        normal[3 * l + 1] = t.y;
        normal[3 * l + 2] = t.z;
    }
}

}  // namespace hvr
