// hipvr.hip -- libhipvr.so: C ABI (include/hipvr.h) over the gfx950 kernels
// of hvr_device.h.  Host side: contexts (framebuffer, rays, LUT, stream,
// events), volumes (device texels in brick layout), FP64 uniform
// preparation and kernel dispatch.
#include "hvr_copy.h"
#include "hvr_launch.h"
#include "hvr_share.h"
#include "../../include/hipvr.h"

#include <math.h>
#include <cmath>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <string>
#include <vector>

using namespace hvr;

// ---------------------------------------------------------------------------
// errors
static thread_local std::string g_err;

// A failed HIP call (an allocation above the device's memory, say) also
// sets the thread's last error, which the launch checks of later calls read:
// once a failure is reported (or handled), the last error is cleared so that
// a later, unrelated call does not report it again.
static int fail(int code, const char *msg)
{
    g_err = msg;
    (void)hipGetLastError();
    return code;
}
static int fail_hip(hipError_t e, const char *where)
{
    g_err = std::string(where) + ": " + hipGetErrorString(e);
    (void)hipGetLastError();
    return e == hipErrorOutOfMemory ? HVR_ENOMEM : HVR_EDEVICE;
}
#define HIPCHK(expr)                                   \
    do {                                               \
        hipError_t e_ = (expr);                        \
        if (e_ != hipSuccess) return fail_hip(e_, #expr); \
    } while (0)

// ---------------------------------------------------------------------------
// fault injection (hvr_debug_inject_fault): one armed entry point fails with
// a chosen code on its n-th call, before any device work
static std::mutex g_fault_mu;
static std::atomic<bool> g_fault_armed{false};
static std::string g_fault_fn;
static int g_fault_code = 0, g_fault_after = -1;

static int fault_point(const char *fn)
{
    if (!g_fault_armed.load(std::memory_order_relaxed)) return HVR_OK;
    std::lock_guard<std::mutex> lock(g_fault_mu);
    if (g_fault_after < 0 || g_fault_fn != fn) return HVR_OK;
    if (g_fault_after-- > 0) return HVR_OK;
    g_fault_armed.store(false);
    g_fault_after = -1;
    return fail(g_fault_code, (std::string("injected fault in ") + fn).c_str());
}
#define HVR_FAULT_POINT(fn)                             \
    do {                                               \
        if (const int rc_ = fault_point(fn)) return rc_; \
    } while (0)

// ---------------------------------------------------------------------------
// objects
struct hvr_volume {
    hvr_ctx *ctx;
    int s0, s1, s2;
    int fmt;               // TexFmt
    int lb;                // log2 of the brick interior edge
    uint32_t nbx, nby, nbz;
    uint32_t brick_bytes;  // (2^lb + 1)^3 texels
    uint64_t bytes;
    void *d_texels;
    size_t block_bytes;    // of the allocation: the texels, then the ranges
    bool scalar_loaded, normals_loaded, cleared;
    float2 *d_range;       // per-brick scalar range (formats with a scalar field)
    uint32_t gen;          // bumped on every upload
};

struct hvr_ctx {
    int device;
    int W, H;
    hipStream_t stream;
    uchar4 *d_out;
    uint32_t *d_counts;
    float4 *d_lut;
    int lut_n;       // entries in d_lut (>= 1)
    int lut_cap;
    void *h_pinned;  // W*H*4 readback staging
    void *h_pinned_dev;   // its device address (the march's target in HVR_READBACK_DIRECT)
    int readback_mode;    // HVR_READBACK_COPY / _DIRECT
    bool last_host;       // the last frame was written to h_pinned
    float *d_stage;  // upload staging
    size_t stage_bytes, max_stage;   // what it holds, and may hold while an upload of parts fits it
    char *h_up;           // pinned ring the uploads go through (upload_host), or nullptr
    hipEvent_t up_ev[3];  // after the last copy out of each of its parts
    hipEvent_t ev[4];
    hipEvent_t rev[4];   // readback chunks (hvr_read)
    hipEvent_t last_ev[3];  // the last frame's events (ev[] or a timing region's)
    bool events_recorded;
    hvr_params params;
    bool params_set;
    hvr_volume *scalar_vol, *normal_vol;
    int scalar_role, normal_role;
    int brick_log2;
    // per-launch timing region (hvr_timing_begin/end)
    std::vector<hipEvent_t> *tev;
    std::vector<char> *tev_ordered;   // whether the frame had a pass before its march
    int timing_max, timing_n;
    // transparent-brick skipping
    int *d_nz;             // prefix counts of non-transparent LUT entries (lut_n + 1)
    int nz_cap;            // entries d_nz holds counts for
    uint32_t lut_gen;
    uint8_t *d_flags;      // per-brick transparent flags of flags_vol
    uint32_t *d_nclear;    // two transparent-brick counters, which k_brick_flags fills in turn
    int nclear_slot;       // the counter of the next k_brick_flags
    uint32_t *h_nclear;    // its copy in pinned host memory, valid once flags_ev completed
    hipEvent_t flags_ev;   // recorded after that copy
    bool flags_count_known;   // flags_clear holds the count of the current flags
    uint64_t flags_cap;
    const hvr_volume *flags_vol;
    uint32_t flags_vol_gen, flags_lut_gen;
    uint64_t flags_clear, flags_total;
    int skip_mode;         // HVR_SKIP_OFF / _ON / _AUTO
    int skip_used;         // whether the last frame's march stepped over bricks
    bool force_global;     // HVR_GATHER=global at creation: 64-bit loads for every volume
    bool force_wide;       // HVR_BUILD=wide at creation: 64-bit voxel offsets for every volume
    int ncu;               // compute units of the device
    size_t pix_cap;        // pixels d_out and h_pinned hold
    size_t counts_cap;     // pixels d_counts holds
    // cost-ordered dispatch of single frames (k_order_blocks)
    uint32_t *d_order;     // block of each dispatch position, then the slots
    size_t order_words;    // words d_order holds
    int order_mode;        // HVR_ORDER_OFF / _ON / _AUTO
    int order_used;        // whether the last frame was cost-ordered
    // LUT uploads (hvr_set_lut): pinned staging slots holding the entries and
    // their prefix counts, each reused once the copy that last read it is done
    void *h_lut_stage[4];
    hipEvent_t lut_ev[4];
    bool lut_ev_live[4];
    size_t lut_stage_bytes;   // bytes each slot holds
    int lut_slot;             // the next slot
};

// HVR_SKIP_AUTO steps over transparent bricks when at least this fraction of
// the bound volume's bricks are transparent for the current LUT.  The skipping
// kernel costs 0-5 % where there is nothing to skip (64^3 thumbnails 7 %, 1.4
// us); time without / with skipping, geometric mean and range over borders, cut
// slabs and scattered holes in five storage formats at 512^2 to 1024^2: 6-13 %
// transparent 1.10 (0.93-1.56), 13-16 % 1.05 (0.96-1.43), 16-20 % 1.19
// (0.95-1.77), 20-25 % 1.34 (1.07-2.29), 25-32 % 1.32 (1.07-2.14).
static constexpr double kSkipAutoFraction = 0.18;

// The rays the device marches at once with one lane each: 8 blocks of 256
// threads per compute unit.
static long long resident_rays(const hvr_ctx *c) { return 2048ll * c->ncu; }


// ---------------------------------------------------------------------------
// Device memory of volumes.  A program that shows a sequence of volumes frees
// one block and allocates another of the same size for each; above 64 MB hipMalloc
// and hipFree take 60 and 265 us, and blocks of hundreds of MB that come and
// go at that rate have stalled hipMalloc for 11 ms at a time.  The last block
// freed on a device is therefore kept for the next volume on it, from any
// context: at most one, of at most kSpareMax bytes.  It is given back when
// the next volume cannot use it (too small, or more than a sixteenth too large),
// when an allocation of this library fails for want of memory, by hvr_trim, and
// with the device's last context; hvr_device_memory counts it as free.  A block
// is put aside only once the device is idle, as hipFree would wait for, so no
// stream still reads it.
static constexpr size_t kSpareMax = (size_t)512 << 20;
static constexpr int kMaxDevices = 64;
struct SpareBlock {
    void *p;
    size_t bytes;
    int contexts;   // live contexts of the device
};
static std::mutex g_spare_mu;
static SpareBlock g_spare[kMaxDevices];

// Take the device's spare block out (nullptr if there is none).
static void *spare_take(int device, size_t *bytes)
{
    if (device < 0 || device >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lock(g_spare_mu);
    void *p = g_spare[device].p;
    *bytes = g_spare[device].bytes;
    g_spare[device].p = nullptr;
    return p;
}
static size_t spare_bytes(int device)
{
    if (device < 0 || device >= kMaxDevices) return 0;
    std::lock_guard<std::mutex> lock(g_spare_mu);
    return g_spare[device].p ? g_spare[device].bytes : 0;
}
// hipMalloc that gives the spare block back before it fails; the device is current.
static hipError_t dev_malloc(int device, void **p, size_t n)
{
    hipError_t e = hipMalloc(p, n);
    if (e == hipErrorOutOfMemory) {
        size_t b;
        if (void *spare = spare_take(device, &b)) {
            (void)hipGetLastError();
            (void)hipFree(spare);
            e = hipMalloc(p, n);
        }
    }
    return e;
}
static hipError_t block_alloc(int device, void **p, size_t n, size_t *got)
{
    size_t b = 0;
    if (void *spare = spare_take(device, &b)) {
        if (b >= n && b - n <= n / 16) {
            *p = spare;
            *got = b;
            return hipSuccess;
        }
        (void)hipFree(spare);
    }
    *got = n;
    return dev_malloc(device, p, n);
}
static void block_free(int device, void *p, size_t n)
{
    if (!p) return;
    if (n <= kSpareMax && device >= 0 && device < kMaxDevices && hipDeviceSynchronize() == hipSuccess) {
        std::lock_guard<std::mutex> lock(g_spare_mu);
        std::swap(g_spare[device].p, p);
        g_spare[device].bytes = n;
    }
    (void)hipFree(p);   // the block before, or this one
}
static void context_count(int device, int by)
{
    if (device < 0 || device >= kMaxDevices) return;
    bool last;
    {
        std::lock_guard<std::mutex> lock(g_spare_mu);
        last = (g_spare[device].contexts += by) == 0;
    }
    size_t b;
    if (last) (void)hipFree(spare_take(device, &b));
}

// ---------------------------------------------------------------------------
// FP64 uniform preparation

// Uniforms -> kernel constants.  The matrices arrive as numpy row-major
// float32 bytes that GLSL reads column-major, i.e. transposed
// (manager.py:192); they are inverted in double and rounded once to float.
static FrameConst frame_const_of(const hvr_params &p, bool params_set, int W, int H)
{
    FrameConst f;
    memset(&f, 0, sizeof(f));
    f.W = W;
    f.H = H;
    f.fW = (float)W;
    f.fH = (float)H;
    double pg[16], vg[16], pinv[16], vinv[16];
    for (int r = 0; r < 4; ++r)
        for (int k = 0; k < 4; ++k) {
            pg[4 * r + k] = (double)p.proj[4 * k + r];
            vg[4 * r + k] = (double)p.view[4 * k + r];
        }
    f.ok = params_set && p.camera_set && inverse4(pg, pinv) && inverse4(vg, vinv);
    if (f.ok) {
        for (int k = 0; k < 8; ++k) f.prow[k] = (float)pinv[k];
        for (int r = 0; r < 3; ++r)
            for (int k = 0; k < 3; ++k) f.rot[3 * r + k] = (float)vinv[4 * r + k];
    }
    for (int k = 0; k < 3; ++k) {
        f.o[k] = p.cam_pos[k];
        f.bmin[k] = p.bmin[k];
        f.bmax[k] = p.bmax[k];
        f.ext[k] = p.bmax[k] - p.bmin[k];  // float subtraction, as in the shader
    }
    f.step = p.step;
    // exp(-a*step/ref) = exp2(-a * log2(e) * step/ref)
    f.alpha_k = (float)(1.4426950408889634 * (double)p.step / (double)p.ref_step);
    f.ka = p.ambient;
    f.kd = p.diffuse;
    f.tau = p.et_threshold;
    f.max_steps = p.max_steps;
    double l[3], ll = 0.0;
    for (int k = 0; k < 3; ++k) {
        l[k] = (double)p.light_target[k] - (double)p.light_pos[k];
        ll += l[k] * l[k];
    }
    f.L_ok = ll > 0.0;
    for (int k = 0; k < 3; ++k) f.L[k] = f.L_ok ? (float)(l[k] / sqrt(ll)) : 0.f;
    for (int k = 0; k < 4; ++k) f.clear[k] = p.clear_rgba[k];
    f.blend = p.blend != 0;
    return f;
}

static FrameConst frame_const(const hvr_ctx *c) { return frame_const_of(c->params, c->params_set, c->W, c->H); }

// Texture descriptor for a frame: texture x samples world z, y samples y,
// z samples x (the shader's swizzle), so k0 = s0/ext_z, k1 = s1/ext_y,
// k2 = s2/ext_x with ext the float box extent of the in-box test.
static TexDesc tex_desc(const hvr_volume *v, int role, const FrameConst &fc)
{
    TexDesc t;
    memset(&t, 0, sizeof(t));
    if (!v) return t;
    t.base = v->d_texels;
    t.s0 = v->s0;
    t.s1 = v->s1;
    t.s2 = v->s2;
    t.k0 = (float)((double)v->s0 / (double)fc.ext[2]);
    t.k1 = (float)((double)v->s1 / (double)fc.ext[1]);
    t.k2 = (float)((double)v->s2 / (double)fc.ext[0]);
    t.lb = v->lb;
    t.nbx = v->nbx;
    t.nby = v->nby;
    t.brick_bytes = v->brick_bytes;
    const uint64_t nbricks = (uint64_t)v->nbx * v->nby * v->nbz;
    t.nbytes32 = v->bytes <= 0xffffffffull && nbricks < (1ull << 24) ? (uint32_t)v->bytes : 0u;
    t.fmt = v->fmt;
    t.role = role;
    return t;
}

// ---------------------------------------------------------------------------
// kernel dispatch
// The generic march instances (runtime format; no scalar field bound).
template <int SF, int NM, bool COUNT>
static void launch_march_generic(const MarchArgs &a)
{
    const size_t lds = NM == NM_ANY ? 0 : 2 * (size_t)a.lut_n * sizeof(float4);
    hipLaunchKernelGGL((k_march<SF, NM, 3, COUNT, false, false>), dim3(a.nblocks), dim3(256), lds, a.stream, a.fc,
                       a.ts, a.tn, a.lut, a.lut_n, a.out, a.counts, a.skip, a.ntx, a.nblocks,
                       a.order, a.rot);
}

// The transparent-brick count of the current flags, once its copy to the
// host has completed (waiting for it when `wait`).  Returns whether
// flags_clear holds it.
static bool flags_count(hvr_ctx *c, bool wait)
{
    if (c->flags_count_known) return true;
    const hipError_t q = wait ? hipEventSynchronize(c->flags_ev) : hipEventQuery(c->flags_ev);
    if (q == hipSuccess) {
        c->flags_clear = *c->h_nclear;
        c->flags_count_known = true;
    } else if (q == hipErrorNotReady) {
        (void)hipGetLastError();   // still in flight, not an error
    }
    return c->flags_count_known;
}

// Transparent-brick flags of volume v for the current LUT.  Returns the flags
// when the march should step over transparent bricks: always in HVR_SKIP_ON; in
// HVR_SKIP_AUTO when enough bricks are transparent, or while the count is not
// back yet (skipping gives the same image, so the choice only affects speed);
// nullptr otherwise.  Where the LUT or the volume changed, `stale` says that
// launch_flags has to recompute them before the march.
static const uint8_t *brick_flags(hvr_ctx *c, const hvr_volume *v, bool *stale)
{
    if (c->skip_mode == HVR_SKIP_OFF || !v || !v->scalar_loaded || !c->d_nz) return nullptr;
    const uint64_t nb = (uint64_t)v->nbx * v->nby * v->nbz;
    // without flags the frame takes the non-skipping kernel: a failure here
    // is handled, not reported
    const auto none = [] {
        (void)hipGetLastError();
        return (const uint8_t *)nullptr;
    };
    if (!(c->flags_vol == v && c->flags_vol_gen == v->gen && c->flags_lut_gen == c->lut_gen)) {
        c->flags_vol = nullptr;
        if (!c->d_nclear) {
            if (hipMalloc(&c->d_nclear, 2 * sizeof(uint32_t)) != hipSuccess) return none();
            hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, c->stream, c->d_nclear, 2, 0u);
        }
        if (nb > c->flags_cap) {
            if (hipStreamSynchronize(c->stream) != hipSuccess) return none();
            (void)hipFree(c->d_flags);
            c->d_flags = nullptr;
            c->flags_cap = 0;
            if (dev_malloc(c->device, (void **)&c->d_flags, nb) != hipSuccess) return none();
            c->flags_cap = nb;
        }
        *stale = true;
        return c->d_flags;
    }
    if (c->skip_mode == HVR_SKIP_ON) return c->d_flags;
    if (!flags_count(c, false)) return c->d_flags;   // not back yet: skipping is exact either way
    return (double)c->flags_clear >= kSkipAutoFraction * (double)c->flags_total ? c->d_flags : nullptr;
}

// The flags of volume v recomputed (memory is there, brick_flags); their count
// comes back to the host without a wait.  Whether the march can use them.
static bool launch_flags(hvr_ctx *c, const hvr_volume *v)
{
    uint32_t *count = c->d_nclear + c->nclear_slot;
    hipLaunchKernelGGL(k_brick_flags, dim3(clearance_tiles(v->nbx, v->nby, v->nbz)), dim3(kClearThreads), 0,
                       c->stream, (const float2 *)v->d_range, (int)v->nbx, (int)v->nby, (int)v->nbz,
                       (const int *)c->d_nz, c->lut_n, c->d_flags, count, c->d_nclear + (c->nclear_slot ^ 1));
    bool ok = hipGetLastError() == hipSuccess;
    if (ok) c->nclear_slot ^= 1;
    ok = ok && hipMemcpyAsync(c->h_nclear, count, sizeof(uint32_t), hipMemcpyDeviceToHost, c->stream) == hipSuccess &&
         hipEventRecord(c->flags_ev, c->stream) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        return false;
    }
    c->flags_vol = v;
    c->flags_vol_gen = v->gen;
    c->flags_lut_gen = c->lut_gen;
    c->flags_count_known = false;
    c->flags_total = (uint64_t)v->nbx * v->nby * v->nbz;
    return true;
}

// Whether a volume is read through buffer loads (32-bit offsets, 24-bit brick
// indices).
static bool volume_buf(const hvr_volume *v)
{
    return v->bytes <= 0xffffffffull && (uint64_t)v->nbx * v->nby * v->nbz < (1ull << 24);
}

// The largest iteration bound that a frame's rays can have.
static double ray_steps(const float *bmin, const float *bmax, double step, int max_steps)
{
    double d2 = 0.0;
    for (int k = 0; k < 3; ++k) d2 += ((double)bmax[k] - bmin[k]) * ((double)bmax[k] - bmin[k]);
    return std::min((double)max_steps, std::sqrt(d2) / step);
}
static double ray_steps(const FrameConst &fc) { return ray_steps(fc.bmin, fc.bmax, fc.step, fc.max_steps); }

// How a frame is marched: the fast instances of the scalar volume's format
// (nm >= 0: normals from the same texels, as (rho, 0, 0) of the same volume,
// or unbound; brick edge 8 or 16), with transparent-brick skipping when the
// flags say so and buffer loads below 4 GiB, else the generic instance.
struct MarchPlan {
    int nm;
    const uint8_t *skip;
    bool stale;   // skip is to be recomputed first (launch_flags)
    bool buf;
    int lanes;
};
static MarchPlan march_plan(hvr_ctx *c, const FrameConst &fc, bool count)
{
    MarchPlan m = {-1, nullptr, false, false, 1};
    const hvr_volume *S = c->scalar_vol, *N = c->normal_vol;
    if (c->lut_n > kLutLdsMax || !S || c->scalar_role != HVR_ROLE_SCALAR || !(S->lb == 3 || S->lb == 4)) return m;
    if (!N) m.nm = NM_ZERO;
    else if (N == S && c->normal_role == HVR_ROLE_SCALAR) m.nm = NM_ALIAS;
    else if (N == S && c->normal_role == HVR_ROLE_NORMAL && fmt_has_normal(S->fmt)) m.nm = NM_SAME;
    if (m.nm < 0) return m;
    m.skip = brick_flags(c, S, &m.stale);
    m.buf = volume_buf(S) && !c->force_global;
    if (m.buf && !count)
        m.lanes = march_lanes((long long)c->W * c->H, resident_rays(c), m.skip != nullptr, ray_steps(fc),
                              texel_bytes(S->fmt), S->bytes);
    return m;
}

// The march of one frame into `out` (W*H RGBA8 on the device).
static void launch_march(hvr_ctx *c, const FrameConst &fc, uchar4 *out, bool count, const MarchPlan &m,
                         const uint32_t *order)
{
    MarchArgs a;
    a.fc = fc;
    a.lanes = m.lanes;
    a.order = order;
    const MarchTile bt = march_tile(m.lanes);
    a.ntx = (c->W + (1 << bt.lbw) - 1) >> bt.lbw;
    a.nblocks = a.ntx * ((c->H + (1 << bt.lbh) - 1) >> bt.lbh);
    a.rot = row_rotation(a.ntx);
    const hvr_volume *S = c->scalar_vol, *N = c->normal_vol;
    a.ts = tex_desc(S, c->scalar_role, fc);
    a.tn = tex_desc(N, c->normal_role, fc);
    a.lut = (const float4 *)c->d_lut;
    a.lut_n = c->lut_n;
    a.out = out;
    a.counts = c->d_counts;
    a.skip = m.skip;
    a.stream = c->stream;
    c->skip_used = 0;
    if (c->lut_n <= kLutLdsMax && !S && !N) {
        a.tn = a.ts = tex_desc(nullptr, 0, fc);
        if (count) launch_march_generic<TF_NONE, NM_ZERO, true>(a);
        else launch_march_generic<TF_NONE, NM_ZERO, false>(a);
        return;
    }
    if (m.nm >= 0) {
        a.tn = tex_desc(nullptr, 0, fc);
        c->skip_used = m.skip != nullptr;
        switch (S->fmt) {   // every format with a scalar field is a fast one
#define HVR_CASE(F) \
    case F: launch_march_##F(a, m.nm, S->lb, count, m.skip != nullptr, m.buf); break;
            HVR_FAST_FORMATS(HVR_CASE)
#undef HVR_CASE
        }
        return;
    }
    if (count) launch_march_generic<TF_NONE, NM_ANY, true>(a);
    else launch_march_generic<TF_NONE, NM_ANY, false>(a);
}

static int enqueue_frame(hvr_ctx *c, bool count, uchar4 *dst, bool count_shaded = false,
                         uint8_t *touched = nullptr)
{
    FrameConst fc = frame_const(c);
    fc.count_shaded = count_shaded;
    fc.touched = touched;
    // events of this frame: the context's own, or the next slots of an
    // open timing region; hvr_last_kernel_ms reads the frame's events
    // (each event is a packet of its own on the stream, for up to 5 us of the
    // frame: a frame in row order has no first event, and flags that are to be
    // recomputed count as the march's)
    hipEvent_t e0 = c->ev[0], e1 = c->ev[1], e2 = c->ev[2];
    const int timed = c->tev && c->timing_n < c->timing_max ? c->timing_n++ : -1;
    if (timed >= 0) {
        const size_t k = 3 * (size_t)timed;
        e0 = (*c->tev)[k];
        e1 = (*c->tev)[k + 1];
        e2 = (*c->tev)[k + 2];
    }
    MarchPlan plan = march_plan(c, fc, count);
    const MarchTile bt = march_tile(plan.lanes);
    const int ntx = (c->W + (1 << bt.lbw) - 1) >> bt.lbw, nty = (c->H + (1 << bt.lbh) - 1) >> bt.lbh;
    // cost-ordered dispatch (hvr_set_dispatch_order): the blocks of the
    // first multiple-of-8 block rows are filed by k_order_blocks and marched
    // in decreasing order of their rays' iteration bounds
    const int head_rows = nty >> 3 << 3, cap = (head_rows >> 3) * ntx;
    const bool ordered =
        head_rows > 0 && (c->order_mode == HVR_ORDER_ON ||
                          (c->order_mode == HVR_ORDER_AUTO &&
                           order_auto((long long)ntx * nty, (long long)c->W * c->H, resident_rays(c),
                                      plan.skip != nullptr, plan.lanes, ray_steps(fc))));
    if (ordered) {
        const size_t words = (size_t)head_rows * ntx * (1 + kOrderBuckets);
        if (words > c->order_words) {
            HIPCHK(hipStreamSynchronize(c->stream));
            (void)hipFree(c->d_order);
            c->d_order = nullptr;
            c->order_words = 0;
            HIPCHK(dev_malloc(c->device, (void **)&c->d_order, words * sizeof(uint32_t)));
            c->order_words = words;
        }
    }
    c->order_used = ordered;
    if (ordered) {
        // the blocks of the head rows only (the others keep row order)
        HIPCHK(hipEventRecord(e0, c->stream));
        hipLaunchKernelGGL(k_order_blocks, dim3(8), dim3(kOrderThreads), 0, c->stream, fc, c->d_order,
                           c->d_order + (size_t)head_rows * ntx, ntx, head_rows, cap, bt.lbw, bt.lbh);
        HIPCHK(hipGetLastError());
    }
    if (timed >= 0) (*c->tev_ordered)[(size_t)timed] = ordered;
    // the march sets up its rays itself
    HIPCHK(hipEventRecord(e1, c->stream));
    if (plan.stale && !launch_flags(c, c->scalar_vol)) plan.skip = nullptr;
    const bool host = !dst && c->readback_mode == HVR_READBACK_DIRECT;
    launch_march(c, fc, dst ? dst : host ? (uchar4 *)c->h_pinned_dev : c->d_out, count, plan,
                 ordered ? c->d_order : nullptr);
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(e2, c->stream));
    c->last_ev[0] = ordered ? e0 : e1;
    c->last_ev[1] = e1;
    c->last_ev[2] = e2;
    c->events_recorded = true;
    if (!dst) c->last_host = host;
    return HVR_OK;
}

// Per-device address of the no-allocation entry point's scratch array,
// looked up once per device at context creation (defined with the batches).
static void noalloc_setup(int device);

// ---------------------------------------------------------------------------
// C ABI
// Build brick rows [by0, by1) of brick layers [bz0, bz1) of volume v (k_build)
// from the source in `a`, whose planes lie `a.plane` voxels apart.
template <int F>
static void launch_build(const hvr_volume *v, const BuildArgs &a, unsigned blocks)
{
    const hipStream_t st = v->ctx->stream;
    const uint64_t voxels = (uint64_t)v->s0 * v->s1 * v->s2;
    // from a field, and more than the last cache (256 MB) holds of both: ONCE
    // gains nothing up to 289 MiB of both (0.98-1.03 in ten sizes), 2-7 % at 295-315,
    // 3-12 % at 340-375 and 14-36 % from 380 to 464
    const bool once = a.field && 4 * voxels + v->bytes >= 288ull << 20;
    // voxel offsets of 32 bits where the field's floats fit 4 GiB
    const auto go = [&](auto index) {
        using I = decltype(index);
        const auto launch = [&](auto o) {
            constexpr bool ONCE = decltype(o)::value;
            if (v->lb == 2) hipLaunchKernelGGL((k_build<F, 2, I, ONCE>), dim3(blocks), dim3(256), 0, st, a);
            else if (v->lb == 3) hipLaunchKernelGGL((k_build<F, 3, I, ONCE>), dim3(blocks), dim3(256), 0, st, a);
            else hipLaunchKernelGGL((k_build<F, 4, I, ONCE>), dim3(blocks), dim3(256), 0, st, a);
        };
        if constexpr (fmt_has_normal(F)) {
            if (once) return launch(std::true_type{});
        }
        launch(std::false_type{});
    };
    if (voxels < (1ull << 30) && !v->ctx->force_wide) go(uint32_t(0));
    else go(uint64_t(0));
}
static int build_group(const hvr_volume *v, BuildArgs a, uint32_t by0, uint32_t by1, uint32_t bz0, uint32_t bz1)
{
    a.dst = (char *)v->d_texels;
    a.s0 = v->s0;
    a.s1 = v->s1;
    a.s2 = v->s2;
    a.nbx = v->nbx;
    a.nby = v->nby;
    a.inv_n12 = 1.0 / ((double)v->s1 * v->s2);
    a.inv_s2 = 1.0 / v->s2;
    a.by0 = by0;
    a.rows = by1 - by0;
    a.bz0 = bz0;
    a.runs = (uint64_t)((v->nbx + build_bricks(v->lb) - 1) / build_bricks(v->lb)) * a.rows * (bz1 - bz0);
    const unsigned blocks = (unsigned)std::min<uint64_t>(a.runs, (1u << 24) - 1);   // below 2^32 threads
    switch (v->fmt) {
#define HVR_BUILD(F) \
    case F: launch_build<F>(v, a, blocks); break;
        HVR_BUILD(TF_S_F32)
        HVR_BUILD(TF_S_F16)
        HVR_BUILD(TF_S_U8)
        HVR_BUILD(TF_N_F32)
        HVR_BUILD(TF_N_SN8)
        HVR_BUILD(TF_C_F32_F32)
        HVR_BUILD(TF_C_F16_F32)
        HVR_BUILD(TF_C_U8_F32)
        HVR_BUILD(TF_C_F32_SN8)
        HVR_BUILD(TF_C_F16_SN8)
        HVR_BUILD(TF_C_U8_SN8)
        HVR_BUILD(TF_C_F16_F16)
        HVR_BUILD(TF_N_F16)
#undef HVR_BUILD
    default: return fail(HVR_EINVAL, "bad texel format");
    }
    HIPCHK(hipGetLastError());
    return HVR_OK;
}

static size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// The context's staging buffer, of at least `need` bytes.
static int need_stage(hvr_ctx *c, size_t need)
{
    if (c->stage_bytes >= need) return HVR_OK;
    HIPCHK(hipStreamSynchronize(c->stream));
    (void)hipFree(c->d_stage);
    c->d_stage = nullptr;
    c->stage_bytes = 0;
    HIPCHK(dev_malloc(c->device, (void **)&c->d_stage, need));
    c->stage_bytes = need;
    return HVR_OK;
}
static constexpr size_t kMaxStage = (size_t)256 << 20;   // what stays allocated

// Whether `src` is plain host memory, which the device cannot read by itself:
// not pinned, registered, managed or its own.
static bool pageable(const void *src)
{
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, src) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return at.type == hipMemoryTypeUnregistered;
}

// Host data to the device, in stream order.  From pageable memory one thread of
// the runtime copies into pinned memory, at 30 GB/s; here four threads do
// (CopyPool), piece by piece through a ring of three pinned parts, while the
// pieces before cross the link (44 GB/s).  The caller's pageable data is read
// when this returns.  What the device can read by itself it copies by itself
// (pinned data at the link's 53 GB/s; 85 MB 1.62 ms, through the ring 1.94);
// less than a piece, and where the ring cannot be had, goes the runtime's way.
static constexpr size_t kUploadPiece = (size_t)4 << 20;
static int upload_host(hvr_ctx *c, void *dst, const void *src, size_t bytes)
{
    const bool ring = bytes >= kUploadPiece && pageable(src);
    if (ring) HVR_FAULT_POINT("hvr_upload_ring");
    if (ring && !c->h_up) {
        bool ok = hipHostMalloc((void **)&c->h_up, 3 * kUploadPiece, hipHostMallocDefault) == hipSuccess;
        for (hipEvent_t &e : c->up_ev)
            if (ok && !e) ok = hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
        if (!ok) {
            (void)hipGetLastError();
            if (c->h_up) (void)hipHostFree(c->h_up);
            c->h_up = nullptr;
        }
    }
    if (!ring || !c->h_up) {
        HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c->stream));
        return HVR_OK;
    }
    for (size_t at = 0, k = 0; at < bytes; at += kUploadPiece, ++k) {
        const size_t n = std::min(kUploadPiece, bytes - at);
        char *part = c->h_up + k % 3 * kUploadPiece;
        HIPCHK(hipEventSynchronize(c->up_ev[k % 3]));   // at once when never recorded
        hvr::CopyPool::get().copy((uint8_t *)part, (const uint8_t *)src + at, n);
        HIPCHK(hipMemcpyAsync((char *)dst + at, part, n, hipMemcpyHostToDevice, c->stream));
        HIPCHK(hipEventRecord(c->up_ev[k % 3], c->stream));
    }
    return HVR_OK;
}

// Device memory for a whole field while a volume is built from it: the staging
// buffer up to kMaxStage, else an allocation given back (after the stream's
// work) at the end of the scope.
struct FieldBuffer {
    hvr_ctx *c;
    char *p = nullptr;
    bool own = false, idle = false;   // idle: the stream has been waited for since the last use
    explicit FieldBuffer(hvr_ctx *ctx) : c(ctx) {}
    FieldBuffer(const FieldBuffer &) = delete;
    int get(size_t bytes)
    {
        if (bytes <= kMaxStage) {
            if (const int rc = need_stage(c, bytes)) return rc;
            p = (char *)c->d_stage;
            return HVR_OK;
        }
        HIPCHK(dev_malloc(c->device, (void **)&p, bytes));
        own = true;
        return HVR_OK;
    }
    ~FieldBuffer()
    {
        // also after a failure: nothing queued may still read the buffer
        // (or, in the caller's frame, the host memory copied from)
        if (!idle) (void)hipStreamSynchronize(c->stream);
        if (own) (void)hipFree(p);
    }
};

extern "C" {

int hvr_abi_version(void) { return HVR_ABI_VERSION; }

int hvr_debug_inject_fault(const char *function, int code, int after)
{
    std::lock_guard<std::mutex> lock(g_fault_mu);
    if (!function) {
        g_fault_armed.store(false);
        g_fault_after = -1;
        g_fault_fn.clear();
        return HVR_OK;
    }
    if (code >= 0 || after < 0) return fail(HVR_EINVAL, "injected faults need a negative code and after >= 0");
    g_fault_fn = function;
    g_fault_code = code;
    g_fault_after = after;
    g_fault_armed.store(true);
    return HVR_OK;
}

const char *hvr_last_error(void) { return g_err.c_str(); }

int hvr_device_count(int *count)
{
    if (!count) return fail(HVR_EINVAL, "count is null");
    HIPCHK(hipGetDeviceCount(count));
    return HVR_OK;
}

int hvr_device_memory(int device, unsigned long long *free_bytes, unsigned long long *total_bytes)
{
    HIPCHK(hipSetDevice(device));
    size_t f = 0, t = 0;
    HIPCHK(hipMemGetInfo(&f, &t));
    if (free_bytes) *free_bytes = f + spare_bytes(device);
    if (total_bytes) *total_bytes = t;
    return HVR_OK;
}

int hvr_kept_memory(hvr_ctx *c, unsigned long long *bytes)
{
    if (!c || !bytes) return fail(HVR_EINVAL, "null argument");
    *bytes = spare_bytes(c->device) + c->stage_bytes;
    return HVR_OK;
}

int hvr_trim(hvr_ctx *c)
{
    if (!c) return fail(HVR_EINVAL, "ctx is null");
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(hipStreamSynchronize(c->stream));
    size_t b;
    if (void *spare = spare_take(c->device, &b)) HIPCHK(hipFree(spare));
    float *const stage = c->d_stage;
    c->d_stage = nullptr;
    c->stage_bytes = 0;
    if (stage) HIPCHK(hipFree(stage));
    char *const ring = c->h_up;
    c->h_up = nullptr;
    if (ring) HIPCHK(hipHostFree(ring));
    return HVR_OK;
}

int hvr_create(int device, int width, int height, hvr_ctx **out)
{
    HVR_FAULT_POINT("hvr_create");
    if (!out) return fail(HVR_EINVAL, "out is null");
    *out = nullptr;
    if (width <= 0 || height <= 0 || (long long)width * height > (1ll << 28))
        return fail(HVR_EINVAL, "width and height must be positive (at most 2^28 pixels)");
    HIPCHK(hipSetDevice(device));
    hvr_ctx *c = new hvr_ctx();
    memset(c, 0, sizeof(*c));
    c->device = device;
    context_count(device, 1);
    c->W = width;
    c->H = height;
    c->brick_log2 = 3;
    c->skip_mode = HVR_SKIP_AUTO;
    c->order_mode = HVR_ORDER_AUTO;
    c->readback_mode = HVR_READBACK_DIRECT;
    const char *gather = getenv("HVR_GATHER");
    c->force_global = gather && strcmp(gather, "global") == 0;
    const char *build = getenv("HVR_BUILD");
    c->force_wide = build && strcmp(build, "wide") == 0;
    c->max_stage = kMaxStage;
    if (const char *stage = getenv("HVR_STAGE"))
        if (const unsigned long long n = strtoull(stage, nullptr, 10)) c->max_stage = (size_t)std::min<uint64_t>(n, kMaxStage);
    const size_t npix = (size_t)width * height;
    noalloc_setup(device);
    hipError_t e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&c->ncu, hipDeviceAttributeMultiprocessorCount, device);
    if (e == hipSuccess) e = dev_malloc(device, (void **)&c->d_out, npix * sizeof(uchar4));
    if (e == hipSuccess) e = hipHostMalloc(&c->h_pinned, npix * 4, hipHostMallocDefault);
    if (e == hipSuccess) e = hipHostGetDevicePointer(&c->h_pinned_dev, c->h_pinned, 0);
    if (e == hipSuccess) e = hipHostMalloc((void **)&c->h_nclear, sizeof(uint32_t), hipHostMallocDefault);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&c->flags_ev, hipEventDisableTiming);
    for (int i = 0; i < 4 && e == hipSuccess; ++i) e = hipEventCreateWithFlags(&c->lut_ev[i], hipEventDisableTiming);
    for (int i = 0; i < 4 && e == hipSuccess; ++i) e = hipEventCreate(&c->ev[i]);
    for (int i = 0; i < 4 && e == hipSuccess; ++i) e = hipEventCreateWithFlags(&c->rev[i], hipEventDisableTiming);
    if (e == hipSuccess) {
        // unbound LUT: a 1-texel (0, 0, 0, 1) texture (GL incomplete texture)
        c->lut_cap = 1;
        c->lut_n = 1;
        e = dev_malloc(device, (void **)&c->d_lut, sizeof(float4));
        const float4 unbound = make_float4(0.f, 0.f, 0.f, 1.f);
        if (e == hipSuccess) e = hipMemcpy(c->d_lut, &unbound, sizeof(float4), hipMemcpyHostToDevice);
    }
    if (e == hipSuccess) e = hipMemset(c->d_out, 0, npix * sizeof(uchar4));
    if (e != hipSuccess) {
        hvr_destroy(c);
        return fail_hip(e, "hvr_create");
    }
    c->pix_cap = npix;
    *out = c;
    return HVR_OK;
}

int hvr_resize(hvr_ctx *c, int width, int height)
{
    HVR_FAULT_POINT("hvr_resize");
    if (!c) return fail(HVR_EINVAL, "ctx is null");
    if (width <= 0 || height <= 0 || (long long)width * height > (1ll << 28))
        return fail(HVR_EINVAL, "width and height must be positive (at most 2^28 pixels)");
    HIPCHK(hipSetDevice(c->device));
    const size_t npix = (size_t)width * height;
    // Frames in flight keep their own sizes (kernel arguments); only
    // buffers that must grow wait for them.
    if (npix > c->pix_cap) {
        HIPCHK(hipStreamSynchronize(c->stream));
        (void)hipFree(c->d_out);
        if (c->h_pinned) (void)hipHostFree(c->h_pinned);
        c->d_out = nullptr;
        c->h_pinned = nullptr;
        c->h_pinned_dev = nullptr;
        c->last_host = false;
        c->pix_cap = 0;
        HIPCHK(dev_malloc(c->device, (void **)&c->d_out, npix * sizeof(uchar4)));
        HIPCHK(hipHostMalloc(&c->h_pinned, npix * 4, hipHostMallocDefault));
        HIPCHK(hipHostGetDevicePointer(&c->h_pinned_dev, c->h_pinned, 0));
        HIPCHK(hipMemset(c->d_out, 0, npix * sizeof(uchar4)));
        c->pix_cap = npix;
    }
    c->W = width;
    c->H = height;
    return HVR_OK;
}

int hvr_destroy(hvr_ctx *c)
{
    if (!c) return HVR_OK;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    (void)hipFree(c->d_out);
    (void)hipFree(c->d_counts);
    (void)hipFree(c->d_lut);
    (void)hipFree(c->d_stage);
    (void)hipFree(c->d_nz);
    (void)hipFree(c->d_flags);
    (void)hipFree(c->d_nclear);
    (void)hipFree(c->d_order);
    if (c->h_pinned) (void)hipHostFree(c->h_pinned);
    if (c->h_nclear) (void)hipHostFree(c->h_nclear);
    if (c->h_up) (void)hipHostFree(c->h_up);
    for (hipEvent_t e : c->up_ev)
        if (e) (void)hipEventDestroy(e);
    if (c->flags_ev) (void)hipEventDestroy(c->flags_ev);
    for (int i = 0; i < 4; ++i) {
        if (c->ev[i]) (void)hipEventDestroy(c->ev[i]);
        if (c->rev[i]) (void)hipEventDestroy(c->rev[i]);
        if (c->lut_ev[i]) (void)hipEventDestroy(c->lut_ev[i]);
        if (c->h_lut_stage[i]) (void)hipHostFree(c->h_lut_stage[i]);
    }
    if (c->tev) {
        for (hipEvent_t e : *c->tev) (void)hipEventDestroy(e);
        delete c->tev;
        delete c->tev_ordered;
    }
    if (c->stream) (void)hipStreamDestroy(c->stream);
    context_count(c->device, -1);
    delete c;
    return HVR_OK;
}

int hvr_set_empty_skip(hvr_ctx *c, int mode)
{
    if (!c) return fail(HVR_EINVAL, "ctx is null");
    if (mode != HVR_SKIP_OFF && mode != HVR_SKIP_ON && mode != HVR_SKIP_AUTO)
        return fail(HVR_EINVAL, "skip mode must be HVR_SKIP_OFF, HVR_SKIP_ON or HVR_SKIP_AUTO");
    c->skip_mode = mode;
    return HVR_OK;
}

int hvr_set_readback(hvr_ctx *c, int mode)
{
    if (!c) return fail(HVR_EINVAL, "ctx is null");
    if (mode != HVR_READBACK_COPY && mode != HVR_READBACK_DIRECT)
        return fail(HVR_EINVAL, "readback mode must be HVR_READBACK_COPY or HVR_READBACK_DIRECT");
    c->readback_mode = mode;
    return HVR_OK;
}

int hvr_set_dispatch_order(hvr_ctx *c, int mode)
{
    if (!c) return fail(HVR_EINVAL, "ctx is null");
    if (mode != HVR_ORDER_OFF && mode != HVR_ORDER_ON && mode != HVR_ORDER_AUTO)
        return fail(HVR_EINVAL, "dispatch order mode must be HVR_ORDER_OFF, HVR_ORDER_ON or HVR_ORDER_AUTO");
    c->order_mode = mode;
    return HVR_OK;
}

int hvr_dispatch_order_info(hvr_ctx *c, int *used)
{
    if (!c) return fail(HVR_EINVAL, "ctx is null");
    if (used) *used = c->order_used;
    return HVR_OK;
}

int hvr_skip_info(hvr_ctx *c, unsigned long long *clear_bricks, unsigned long long *bricks, int *used)
{
    if (!c) return fail(HVR_EINVAL, "ctx is null");
    const bool valid = c->flags_vol != nullptr;
    if (valid && !flags_count(c, true)) return fail(HVR_EDEVICE, "hvr_skip_info: reading the brick count failed");
    if (clear_bricks) *clear_bricks = valid ? c->flags_clear : 0;
    if (bricks) *bricks = valid ? c->flags_total : 0;
    if (used) *used = c->skip_used;
    return HVR_OK;
}

int hvr_set_brick_log2(hvr_ctx *c, int lb)
{
    if (!c) return fail(HVR_EINVAL, "ctx is null");
    if (lb < 2 || lb > 4) return fail(HVR_EINVAL, "brick log2 must be in [2, 4]");
    c->brick_log2 = lb;
    return HVR_OK;
}

static int texel_format(int sf, int nf)
{
    if (nf == HVR_NORMAL_NONE) {
        if (sf == HVR_SCALAR_F32) return TF_S_F32;
        if (sf == HVR_SCALAR_F16) return TF_S_F16;
        if (sf == HVR_SCALAR_U8) return TF_S_U8;
        return -1;
    }
    if (nf == HVR_NORMAL_F32X3) {
        if (sf == HVR_SCALAR_NONE) return TF_N_F32;
        if (sf == HVR_SCALAR_F32) return TF_C_F32_F32;
        if (sf == HVR_SCALAR_F16) return TF_C_F16_F32;
        if (sf == HVR_SCALAR_U8) return TF_C_U8_F32;
        return -1;
    }
    if (nf == HVR_NORMAL_SN8X3) {
        if (sf == HVR_SCALAR_NONE) return TF_N_SN8;
        if (sf == HVR_SCALAR_F32) return TF_C_F32_SN8;
        if (sf == HVR_SCALAR_F16) return TF_C_F16_SN8;
        if (sf == HVR_SCALAR_U8) return TF_C_U8_SN8;
        return -1;
    }
    if (nf == HVR_NORMAL_F16X3) {
        // 8-byte texels; FP32 and UNORM8 scalars are not paired with it
        if (sf == HVR_SCALAR_NONE) return TF_N_F16;
        if (sf == HVR_SCALAR_F16) return TF_C_F16_F16;
    }
    return -1;
}

int hvr_volume_create(hvr_ctx *c, int s0, int s1, int s2, int sf, int nf, hvr_volume **out)
{
    HVR_FAULT_POINT("hvr_volume_create");
    if (!c || !out) return fail(HVR_EINVAL, "null argument");
    *out = nullptr;
    if (s0 <= 0 || s1 <= 0 || s2 <= 0) return fail(HVR_EINVAL, "volume dimensions must be positive");
    const int fmt = texel_format(sf, nf);
    if (fmt < 0) return fail(HVR_EINVAL, "unsupported scalar/normal format combination");
    if (s0 > (1 << 20) || s1 > (1 << 20) || s2 > (1 << 20))
        return fail(HVR_EINVAL, "volume dimension above 2^20");
    const int lb = c->brick_log2;
    const uint64_t E = (1u << lb) + 1u;
    hvr_volume *v = new hvr_volume();
    memset(v, 0, sizeof(*v));
    v->ctx = c;
    v->s0 = s0;
    v->s1 = s1;
    v->s2 = s2;
    v->fmt = fmt;
    v->lb = lb;
    v->nbx = bricks_along(s0, lb);
    v->nby = bricks_along(s1, lb);
    v->nbz = bricks_along(s2, lb);
    v->brick_bytes = (uint32_t)(E * E * E * (uint64_t)texel_bytes(fmt));
    const uint64_t nbricks = (uint64_t)v->nbx * v->nby * v->nbz;
    if (nbricks >= (1ull << 32)) {
        delete v;
        return fail(HVR_EINVAL, "volume too large (brick index exceeds 32 bits)");
    }
    v->bytes = nbricks * v->brick_bytes;
    const size_t range_at = align_up((size_t)v->bytes, 256),
                 bytes = fmt_has_scalar(fmt) ? range_at + (size_t)nbricks * sizeof(float2) : (size_t)v->bytes;
    hipError_t e = hipSetDevice(c->device);
    if (e == hipSuccess) e = block_alloc(c->device, &v->d_texels, bytes, &v->block_bytes);
    if (e != hipSuccess) {
        delete v;
        return fail_hip(e, "hvr_volume_create");
    }
    if (fmt_has_scalar(fmt)) v->d_range = (float2 *)((char *)v->d_texels + range_at);
    *out = v;
    return HVR_OK;
}

// The scalar (part 1) or normal (part 2) field of volume v from host data, in
// groups of bricks whose source fits the staging buffer (upload_group).
static int upload_part(hvr_volume *v, const float *data, int part)
{
    hvr_ctx *c = v->ctx;
    HIPCHK(hipSetDevice(c->device));
    const uint64_t comps = part == 1 ? 1 : 3, plane = (uint64_t)v->s0 * v->s1;
    const size_t row = (size_t)(v->s0 * comps * sizeof(float));
    const UploadGroup g = upload_group(row, v->s1, v->s2, v->lb, c->max_stage);
    FieldBuffer f(c);
    if (const int rc = f.get((size_t)g.bytes)) return rc;
    BuildArgs a;
    memset(&a, 0, sizeof(a));
    (part == 1 ? a.scalar : a.normal) = (const float *)f.p;
    a.keep = part == 1 ? v->normals_loaded : v->scalar_loaded;
    a.range = part == 1 ? v->d_range : nullptr;
    for (uint32_t bz = 0; bz < v->nbz; bz += g.layers)
        for (uint32_t by = 0; by < v->nby; by += g.rows) {
            const int z0 = source_begin(bz, v->lb, v->s2), z1 = source_end(bz, g.layers, v->lb, v->s2),
                      y0 = source_begin(by, v->lb, v->s1), y1 = source_end(by, g.rows, v->lb, v->s1);
            const uint64_t lines = (uint64_t)(y1 - y0);
            a.plane = lines * v->s0;
            a.first = (uint64_t)z0 * a.plane + (uint64_t)y0 * v->s0;
            const auto at = [&](int z) { return data + ((uint64_t)z * plane + (uint64_t)y0 * v->s0) * comps; };
            if (lines == (uint64_t)v->s1) {
                if (const int rc = upload_host(c, f.p, at(z0), (size_t)(z1 - z0) * lines * row)) return rc;
            } else {
                for (int z = z0; z < z1; ++z)
                    if (const int rc = upload_host(c, f.p + (size_t)(z - z0) * lines * row, at(z), lines * row)) return rc;
            }
            if (const int rc = build_group(v, a, by, std::min(v->nby, by + g.rows), bz, std::min(v->nbz, bz + g.layers)))
                return rc;
            // the staging buffer is reused by the next group
            HIPCHK(hipStreamSynchronize(c->stream));
        }
    f.idle = true;
    return HVR_OK;
}

// Scalar part (and, with `normals`, the normal part computed on the device)
// of volume v from a device float32 field in numpy C order.
static int volume_from_field(hvr_volume *v, const float *d_field, bool normals)
{
    hvr_ctx *c = v->ctx;
    if (!fmt_has_scalar(v->fmt)) return fail(HVR_EINVAL, "the volume has no scalar field");
    BuildArgs a;
    memset(&a, 0, sizeof(a));
    normals = normals && fmt_has_normal(v->fmt);
    (normals ? a.field : a.scalar) = d_field;
    a.keep = !normals && v->normals_loaded;
    a.range = v->d_range;
    a.plane = (uint64_t)v->s0 * v->s1;
    if (const int rc = build_group(v, a, 0, v->nby, 0, v->nbz)) return rc;
    HIPCHK(hipStreamSynchronize(c->stream));
    v->scalar_loaded = true;
    if (normals) v->normals_loaded = true;
    ++v->gen;
    return HVR_OK;
}

int hvr_volume_upload_scalar_normals(hvr_volume *v, const float *data)
{
    HVR_FAULT_POINT("hvr_volume_upload_scalar_normals");
    if (!v || !data) return fail(HVR_EINVAL, "null argument");
    if (!fmt_has_scalar(v->fmt) || !fmt_has_normal(v->fmt))
        return fail(HVR_ESTATE, "the volume needs scalar and normal fields");
    if (v->s0 < 2 || v->s1 < 2 || v->s2 < 2)
        return fail(HVR_EINVAL, "normals need at least 2 voxels along every axis (np.gradient)");
    hvr_ctx *c = v->ctx;
    HIPCHK(hipSetDevice(c->device));
    const size_t bytes = (size_t)v->s0 * v->s1 * v->s2 * sizeof(float);
    FieldBuffer f(c);
    if (const int rc = f.get(bytes)) return rc;
    if (const int rc = upload_host(c, f.p, data, bytes)) return rc;
    return volume_from_field(v, (const float *)f.p, true);
}

int hvr_volume_generate_blobs(hvr_volume *v, int n_blobs, const double *centers, const double *sigmas,
                              const double *amps, double noise, unsigned long long seed)
{
    HVR_FAULT_POINT("hvr_volume_generate_blobs");
    if (!v || (n_blobs > 0 && (!centers || !sigmas || !amps))) return fail(HVR_EINVAL, "null argument");
    if (n_blobs < 0 || n_blobs > kMaxBlobs) return fail(HVR_EINVAL, "0 to 32 blobs");
    if (!fmt_has_scalar(v->fmt)) return fail(HVR_ESTATE, "the volume has no scalar field");
    const bool normals = fmt_has_normal(v->fmt);
    if (normals && (v->s0 < 2 || v->s1 < 2 || v->s2 < 2))
        return fail(HVR_EINVAL, "normals need at least 2 voxels along every axis (np.gradient)");
    hvr_ctx *c = v->ctx;
    HIPCHK(hipSetDevice(c->device));
    BlobSpec spec;
    memset(&spec, 0, sizeof(spec));
    spec.n = n_blobs;
    for (int b = 0; b < n_blobs; ++b) {
        for (int k = 0; k < 3; ++k) spec.c[3 * b + k] = centers[3 * b + k];
        spec.s[b] = sigmas[b];
        spec.a[b] = amps[b];
    }
    spec.noise = noise;
    spec.seed = seed;
    const uint64_t nvox = (uint64_t)v->s0 * v->s1 * v->s2, len = (uint64_t)v->s0 + v->s1 + v->s2;
    // the parameters, the factors, then the field
    const size_t fac_at = align_up(sizeof(spec), 256), field_at = fac_at + align_up(len * n_blobs * sizeof(double), 256);
    FieldBuffer f(c);
    if (const int rc = f.get(field_at + nvox * sizeof(float))) return rc;
    const BlobSpec *d_spec = (const BlobSpec *)f.p;
    double *fac = (double *)(f.p + fac_at);
    float *field = (float *)(f.p + field_at);
    if (hipMemcpyAsync(f.p, &spec, sizeof(spec), hipMemcpyHostToDevice, c->stream) != hipSuccess)
        return fail(HVR_EDEVICE, "staging the blob parameters failed");
    if (n_blobs)
        hipLaunchKernelGGL(k_blob_factors, dim3((unsigned)std::min<uint64_t>((len * n_blobs + 255) / 256, 1u << 20)),
                           dim3(256), 0, c->stream, fac, v->s0, v->s1, v->s2, d_spec);
    const uint64_t waves = (((uint64_t)v->s2 + 63) / 64) * (((uint64_t)v->s1 + kBlobRows - 1) / kBlobRows) * v->s0;
    hipLaunchKernelGGL(k_blob_field, dim3((unsigned)std::min<uint64_t>((waves + 3) / 4, (1u << 24) - 1)), dim3(256), 0,
                       c->stream, field, v->s0, v->s1, v->s2, d_spec, (const double *)fac);
    if (hipGetLastError() != hipSuccess) return fail(HVR_EDEVICE, "blob field kernel launch failed");
    return volume_from_field(v, field, normals);
}

int hvr_volume_upload_scalar(hvr_volume *v, const float *data)
{
    HVR_FAULT_POINT("hvr_volume_upload_scalar");
    if (!v || !data) return fail(HVR_EINVAL, "null argument");
    if (!fmt_has_scalar(v->fmt)) return fail(HVR_ESTATE, "volume has no scalar field");
    int rc = upload_part(v, data, 1);
    if (rc != HVR_OK) return rc;
    v->scalar_loaded = true;
    ++v->gen;
    return HVR_OK;
}

int hvr_volume_upload_normals(hvr_volume *v, const float *data)
{
    HVR_FAULT_POINT("hvr_volume_upload_normals");
    if (!v || !data) return fail(HVR_EINVAL, "null argument");
    if (!fmt_has_normal(v->fmt)) return fail(HVR_ESTATE, "volume has no normal field");
    int rc = upload_part(v, data, 2);
    if (rc == HVR_OK) {
        v->normals_loaded = true;
        ++v->gen;
    }
    return rc;
}

int hvr_volume_bytes(const hvr_volume *v, uint64_t *bytes)
{
    if (!v || !bytes) return fail(HVR_EINVAL, "null argument");
    *bytes = v->bytes;
    return HVR_OK;
}

int hvr_volume_destroy(hvr_volume *v)
{
    if (!v) return HVR_OK;
    hvr_ctx *c = v->ctx;
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    if (c->scalar_vol == v) c->scalar_vol = nullptr;
    if (c->normal_vol == v) c->normal_vol = nullptr;
    if (c->flags_vol == v) c->flags_vol = nullptr;
    block_free(c->device, v->d_texels, v->block_bytes);
    delete v;
    return HVR_OK;
}

int hvr_set_lut(hvr_ctx *c, const float *rgba, int n)
{
    HVR_FAULT_POINT("hvr_set_lut");
    if (!c) return fail(HVR_EINVAL, "ctx is null");
    if (n < 0 || (n > 0 && !rgba)) return fail(HVR_EINVAL, "bad LUT");
    HIPCHK(hipSetDevice(c->device));
    const float unbound[4] = {0.f, 0.f, 0.f, 1.f};
    const float *src = n > 0 ? rgba : unbound;
    const int cnt = n > 0 ? n : 1;
    // The copies are ordered on the stream after the frames already queued
    // (which read the previous LUT), through pinned staging, so a LUT change
    // does not wait for them; growing a buffer does.
    const size_t lut_bytes = (size_t)cnt * sizeof(float4), nz_bytes = ((size_t)cnt + 1) * sizeof(int);
    if (cnt > c->lut_cap || cnt > c->nz_cap || lut_bytes + nz_bytes > c->lut_stage_bytes)
        HIPCHK(hipStreamSynchronize(c->stream));
    if (cnt > c->lut_cap) {
        (void)hipFree(c->d_lut);
        c->d_lut = nullptr;
        c->lut_cap = 0;
        HIPCHK(dev_malloc(c->device, (void **)&c->d_lut, lut_bytes));
        c->lut_cap = cnt;
    }
    if (cnt > c->nz_cap) {
        (void)hipFree(c->d_nz);
        c->d_nz = nullptr;
        c->nz_cap = 0;
        HIPCHK(dev_malloc(c->device, (void **)&c->d_nz, nz_bytes));
        c->nz_cap = cnt;
    }
    if (lut_bytes + nz_bytes > c->lut_stage_bytes) {
        size_t want = 4096;
        while (want < lut_bytes + nz_bytes) want *= 2;
        for (int i = 0; i < 4; ++i) {
            if (c->h_lut_stage[i]) (void)hipHostFree(c->h_lut_stage[i]);
            c->h_lut_stage[i] = nullptr;
            c->lut_ev_live[i] = false;
        }
        c->lut_stage_bytes = 0;
        for (int i = 0; i < 4; ++i) HIPCHK(hipHostMalloc(&c->h_lut_stage[i], want, hipHostMallocDefault));
        c->lut_stage_bytes = want;
    }
    const int k = c->lut_slot;
    c->lut_slot = (k + 1) & 3;
    if (c->lut_ev_live[k]) HIPCHK(hipEventSynchronize(c->lut_ev[k]));
    char *stage = (char *)c->h_lut_stage[k];
    memcpy(stage, src, lut_bytes);
    lut_prefix_counts(src, cnt, (int *)(stage + lut_bytes));
    HIPCHK(hipMemcpyAsync(c->d_lut, stage, lut_bytes, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->d_nz, stage + lut_bytes, nz_bytes, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipEventRecord(c->lut_ev[k], c->stream));
    c->lut_ev_live[k] = true;
    c->lut_n = cnt;
    ++c->lut_gen;
    return HVR_OK;
}

static int check_params(const hvr_params *p)
{
    if (!(p->step > 0.f) || !(p->ref_step > 0.f)) return fail(HVR_EINVAL, "step sizes must be positive");
    if (p->max_steps < 0) return fail(HVR_EINVAL, "max_steps must be >= 0");
    for (int k = 0; k < 3; ++k) {
        // the float extent of the in-box test must be positive, with the
        // texel scale (size / extent) finite
        const float ext = p->bmax[k] - p->bmin[k];
        if (!std::isfinite(p->bmin[k]) || !std::isfinite(p->bmax[k]) || !(ext >= 1e-20f) || !std::isfinite(ext))
            return fail(HVR_EINVAL, "box bounds must be finite with bmax - bmin >= 1e-20 on every axis");
    }
    return HVR_OK;
}

int hvr_set_params(hvr_ctx *c, const hvr_params *p)
{
    HVR_FAULT_POINT("hvr_set_params");
    if (!c || !p) return fail(HVR_EINVAL, "null argument");
    if (const int rc = check_params(p)) return rc;
    c->params = *p;
    c->params_set = true;
    return HVR_OK;
}

int hvr_bind(hvr_ctx *c, hvr_volume *s, int srole, hvr_volume *n, int nrole)
{
    HVR_FAULT_POINT("hvr_bind");
    if (!c) return fail(HVR_EINVAL, "ctx is null");
    if ((s && s->ctx != c) || (n && n->ctx != c)) return fail(HVR_EINVAL, "volume belongs to another context");
    if (srole != HVR_ROLE_SCALAR && srole != HVR_ROLE_NORMAL) return fail(HVR_EINVAL, "bad scalar role");
    if (nrole != HVR_ROLE_SCALAR && nrole != HVR_ROLE_NORMAL) return fail(HVR_EINVAL, "bad normal role");
    for (int k = 0; k < 2; ++k) {
        const hvr_volume *v = k ? n : s;
        const int role = k ? nrole : srole;
        if (!v) continue;
        if (role == HVR_ROLE_SCALAR && !fmt_has_scalar(v->fmt)) return fail(HVR_EINVAL, "volume has no scalar field");
        if (role == HVR_ROLE_NORMAL && !fmt_has_normal(v->fmt)) return fail(HVR_EINVAL, "volume has no normal field");
    }
    // a volume that was never loaded reads as zeros (a load writes every texel)
    for (hvr_volume *v : {s, n})
        if (v && !v->scalar_loaded && !v->normals_loaded && !v->cleared) {
            HIPCHK(hipSetDevice(c->device));
            HIPCHK(hipMemsetAsync(v->d_texels, 0, (size_t)v->bytes, c->stream));
            HIPCHK(hipStreamSynchronize(c->stream));
            v->cleared = true;
        }
    c->scalar_vol = s;
    c->normal_vol = n;
    c->scalar_role = srole;
    c->normal_role = nrole;
    return HVR_OK;
}

int hvr_render_async(hvr_ctx *c)
{
    HVR_FAULT_POINT("hvr_render_async");
    if (!c) return fail(HVR_EINVAL, "ctx is null");
    HIPCHK(hipSetDevice(c->device));
    return enqueue_frame(c, false, nullptr);
}

int hvr_render_async_to(hvr_ctx *c, void *dst)
{
    HVR_FAULT_POINT("hvr_render_async_to");
    if (!c) return fail(HVR_EINVAL, "ctx is null");
    HIPCHK(hipSetDevice(c->device));
    return enqueue_frame(c, false, (uchar4 *)dst);
}

int hvr_device_alloc(hvr_ctx *c, uint64_t bytes, void **ptr)
{
    if (!c || !ptr) return fail(HVR_EINVAL, "null argument");
    *ptr = nullptr;
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(dev_malloc(c->device, ptr, bytes ? bytes : 1));
    return HVR_OK;
}

int hvr_device_free(hvr_ctx *c, void *ptr)
{
    if (!c) return fail(HVR_EINVAL, "ctx is null");
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(hipStreamSynchronize(c->stream));
    HIPCHK(hipFree(ptr));
    return HVR_OK;
}

int hvr_copy_to_host(hvr_ctx *c, void *host, const void *dev, uint64_t bytes)
{
    if (!c || !host || !dev) return fail(HVR_EINVAL, "null argument");
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return HVR_OK;
}

int hvr_device_copy(hvr_ctx *c, void *dst, const void *src, uint64_t bytes)
{
    if (!c || !dst || !src) return fail(HVR_EINVAL, "null argument");
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return HVR_OK;
}

int hvr_timing_begin(hvr_ctx *c, int max_frames)
{
    if (!c) return fail(HVR_EINVAL, "ctx is null");
    if (max_frames <= 0 || max_frames > (1 << 16)) return fail(HVR_EINVAL, "max_frames out of range");
    HIPCHK(hipSetDevice(c->device));
    if (!c->tev) {
        c->tev = new std::vector<hipEvent_t>();
        c->tev_ordered = new std::vector<char>();
    }
    c->tev_ordered->assign((size_t)max_frames, 0);
    while (c->tev->size() < 3 * (size_t)max_frames) {
        hipEvent_t e;
        HIPCHK(hipEventCreate(&e));
        c->tev->push_back(e);
    }
    c->timing_max = max_frames;
    c->timing_n = 0;
    return HVR_OK;
}

int hvr_timing_end(hvr_ctx *c, double *march_ms, double *setup_ms, int *frames)
{
    if (!c || !c->tev) return fail(HVR_ESTATE, "no timing region");
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(hipStreamSynchronize(c->stream));
    double m = 0.0, s = 0.0;
    for (int i = 0; i < c->timing_n; ++i) {
        float a = 0.f, b = 0.f;
        if ((*c->tev_ordered)[i]) HIPCHK(hipEventElapsedTime(&a, (*c->tev)[3 * i], (*c->tev)[3 * i + 1]));
        HIPCHK(hipEventElapsedTime(&b, (*c->tev)[3 * i + 1], (*c->tev)[3 * i + 2]));
        s += a;
        m += b;
    }
    if (march_ms) *march_ms = m;
    if (setup_ms) *setup_ms = s;
    if (frames) *frames = c->timing_n;
    c->timing_max = 0;
    c->timing_n = 0;
    return HVR_OK;
}

// The copy runs through the pinned buffer in chunks of at least 1 MiB (at
// most four): each chunk's host copy into `out` starts as soon as its
// device-to-host copy has landed, overlapping the transfer of the next.
// Images up to 1 MiB take one copy, since the per-chunk synchronisation
// costs more than the overlap saves there.

int hvr_read(hvr_ctx *c, uint8_t *out)
{
    HVR_FAULT_POINT("hvr_read");
    if (!c || !out) return fail(HVR_EINVAL, "null argument");
    HIPCHK(hipSetDevice(c->device));
    const size_t bytes = (size_t)c->W * c->H * 4;
    if (c->last_host) {
        // the march wrote the frame to the pinned buffer: wait, copy once
        HIPCHK(hipStreamSynchronize(c->stream));
        hvr::CopyPool::get().copy(out, (const uint8_t *)c->h_pinned, bytes);
        return HVR_OK;
    }
    constexpr int KMAX = 4;
    const int K = (int)std::min<size_t>(KMAX, std::max<size_t>(1, bytes >> 20));
    const size_t chunk = ((bytes + K - 1) / K + 4095) & ~(size_t)4095;
    size_t off[KMAX + 1];
    for (int k = 0; k <= K; ++k) off[k] = std::min(bytes, (size_t)k * chunk);
    uint8_t *h = (uint8_t *)c->h_pinned;
    const uint8_t *d = (const uint8_t *)c->d_out;
    for (int k = 0; k < K; ++k) {
        if (off[k + 1] > off[k])
            HIPCHK(hipMemcpyAsync(h + off[k], d + off[k], off[k + 1] - off[k], hipMemcpyDeviceToHost, c->stream));
        HIPCHK(hipEventRecord(c->rev[k], c->stream));
    }
    for (int k = 0; k < K; ++k) {
        HIPCHK(hipEventSynchronize(c->rev[k]));
        memcpy(out + off[k], h + off[k], off[k + 1] - off[k]);
    }
    return HVR_OK;
}

int hvr_read_pinned(hvr_ctx *c, const uint8_t **rgba)
{
    if (!c || !rgba) return fail(HVR_EINVAL, "null argument");
    *rgba = nullptr;
    HIPCHK(hipSetDevice(c->device));
    const size_t bytes = (size_t)c->W * c->H * 4;
    if (!c->last_host) HIPCHK(hipMemcpyAsync(c->h_pinned, c->d_out, bytes, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    *rgba = (const uint8_t *)c->h_pinned;
    return HVR_OK;
}

int hvr_render(hvr_ctx *c, uint8_t *out)
{
    int rc = hvr_render_async(c);
    if (rc != HVR_OK) return rc;
    return hvr_read(c, out);
}

int hvr_synchronize(hvr_ctx *c)
{
    if (!c) return fail(HVR_EINVAL, "ctx is null");
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(hipStreamSynchronize(c->stream));
    return HVR_OK;
}

int hvr_framebuffer(hvr_ctx *c, void **ptr)
{
    if (!c || !ptr) return fail(HVR_EINVAL, "null argument");
    *ptr = c->d_out;
    return HVR_OK;
}

static int sample_counts(hvr_ctx *c, uint32_t *counts, bool shaded)
{
    if (!c || !counts) return fail(HVR_EINVAL, "null argument");
    HIPCHK(hipSetDevice(c->device));
    const size_t npix = (size_t)c->W * c->H;
    if (c->counts_cap < npix) {
        (void)hipFree(c->d_counts);
        c->d_counts = nullptr;
        c->counts_cap = 0;
        HIPCHK(dev_malloc(c->device, (void **)&c->d_counts, npix * sizeof(uint32_t)));
        c->counts_cap = npix;
    }
    int rc = enqueue_frame(c, true, nullptr, shaded);
    if (rc != HVR_OK) return rc;
    HIPCHK(hipMemcpyAsync(counts, c->d_counts, npix * sizeof(uint32_t), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return HVR_OK;
}

int hvr_sample_counts(hvr_ctx *c, uint32_t *counts)
{
    HVR_FAULT_POINT("hvr_sample_counts");
    return sample_counts(c, counts, false);
}

int hvr_shaded_sample_counts(hvr_ctx *c, uint32_t *counts)
{
    return sample_counts(c, counts, true);
}

int hvr_touched_bricks(hvr_ctx *c, unsigned long long *touched, unsigned long long *bricks,
                       unsigned long long *brick_bytes)
{
    if (!c || !touched) return fail(HVR_EINVAL, "null argument");
    const hvr_volume *S = c->scalar_vol;
    if (!S || !(S->lb == 3 || S->lb == 4) || c->lut_n > kLutLdsMax)
        return fail(HVR_ESTATE, "hvr_touched_bricks: needs a bound scalar volume with 8^3 or 16^3 bricks and a LUT "
                                "of at most 2048 entries");
    HIPCHK(hipSetDevice(c->device));
    const size_t npix = (size_t)c->W * c->H;
    if (c->counts_cap < npix) {
        (void)hipFree(c->d_counts);
        c->d_counts = nullptr;
        c->counts_cap = 0;
        HIPCHK(dev_malloc(c->device, (void **)&c->d_counts, npix * sizeof(uint32_t)));
        c->counts_cap = npix;
    }
    const uint64_t nb = (uint64_t)S->nbx * S->nby * S->nbz;
    uint8_t *d_marks = nullptr;
    HIPCHK(dev_malloc(c->device, (void **)&d_marks, nb));
    std::vector<uint8_t> marks(nb);
    int rc = hipMemsetAsync(d_marks, 0, nb, c->stream) == hipSuccess ? HVR_OK : fail(HVR_EDEVICE, "memset");
    if (rc == HVR_OK) rc = enqueue_frame(c, true, nullptr, false, d_marks);
    if (rc == HVR_OK && (hipMemcpyAsync(marks.data(), d_marks, nb, hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
                         hipStreamSynchronize(c->stream) != hipSuccess))
        rc = fail(HVR_EDEVICE, "hvr_touched_bricks: reading the marks failed");
    (void)hipStreamSynchronize(c->stream);   // nothing queued may still write the marks
    (void)hipFree(d_marks);
    if (rc != HVR_OK) return rc;
    unsigned long long n = 0;
    for (uint8_t m : marks) n += m != 0;
    *touched = n;
    if (bricks) *bricks = nb;
    if (brick_bytes) *brick_bytes = S->brick_bytes;
    return HVR_OK;
}

int hvr_last_kernel_ms(hvr_ctx *c, float *march_ms, float *setup_ms)
{
    if (!c) return fail(HVR_EINVAL, "ctx is null");
    if (!c->events_recorded) return fail(HVR_ESTATE, "no frame rendered yet");
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(hipEventSynchronize(c->last_ev[2]));
    float a = 0.f, b = 0.f;
    if (c->last_ev[0] != c->last_ev[1]) HIPCHK(hipEventElapsedTime(&a, c->last_ev[0], c->last_ev[1]));
    HIPCHK(hipEventElapsedTime(&b, c->last_ev[1], c->last_ev[2]));
    if (setup_ms) *setup_ms = a;
    if (march_ms) *march_ms = b;
    return HVR_OK;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Batches: requests staged on the host, rendered by one persistent launch
// per kernel class, captured once in a hipGraph per batch shape (classes,
// LUT capacity, staging block) and replayed with new staged contents.

struct BatchReq {
    hvr_volume *vol;
    int nm;                  // NM_ZERO / NM_ALIAS / NM_SAME
    hvr_params params;
    int W, H;
    std::vector<float> lut;  // n x RGBA
    uint64_t lut_hash;       // float_hash
};

// A captured launch and the shape it was captured for.  The shape holds each
// class's kernel, which its number of rays chooses (batch_lanes), so batches of
// changing sizes come back to a few shapes: each keeps its graph, up to
// kBatchGraphs of them (capturing and instantiating one takes 9 us of a 31 us
// launch, and milliseconds the first time a kernel is used).
struct BatchGraph {
    std::string key;
    hipGraph_t graph;
    hipGraphExec_t exec;
};
constexpr size_t kBatchGraphs = 8;

struct hvr_batch {
    hvr_ctx *ctx;
    hipStream_t stream;
    std::vector<BatchReq> reqs;
    int tile_shape;                       // HVR_TILE_8X8 / HVR_TILE_16X4
    int variant;                          // kernel variant of non-counting runs (BV_*)
    char *h_stage, *d_stage;              // staged block (pinned host, device)
    size_t stage_cap;
    uchar4 *d_out;                        // output pool, one RGBA8 image per request
    uint8_t *h_out;                       // its pinned host copy
    uchar4 *h_out_dev;                    // h_out's device address (HVR_READBACK_DIRECT)
    const uint8_t *h_out_dev_of;          // the h_out that h_out_dev maps
    size_t out_cap;
    int readback;                         // HVR_READBACK_DIRECT (default) / HVR_READBACK_COPY
    uint32_t *d_counts, *h_counts;        // sample-count pool (counting runs)
    size_t counts_cap;                    // in pixels
    uint8_t *d_flags;                     // transparent-brick flags, per request
    size_t flags_cap;
    uint32_t *d_counters;                 // tile counter per class
    std::vector<size_t> out_off;          // per request (add order): pixel offset in the pools
    std::vector<BatchGraph> graphs;       // captured launches, most recently used first
    hipEvent_t ev0, ev1, ev2;             // graph start / end, copies back done
    bool ran, counted;
    size_t out_pixels;
    int ncu;
};

// The serving layer's memory budget bounds a staged request by 512 bytes of
// descriptor (pyvr_amd/hip_renderer/serve.py, batch_pool_bytes).
static_assert(sizeof(ReqDesc) <= 512, "request descriptor above the serving budget's bound");

// The batched launcher for a class: format, normal mode, brick log2, counting,
// ray tile, buffer loads and kernel variant (BV_*); nullptr when the library
// has no such instance.  buf: the volume is read through buffer loads
// (below 4 GiB and 2^24 bricks).
static BatchLaunchFn batch_fn(int fmt, int nm, int lb, bool count, int ts, bool buf, int variant = BV_DEFAULT)
{
    switch (fmt) {
#define HVR_CASE(F) \
    case F: return batch_fn_##F(nm, lb, count, ts, buf, variant);
        HVR_FAST_FORMATS(HVR_CASE)
#undef HVR_CASE
    default: return nullptr;
    }
}

// Grow a device (and optionally pinned host) buffer to at least `need` bytes.
// After a failure its capacity is 0.
static int grow(int device, void **d, void **h, size_t *cap, size_t need)
{
    if (need <= *cap) return HVR_OK;
    size_t n = *cap ? *cap : 4096;
    while (n < need) n *= 2;
    (void)hipFree(*d);
    *d = nullptr;
    if (h) {
        (void)hipHostFree(*h);
        *h = nullptr;
    }
    *cap = 0;
    HVR_FAULT_POINT("hvr_batch_grow");
    HIPCHK(dev_malloc(device, d, n));
    if (h) HIPCHK(hipHostMalloc(h, n, hipHostMallocDefault));
    *cap = n;
    return HVR_OK;
}

// Drop the graphs from the n-th most recently used on (no launch in flight).
static void batch_drop_graphs(hvr_batch *b, size_t n = 0)
{
    for (size_t k = n; k < b->graphs.size(); ++k) {
        (void)hipGraphExecDestroy(b->graphs[k].exec);
        (void)hipGraphDestroy(b->graphs[k].graph);
    }
    if (n < b->graphs.size()) b->graphs.resize(n);
}

// The batch's pools of at least these bytes (no launch in flight).  What holds
// their addresses goes before any of them moves, since a later one may fail.
static int batch_grow(hvr_batch *b, size_t stage, size_t out, size_t flags)
{
    const int device = b->ctx->device;
    if (stage > b->stage_cap) batch_drop_graphs(b);
    if (out > b->out_cap) b->h_out_dev_of = nullptr;   // a new pinned pool may reuse the old address
    if (const int rc = grow(device, (void **)&b->d_stage, (void **)&b->h_stage, &b->stage_cap, stage)) return rc;
    if (const int rc = grow(device, (void **)&b->d_out, (void **)&b->h_out, &b->out_cap, out)) return rc;
    return grow(device, (void **)&b->d_flags, nullptr, &b->flags_cap, flags);
}

extern "C" {

int hvr_batch_create(hvr_ctx *c, hvr_batch **out)
{
    HVR_FAULT_POINT("hvr_batch_create");
    if (!c || !out) return fail(HVR_EINVAL, "null argument");
    *out = nullptr;
    HIPCHK(hipSetDevice(c->device));
    hvr_batch *b = new hvr_batch();
    b->ctx = c;
    b->tile_shape = HVR_TILE_8X8;
    b->variant = BV_DEFAULT;
    b->readback = HVR_READBACK_DIRECT;
    hipError_t e = hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreate(&b->ev0);
    if (e == hipSuccess) e = hipEventCreate(&b->ev1);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&b->ev2, hipEventDisableTiming);
    if (e == hipSuccess) e = hipMalloc(&b->d_counters, kBatchMaxClasses * sizeof(uint32_t));
    if (e == hipSuccess) e = hipDeviceGetAttribute(&b->ncu, hipDeviceAttributeMultiprocessorCount, c->device);
    if (e != hipSuccess) {
        hvr_batch_destroy(b);
        return fail_hip(e, "hvr_batch_create");
    }
    *out = b;
    return HVR_OK;
}

int hvr_batch_destroy(hvr_batch *b)
{
    if (!b) return HVR_OK;
    (void)hipSetDevice(b->ctx->device);
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    batch_drop_graphs(b);
    (void)hipFree(b->d_stage);
    (void)hipFree(b->d_out);
    (void)hipFree(b->d_counts);
    (void)hipFree(b->d_flags);
    (void)hipFree(b->d_counters);
    if (b->h_stage) (void)hipHostFree(b->h_stage);
    if (b->h_out) (void)hipHostFree(b->h_out);
    if (b->h_counts) (void)hipHostFree(b->h_counts);
    if (b->ev0) (void)hipEventDestroy(b->ev0);
    if (b->ev1) (void)hipEventDestroy(b->ev1);
    if (b->ev2) (void)hipEventDestroy(b->ev2);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    delete b;
    return HVR_OK;
}

int hvr_batch_clear(hvr_batch *b)
{
    if (!b) return fail(HVR_EINVAL, "batch is null");
    b->reqs.clear();
    b->ran = b->counted = false;
    return HVR_OK;
}

int hvr_batch_set_tile_shape(hvr_batch *b, int shape)
{
    if (!b) return fail(HVR_EINVAL, "batch is null");
    if (shape != HVR_TILE_8X8 && shape != HVR_TILE_16X4) return fail(HVR_EINVAL, "unknown tile shape");
    b->tile_shape = shape;
    return HVR_OK;
}

int hvr_batch_set_readback(hvr_batch *b, int mode)
{
    if (!b) return fail(HVR_EINVAL, "batch is null");
    if (mode != HVR_READBACK_COPY && mode != HVR_READBACK_DIRECT)
        return fail(HVR_EINVAL, "readback mode must be HVR_READBACK_COPY or HVR_READBACK_DIRECT");
    // the next run's descriptors point the march at the chosen pool; a run
    // in flight keeps the one it was enqueued with, and its images end in
    // the pinned pool either way
    b->readback = mode;
    return HVR_OK;
}

int hvr_batch_set_kernel(hvr_batch *b, int waves_per_block, int skip, int gate)
{
    if (!b) return fail(HVR_EINVAL, "batch is null");
    int v = -1;
    if (waves_per_block == 4 && skip && gate) v = BV_DEFAULT;
    else if (waves_per_block == 2 && skip && gate) v = BV_WAVES2;
    else if (waves_per_block == 8 && skip && gate) v = BV_WAVES8;
    else if (waves_per_block == 4 && skip && !gate) v = BV_NOGATE;
    else if (waves_per_block == 4 && !skip && gate) v = BV_NOSKIP;
    if (v < 0)
        return fail(HVR_EINVAL, "kernel variants: 4 waves with skipping and gating, or one of 2 / 8 waves, "
                                "no gating, no skipping");
    b->variant = v;
    return HVR_OK;
}

int hvr_batch_add(hvr_batch *b, hvr_volume *s, int srole, hvr_volume *n, int nrole, const float *lut_rgba,
                  int lut_n, const hvr_params *p, int width, int height, int *index)
{
    HVR_FAULT_POINT("hvr_batch_add");
    if (!b || !p) return fail(HVR_EINVAL, "null argument");
    if (!s || s->ctx != b->ctx || (n && n->ctx != b->ctx))
        return fail(HVR_EINVAL, "a batch request needs a scalar volume of the batch's context");
    if (srole != HVR_ROLE_SCALAR || !fmt_has_scalar(s->fmt) || !s->scalar_loaded)
        return fail(HVR_EINVAL, "the scalar sampler must read an uploaded scalar field");
    int nm;
    if (!n) nm = NM_ZERO;
    else if (n == s && nrole == HVR_ROLE_SCALAR) nm = NM_ALIAS;
    else if (n == s && nrole == HVR_ROLE_NORMAL && fmt_has_normal(s->fmt)) nm = NM_SAME;
    else return fail(HVR_EINVAL, "a batch request reads its normals from its scalar volume, or none");
    if (!batch_fn(s->fmt, nm, s->lb, false, HVR_TILE_8X8, true))
        return fail(HVR_EINVAL, "this volume layout and normal binding need the single-request path");
    if (lut_n < 0 || lut_n > kLutLdsMax || (lut_n > 0 && !lut_rgba))
        return fail(HVR_EINVAL, "batched LUTs hold 0 to 2048 entries");
    if (width <= 0 || height <= 0 || (long long)width * height > (1ll << 28))
        return fail(HVR_EINVAL, "width and height must be positive (at most 2^28 pixels)");
    if (const int rc = check_params(p)) return rc;
    BatchReq r;
    r.vol = s;
    r.nm = nm;
    r.params = *p;
    r.W = width;
    r.H = height;
    if (lut_n > 0) r.lut.assign(lut_rgba, lut_rgba + 4 * (size_t)lut_n);
    else r.lut = {0.f, 0.f, 0.f, 1.f};  // unbound LUT texture
    r.lut_hash = float_hash(r.lut.data(), r.lut.size());
    b->reqs.push_back(std::move(r));
    b->ran = b->counted = false;
    if (index) *index = (int)b->reqs.size() - 1;
    return HVR_OK;
}

int hvr_batch_reserve(hvr_batch *b, int max_requests, unsigned long long max_pixels, unsigned long long max_bricks)
{
    if (!b || max_requests < 0) return fail(HVR_EINVAL, "bad argument");
    HIPCHK(hipSetDevice(b->ctx->device));
    // growing frees buffers the previous run may still read
    HIPCHK(hipStreamSynchronize(b->stream));
    const size_t nreq = (size_t)max_requests;
    // the largest staged block: header, descriptors, LUTs of 2048 entries
    // and their prefix counts (the layout of hvr_batch_run_async)
    const size_t desc_off = align_up(sizeof(BatchHeader), 256);
    const size_t lut_off = align_up(desc_off + nreq * sizeof(ReqDesc), 256);
    const size_t nz_off = align_up(lut_off + nreq * kLutLdsMax * sizeof(float4), 256);
    const size_t stage = align_up(nz_off + nreq * (kLutLdsMax + 1) * sizeof(int), 256);
    const size_t pixels = (size_t)max_pixels + 64 * nreq;   // each request padded to 64 pixels
    const size_t flags = nreq * align_up((size_t)max_bricks, 256);
    return batch_grow(b, stage, pixels * 4, flags);
}

int hvr_batch_run_async(hvr_batch *b, int count)
{
    HVR_FAULT_POINT("hvr_batch_run_async");
    if (!b) return fail(HVR_EINVAL, "batch is null");
    hvr_ctx *c = b->ctx;
    HIPCHK(hipSetDevice(c->device));
    // the previous run's copies read and write the pinned buffers
    HIPCHK(hipStreamSynchronize(b->stream));
    const int nreq = (int)b->reqs.size();
    b->ran = b->counted = false;
    if (nreq == 0) return HVR_OK;
    // classes: one kernel instance each, in order of first appearance
    struct Cls {
        int fmt, nm, lb;
        bool buf;
        std::vector<int> members;
        int variant, bx, by;   // kernel variant and the pixels of its block tile
    };
    std::vector<Cls> cls;
    int lut_cap = 1;
    for (int i = 0; i < nreq; ++i) {
        const BatchReq &r = b->reqs[i];
        const bool buf = volume_buf(r.vol) && !c->force_global;
        int k = 0;
        while (k < (int)cls.size() && !(cls[k].fmt == r.vol->fmt && cls[k].nm == r.nm && cls[k].lb == r.vol->lb &&
                                        cls[k].buf == buf))
            ++k;
        if (k == (int)cls.size()) {
            if (k == kBatchMaxClasses) return fail(HVR_EINVAL, "a batch mixes more than 8 volume layouts");
            cls.push_back({r.vol->fmt, r.nm, r.vol->lb, buf, {}, 0, 0, 0});
        }
        cls[k].members.push_back(i);
        lut_cap = std::max(lut_cap, (int)(r.lut.size() / 4));
    }
    // LDS capacity in steps of 256 entries, so that graphs are reused
    lut_cap = (int)align_up((size_t)lut_cap, 256);
    // costliest requests first inside each class (tail balance)
    for (Cls &k : cls)
        std::stable_sort(k.members.begin(), k.members.end(), [&](int a, int z) {
            return (long long)b->reqs[a].W * b->reqs[a].H > (long long)b->reqs[z].W * b->reqs[z].H;
        });
    // sizes
    // the block tile of k_batch: 2 waves across, W / 2 down (counting runs
    // use the default variant)
    for (Cls &k : cls) {
        k.variant = count ? (int)BV_DEFAULT : b->variant;
        k.bx = b->tile_shape == HVR_TILE_16X4 ? 32 : 16;
        k.by = (b->tile_shape == HVR_TILE_16X4 ? 4 : 8) * (batch_variant_waves(k.variant) / 2);
        // few rays: several lanes each
        double rays = 0.0, samples = 0.0;
        for (int i : k.members) {
            const BatchReq &r = b->reqs[i];
            const double n = (double)r.W * r.H;
            rays += n;
            samples += n * ray_steps(r.params.bmin, r.params.bmax, r.params.step, r.params.max_steps);
        }
        const int lanes = batch_lanes((long long)rays, 2048ll * b->ncu, samples / rays);
        if (lanes > 1 && !count && k.buf && k.variant == BV_DEFAULT && b->tile_shape == HVR_TILE_8X8) {
            const MarchTile bt = march_tile(lanes);
            k.variant = lanes == 4 ? BV_LANES4 : BV_LANES2;
            k.bx = 1 << bt.lbw;
            k.by = 1 << bt.lbh;
        }
    }
    size_t desc_off = align_up(sizeof(BatchHeader), 256);
    size_t lut_off = align_up(desc_off + (size_t)nreq * sizeof(ReqDesc), 256);
    size_t lut_bytes = 0, nz_bytes = 0, pixels = 0, flag_bytes = 0;
    b->out_off.assign(nreq, 0);
    for (int i = 0; i < nreq; ++i) {
        const BatchReq &r = b->reqs[i];
        lut_bytes += r.lut.size() * sizeof(float);
        nz_bytes += (r.lut.size() / 4 + 1) * sizeof(int);
        b->out_off[i] = pixels;
        pixels += align_up((size_t)r.W * r.H, 64);
        flag_bytes += align_up((size_t)r.vol->nbx * r.vol->nby * r.vol->nbz, 256);
    }
    const size_t nz_off = align_up(lut_off + lut_bytes, 256);
    const size_t stage_need = align_up(nz_off + nz_bytes, 256);
    if (const int rc = batch_grow(b, stage_need, pixels * 4, flag_bytes)) return rc;
    if (count) {
        size_t cb = b->counts_cap * 4;
        const int rc = grow(b->ctx->device, (void **)&b->d_counts, (void **)&b->h_counts, &cb, pixels * 4);
        b->counts_cap = cb / 4;
        if (rc) return rc;
    }
    // direct: the march stores each pixel straight into the pinned pool
    // through its device address (posted writes over the host link while
    // the batch runs, no copy after it)
    const bool direct = b->readback == HVR_READBACK_DIRECT;
    if (direct && b->h_out_dev_of != b->h_out) {
        HIPCHK(hipHostGetDevicePointer((void **)&b->h_out_dev, b->h_out, 0));
        b->h_out_dev_of = b->h_out;
    }
    uchar4 *const out_pool = direct ? b->h_out_dev : b->d_out;
    // stage: header, descriptors (class by class), LUTs, prefix counts
    memset(b->h_stage, 0, desc_off);
    BatchHeader *hdr = (BatchHeader *)b->h_stage;
    hdr->nclass = (int)cls.size();
    hdr->nreq = nreq;
    hdr->all_offset = (uint32_t)desc_off;
    ReqDesc *descs = (ReqDesc *)(b->h_stage + desc_off);
    size_t lut_at = lut_off, nz_at = nz_off, flag_at = 0;
    int slot = 0;
    uint32_t flag_tiles = 0;
    // views of one volume through one LUT share its staged copy and flags
    ShareTable firsts((size_t)nreq);
    std::vector<int> request((size_t)nreq);   // of each descriptor
    for (size_t k = 0; k < cls.size(); ++k) {
        hdr->cls[k].desc_offset = (uint32_t)(desc_off + (size_t)slot * sizeof(ReqDesc));
        hdr->cls[k].nreq = (int)cls[k].members.size();
        int tiles = 0;
        for (int i : cls[k].members) {
            const BatchReq &r = b->reqs[i];
            ReqDesc &d = descs[slot++];
            memset(&d, 0, sizeof(d));
            d.fc = frame_const_of(r.params, true, r.W, r.H);
            d.ts = tex_desc(r.vol, HVR_ROLE_SCALAR, d.fc);
            const int n = (int)(r.lut.size() / 4);
            request[slot - 1] = i;
            const int first = firsts.find_or_add(
                r.lut_hash ^ (uint64_t)(uintptr_t)r.vol * 0x9e3779b97f4a7c15ull, slot - 1, [&](int other) {
                    const BatchReq &o = b->reqs[request[other]];
                    return o.vol == r.vol && o.lut.size() == r.lut.size() &&
                           memcmp(o.lut.data(), r.lut.data(), r.lut.size() * sizeof(float)) == 0;
                });
            d.lut_n = n;
            d.range = r.vol->d_range;
            d.nbz = r.vol->nbz;
            if (first >= 0) {
                d.lut = descs[first].lut;
                d.nz = descs[first].nz;
                d.flags = descs[first].flags;
            } else {
                memcpy(b->h_stage + lut_at, r.lut.data(), r.lut.size() * sizeof(float));
                lut_prefix_counts(r.lut.data(), n, (int *)(b->h_stage + nz_at));
                d.lut = (const float4 *)(b->d_stage + lut_at);
                d.nz = (const int *)(b->d_stage + nz_at);
                lut_at += r.lut.size() * sizeof(float);
                nz_at += (size_t)(n + 1) * sizeof(int);
                d.flags = b->d_flags + flag_at;
                flag_at += align_up((size_t)r.vol->nbx * r.vol->nby * r.vol->nbz, 256);
                flag_tiles += clearance_tiles(r.vol->nbx, r.vol->nby, r.vol->nbz);
            }
            d.flag_end = flag_tiles;
            d.out = out_pool + b->out_off[i];
            d.counts = count ? b->d_counts + b->out_off[i] : nullptr;
            d.ntx = (r.W + cls[k].bx - 1) / cls[k].bx;
            tiles += d.ntx * ((r.H + cls[k].by - 1) / cls[k].by);
            d.tile_end = tiles;
        }
    }
    // the graph for this shape
    std::string key = std::to_string(b->stage_cap) + "/" + std::to_string(lut_cap) + "/" +
                      std::to_string(count) + "/" + std::to_string(b->tile_shape);
    for (const Cls &k : cls)
        key += "/" + std::to_string(k.fmt) + "." + std::to_string(k.nm) + "." + std::to_string(k.lb) + "." +
               std::to_string(k.buf) + "." + std::to_string(k.variant);
    const auto known = std::find_if(b->graphs.begin(), b->graphs.end(), [&](const BatchGraph &g) { return g.key == key; });
    if (known != b->graphs.end()) {
        std::rotate(b->graphs.begin(), known, known + 1);
    } else {
        HVR_FAULT_POINT("hvr_batch_capture");
        batch_drop_graphs(b, kBatchGraphs - 1);
        HIPCHK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
        int rc = HVR_OK;
        if (hipMemcpyAsync(b->d_stage, b->h_stage, b->stage_cap, hipMemcpyHostToDevice, b->stream) != hipSuccess)
            rc = HVR_EDEVICE;
        if (rc == HVR_OK) {
            // counters reset by a kernel (a graph replays kernels reliably)
            hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, b->stream, b->d_counters, kBatchMaxClasses, 0u);
            hipLaunchKernelGGL(k_batch_flags, dim3(512), dim3(kClearThreads), 0, b->stream, (const char *)b->d_stage);
            if (hipGetLastError() != hipSuccess) rc = HVR_EDEVICE;
        }
        for (size_t k = 0; k < cls.size() && rc == HVR_OK; ++k) {
            const BatchLaunchFn fn =
                batch_fn(cls[k].fmt, cls[k].nm, cls[k].lb, count != 0, b->tile_shape, cls[k].buf, cls[k].variant);
            rc = fn ? fn(b->d_stage, (int)k, b->d_counters + k, lut_cap, b->ncu, b->stream) : HVR_EINVAL;
        }
        BatchGraph g = {key, nullptr, nullptr};
        const hipError_t e = hipStreamEndCapture(b->stream, &g.graph);
        if (rc != HVR_OK || e != hipSuccess) {
            if (g.graph) (void)hipGraphDestroy(g.graph);
            return fail(HVR_EDEVICE, "capturing the batch graph failed");
        }
        if (const hipError_t ei = hipGraphInstantiate(&g.exec, g.graph, nullptr, nullptr, 0)) {
            (void)hipGraphDestroy(g.graph);
            return fail_hip(ei, "instantiating the batch graph");
        }
        b->graphs.insert(b->graphs.begin(), std::move(g));
    }
    HIPCHK(hipEventRecord(b->ev0, b->stream));
    HIPCHK(hipGraphLaunch(b->graphs.front().exec, b->stream));
    HIPCHK(hipEventRecord(b->ev1, b->stream));
    if (!direct) HIPCHK(hipMemcpyAsync(b->h_out, b->d_out, pixels * 4, hipMemcpyDeviceToHost, b->stream));
    if (count) HIPCHK(hipMemcpyAsync(b->h_counts, b->d_counts, pixels * 4, hipMemcpyDeviceToHost, b->stream));
    HIPCHK(hipEventRecord(b->ev2, b->stream));
    b->out_pixels = pixels;
    b->ran = true;
    b->counted = count != 0;
    return HVR_OK;
}

int hvr_batch_wait(hvr_batch *b)
{
    HVR_FAULT_POINT("hvr_batch_wait");
    if (!b) return fail(HVR_EINVAL, "batch is null");
    HIPCHK(hipSetDevice(b->ctx->device));
    HIPCHK(hipStreamSynchronize(b->stream));
    return HVR_OK;
}

int hvr_batch_query(hvr_batch *b, int *done)
{
    HVR_FAULT_POINT("hvr_batch_query");
    if (!b || !done) return fail(HVR_EINVAL, "null argument");
    if (!b->ran) {
        *done = 1;
        return HVR_OK;
    }
    HIPCHK(hipSetDevice(b->ctx->device));
    const hipError_t e = hipEventQuery(b->ev2);
    if (e == hipSuccess) *done = 1;
    else if (e == hipErrorNotReady) {
        *done = 0;
        (void)hipGetLastError();   // still in flight, not an error
    }
    else return fail_hip(e, "hvr_batch_query");
    return HVR_OK;
}

int hvr_batch_run(hvr_batch *b, int count)
{
    if (const int rc = hvr_batch_run_async(b, count)) return rc;
    return hvr_batch_wait(b);
}

int hvr_batch_output(hvr_batch *b, int index, const uint8_t **rgba)
{
    if (!b || !rgba) return fail(HVR_EINVAL, "null argument");
    if (!b->ran) return fail(HVR_ESTATE, "the batch has not been run since its last change");
    if (index < 0 || index >= (int)b->reqs.size()) return fail(HVR_EINVAL, "request index out of range");
    *rgba = b->h_out + 4 * b->out_off[index];
    return HVR_OK;
}

int hvr_batch_counts(hvr_batch *b, int index, const uint32_t **counts)
{
    if (!b || !counts) return fail(HVR_EINVAL, "null argument");
    if (!b->ran || !b->counted) return fail(HVR_ESTATE, "the batch has not been run with counting");
    if (index < 0 || index >= (int)b->reqs.size()) return fail(HVR_EINVAL, "request index out of range");
    *counts = b->h_counts + b->out_off[index];
    return HVR_OK;
}

int hvr_batch_last_ms(hvr_batch *b, float *ms)
{
    if (!b || !ms) return fail(HVR_EINVAL, "null argument");
    if (!b->ran) return fail(HVR_ESTATE, "the batch has not been run");
    HIPCHK(hipSetDevice(b->ctx->device));
    HIPCHK(hipEventSynchronize(b->ev1));
    HIPCHK(hipEventElapsedTime(ms, b->ev0, b->ev1));
    return HVR_OK;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// A frame rendered without allocating (hvr_render_async_to_noalloc): the
// one-request form of the batch launch, whose block (descriptor, tile
// counter) and per-brick transparency flags live in a static device array
// instead of buffers the library allocates.  The block is written on the
// device by k_stage_request from kernel arguments, so the frame is three
// kernels on the context's stream: stage, brick flags, persistent march.

static constexpr size_t kNoallocFlagsOffset = 4096;
static_assert(HVR_NOALLOC_SCRATCH_BYTES == kNoallocFlagsOffset + HVR_NOALLOC_MAX_BRICKS, "scratch layout");

// Layout of the scratch array: the batch header at offset 0 (the batch
// kernels read it at the block's start), the tile counter, the prefix counts
// of the unbound LUT, the request descriptor, then one flag byte per brick.
static constexpr StageOffsets kNoallocOffsets = {128u, 192u, 256u};
static_assert(sizeof(BatchHeader) <= 128, "header fits before the counter");
static_assert(256 + sizeof(ReqDesc) <= kNoallocFlagsOffset, "descriptor fits before the flags");

static __device__ __align__(256) unsigned char scratch[HVR_NOALLOC_SCRATCH_BYTES];

static std::mutex g_scratch_mu;
static void *g_scratch_ptr[kMaxDevices];         // device address of `scratch` per device
static hipError_t g_scratch_err[kMaxDevices];    // the lookup's result per device

// With `device` current: the address of this device's copy of `scratch`
// (each device holds its own), looked up once.  The array's name is a
// host-side handle, not a device address; only this pointer is passed to
// kernels.
static void noalloc_setup(int device)
{
    if (device < 0 || device >= kMaxDevices) return;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[device]) return;
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    g_scratch_err[device] = e;
    if (e == hipSuccess) g_scratch_ptr[device] = p;
}

static int noalloc_scratch(int device, char **out)
{
    *out = nullptr;
    if (device < 0 || device >= kMaxDevices) return fail(HVR_EINVAL, "device index out of range for scratch");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        const hipError_t e = g_scratch_err[device];
        g_err = std::string("no scratch address for this device (hipGetSymbolAddress: ") +
                (e == hipSuccess ? "not looked up" : hipGetErrorString(e)) + ")";
        return HVR_EDEVICE;
    }
    *out = (char *)g_scratch_ptr[device];
    return HVR_OK;
}

extern "C" {

int hvr_render_async_to_noalloc(hvr_ctx *c, void *dst)
{
    if (!c || !dst) return fail(HVR_EINVAL, "null argument");
    HIPCHK(hipSetDevice(c->device));
    const hvr_volume *S = c->scalar_vol, *N = c->normal_vol;
    if (!S || c->scalar_role != HVR_ROLE_SCALAR || !fmt_has_scalar(S->fmt) || !S->scalar_loaded)
        return fail(HVR_ESTATE, "hvr_render_async_to_noalloc: the scalar sampler must read an uploaded scalar field");
    int nm;
    if (!N) nm = NM_ZERO;
    else if (N == S && c->normal_role == HVR_ROLE_SCALAR) nm = NM_ALIAS;
    else if (N == S && c->normal_role == HVR_ROLE_NORMAL && fmt_has_normal(S->fmt)) nm = NM_SAME;
    else return fail(HVR_ESTATE, "hvr_render_async_to_noalloc: normals must come from the scalar volume, or none");
    const bool buf = volume_buf(S) && !c->force_global;
    const FrameConst fc = frame_const(c);
    const int lanes = buf ? batch_lanes((long long)c->W * c->H, resident_rays(c), ray_steps(fc)) : 1;
    const BatchLaunchFn fn = batch_fn(S->fmt, nm, S->lb, false, HVR_TILE_8X8, buf,
                                      lanes == 4 ? BV_LANES4 : lanes == 2 ? BV_LANES2 : BV_DEFAULT);
    if (!fn) return fail(HVR_EINVAL, "hvr_render_async_to_noalloc: brick edge must be 8 or 16 (log2 3 or 4)");
    if (c->lut_n > kLutLdsMax) return fail(HVR_EINVAL, "hvr_render_async_to_noalloc: LUT above 2048 entries");
    const uint64_t nb = (uint64_t)S->nbx * S->nby * S->nbz;
    if (nb > HVR_NOALLOC_MAX_BRICKS)
        return fail(HVR_EINVAL, "hvr_render_async_to_noalloc: volume has more bricks than the scratch array's "
                                "flags hold (HVR_NOALLOC_MAX_BRICKS)");
    char *blk = nullptr;
    if (const int rc = noalloc_scratch(c->device, &blk)) return rc;

    const StageOffsets off = kNoallocOffsets;
    BatchHeader hdr;
    memset(&hdr, 0, sizeof(hdr));
    hdr.nclass = 1;
    hdr.nreq = 1;
    hdr.all_offset = off.desc;
    hdr.cls[0].desc_offset = off.desc;
    hdr.cls[0].nreq = 1;
    const MarchTile bt = march_tile(lanes);   // the block tile of k_batch
    const int bx = 1 << bt.lbw, by = 1 << bt.lbh;
    ReqDesc d;
    memset(&d, 0, sizeof(d));
    d.fc = fc;
    d.ts = tex_desc(S, HVR_ROLE_SCALAR, fc);
    d.lut = c->d_lut;
    d.nz = c->d_nz ? (const int *)c->d_nz : (const int *)(blk + off.unbound_nz);
    d.range = S->d_range;
    d.flags = (uint8_t *)(blk + kNoallocFlagsOffset);
    d.out = (uchar4 *)dst;
    d.counts = nullptr;
    d.nbz = S->nbz;
    d.flag_end = clearance_tiles(S->nbx, S->nby, S->nbz);
    d.lut_n = c->lut_n;
    d.ntx = (c->W + bx - 1) / bx;
    d.tile_end = d.ntx * ((c->H + by - 1) / by);

    hipEvent_t e0 = c->ev[0], e1 = c->ev[1], e2 = c->ev[2];
    HIPCHK(hipEventRecord(e0, c->stream));
    hipLaunchKernelGGL(k_stage_request, dim3(1), dim3(64), 0, c->stream, blk, off, hdr, d);
    hipLaunchKernelGGL(k_batch_flags, dim3(512), dim3(kClearThreads), 0, c->stream, (const char *)blk);
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(e1, c->stream));
    if (const int rc = fn(blk, 0, (uint32_t *)(blk + off.counter), (int)align_up((size_t)c->lut_n, 256), c->ncu,
                          c->stream))
        return fail(rc, "hvr_render_async_to_noalloc: march launch failed");
    HIPCHK(hipEventRecord(e2, c->stream));
    c->last_ev[0] = e0;
    c->last_ev[1] = e1;
    c->last_ev[2] = e2;
    c->events_recorded = true;
    return HVR_OK;
}

int hvr_volume_download(hvr_volume *v, float *scalar, float *normals)
{
    if (!v || (!scalar && !normals)) return fail(HVR_EINVAL, "null argument");
    if (scalar && (!fmt_has_scalar(v->fmt) || !v->scalar_loaded))
        return fail(HVR_ESTATE, "the volume holds no uploaded scalar field");
    if (normals && (!fmt_has_normal(v->fmt) || !v->normals_loaded))
        return fail(HVR_ESTATE, "the volume holds no uploaded normal field");
    hvr_ctx *c = v->ctx;
    HIPCHK(hipSetDevice(c->device));
    const uint64_t plane = (uint64_t)v->s0 * v->s1;
    // whole z-planes per chunk, up to 256 MiB of floats (scalar + normals)
    const uint64_t per_voxel = (scalar ? 4 : 0) + (normals ? 12 : 0);
    uint64_t zper = ((uint64_t)256 << 20) / (plane * per_voxel);
    zper = std::max<uint64_t>(1, std::min<uint64_t>(zper, (uint64_t)v->s2));
    float *d_s = nullptr, *d_n = nullptr;
    int rc = HVR_OK;
    if (scalar && dev_malloc(c->device, (void **)&d_s, zper * plane * 4) != hipSuccess) rc = fail(HVR_ENOMEM, "download staging");
    if (rc == HVR_OK && normals && dev_malloc(c->device, (void **)&d_n, zper * plane * 12) != hipSuccess)
        rc = fail(HVR_ENOMEM, "download staging");
    for (uint64_t z0 = 0; rc == HVR_OK && z0 < (uint64_t)v->s2; z0 += zper) {
        const uint64_t nz = std::min<uint64_t>(zper, (uint64_t)v->s2 - z0);
        const uint64_t nvox = nz * plane;
        const unsigned nblk = (unsigned)((nvox + 255) / 256);
#define HVR_DL(F)                                                                                          \
    case F:                                                                                                \
        hipLaunchKernelGGL(k_download<F>, dim3(nblk), dim3(256), 0, c->stream, (const char *)v->d_texels,  \
                           v->s0, v->s1, v->lb, v->nbx, v->nby, v->brick_bytes, (int)z0, nvox, d_s, d_n); \
        break;
        switch (v->fmt) {
            HVR_DL(TF_S_F32)
            HVR_DL(TF_S_F16)
            HVR_DL(TF_S_U8)
            HVR_DL(TF_N_F32)
            HVR_DL(TF_N_SN8)
            HVR_DL(TF_C_F32_F32)
            HVR_DL(TF_C_F16_F32)
            HVR_DL(TF_C_U8_F32)
            HVR_DL(TF_C_F32_SN8)
            HVR_DL(TF_C_F16_SN8)
            HVR_DL(TF_C_U8_SN8)
            HVR_DL(TF_C_F16_F16)
            HVR_DL(TF_N_F16)
        default: rc = fail(HVR_EINVAL, "bad texel format");
        }
#undef HVR_DL
        if (rc != HVR_OK) break;
        if (hipGetLastError() != hipSuccess) rc = fail(HVR_EDEVICE, "download kernel launch failed");
        if (rc == HVR_OK && scalar &&
            hipMemcpyAsync(scalar + z0 * plane, d_s, nvox * 4, hipMemcpyDeviceToHost, c->stream) != hipSuccess)
            rc = fail(HVR_EDEVICE, "download copy failed");
        if (rc == HVR_OK && normals &&
            hipMemcpyAsync(normals + 3 * z0 * plane, d_n, nvox * 12, hipMemcpyDeviceToHost, c->stream) != hipSuccess)
            rc = fail(HVR_EDEVICE, "download copy failed");
        if (rc == HVR_OK && hipStreamSynchronize(c->stream) != hipSuccess) rc = fail(HVR_EDEVICE, "download wait");
    }
    (void)hipStreamSynchronize(c->stream);
    (void)hipFree(d_s);
    (void)hipFree(d_n);
    return rc;
}

}  // extern "C"
