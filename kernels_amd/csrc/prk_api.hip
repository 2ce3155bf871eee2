// C ABI of libprkstencil.so: the drop-in operator table, the fused sweep,
// initialisation, the device L1 norm, the driver loop and the HBM
// calibration kernels.  Declarations and reference citations: prk_stencil.h.
#include <execinfo.h>
#include <hip/hip_runtime.h>
#include <signal.h>
#include <unistd.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "pass.hpp"
#include "prk_internal.hpp"
#include "sweep.hpp"

namespace prk {

// ---------------------------------------------------------------------------
// Errors
// ---------------------------------------------------------------------------
static thread_local std::string g_last_error;

int set_error(int code, const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return code;
}

void clear_error() { g_last_error.clear(); }

int check_hip(hipError_t e, const char *what)
{
    if (e == hipSuccess) return PRK_OK;
    return set_error(PRK_EHIP, "%s: %s", what, hipGetErrorString(e));
}

// Process-wide overrides of the tuned tiling (tests and tuning probes).
static int g_rows_per_wave = 0;  // 0: tuned / default
static int g_variant_override = -1;
static int g_order = -1;
static int g_wgs_per_cu = -1;

static bool valid_dtype(int dt) { return dt == F64 || dt == F32 || dt == BF16; }

static int vec_width(int dt) { return dt == F64 ? 2 : dt == F32 ? 4 : 8; }

int plan_sweep(int pattern, int radius, int dtype, int n, long long pitch, const void *in,
               const void *in_next, const void *out, int rows_per_wave, SweepPlan *plan, int nrows)
{
    if (pattern != STAR && pattern != GRID)
        return set_error(PRK_EINVAL, "pattern must be 0 (star) or 1 (grid), got %d", pattern);
    if (radius < 1 || radius > kMaxRadius)
        return set_error(PRK_ENOSTENCIL, "no stencil for radius %d (supported 1..%d)", radius,
                         kMaxRadius);
    if (!valid_dtype(dtype)) return set_error(PRK_EINVAL, "unknown dtype %d", dtype);
    if (n < 1) return set_error(PRK_EINVAL, "grid dimension must be positive, got %d", n);
    if (2 * radius + 1 > n)
        return set_error(PRK_EINVAL, "stencil radius %d too large for n=%d", radius, n);
    if (pitch < n) return set_error(PRK_EINVAL, "pitch %lld < n %d", pitch, n);
    if (!in || !out) return set_error(PRK_EINVAL, "null grid pointer");
    if (in_next && (in_next == in || in_next == out))
        return set_error(PRK_EINVAL, "in_next must be a separate buffer");
    const size_t es = dtype_size(dtype);
    if ((unsigned long long)pitch * es >= (1ull << 31))
        return set_error(PRK_EINVAL, "row of %lld elements exceeds 2 GiB", pitch);
    const unsigned long long ptrs =
        (uintptr_t)in | (uintptr_t)out | (uintptr_t)in_next | (unsigned long long)pitch * es;  // the bits every row's address has
    plan->dtype = dtype;
    plan->pattern = pattern;
    plan->radius = radius;
    plan->n = n;
    plan->span = whole_grid(n);
    plan->pitch = pitch;
    plan->pad_writable = false;
    const bool short_rows = (unsigned long long)n * es < 16;  // MODE_DWORD reads up to 16 bytes of the next row
    plan->mode = ptrs % 16 == 0                 ? (n % vec_width(dtype) != 0 ? MODE_RAGGED : MODE_VEC)
                 : ptrs % 4 != 0 || short_rows ? MODE_ELEM
                                                : MODE_DWORD;
    const prk_tuning t = choose_tuning(pattern, radius, dtype, n, nrows > 0 ? nrows : n);
    plan->variant = g_variant_override >= 0 ? g_variant_override : t.variant;
    plan->order = g_order >= 0 ? g_order : t.order;
    plan->wgs_per_cu = g_wgs_per_cu >= 0 ? g_wgs_per_cu : t.wgs_per_cu;
    int rows = rows_per_wave > 0 ? rows_per_wave : (g_rows_per_wave > 0 ? g_rows_per_wave : t.rows_per_wave);
    plan->rows_per_wave = std::max(1, std::min(rows, n));
    return PRK_OK;
}

int launch_sweep(const SweepPlan &p, const void *in, void *in_next, void *out, hipStream_t s)
{
    switch (p.dtype) {
    case F64: return launch_sweep_f64(p, in, in_next, out, s);
    case F32: return launch_sweep_f32(p, in, in_next, out, s);
    case BF16: return launch_sweep_bf16(p, in, in_next, out, s);
    }
    return set_error(PRK_EINVAL, "unknown dtype %d", p.dtype);
}

int launch_pass(const SweepPlan &p, int sweeps, bool any, const void *in, void *in_next, void *out, hipStream_t s)
{
    switch (p.dtype) {
    case F64: return launch_pass_f64(p, sweeps, any, in, in_next, out, s);
    case F32: return launch_pass_f32(p, sweeps, any, in, in_next, out, s);
    case BF16: return launch_pass_bf16(p, sweeps, any, in, in_next, out, s);
    }
    return set_error(PRK_EINVAL, "unknown dtype %d", p.dtype);
}

// ---------------------------------------------------------------------------
// in += 1 over a pitched grid (elementwise; 16-byte vectors when aligned).
// ---------------------------------------------------------------------------
template <int DT, bool VEC>
__global__ __launch_bounds__(256) void add_one_kernel(void *buf, int n, long long pitch)
{
    typedef typename DTypeTraits<DT>::T T;
    constexpr int V = DTypeTraits<DT>::V;
    for (int row = blockIdx.y; row < n; row += gridDim.y) {
        T *p = (T *)buf + (long long)row * pitch;
        for (int c = (blockIdx.x * 256 + threadIdx.x) * V; c < n; c += gridDim.x * 256 * V) {
            if (VEC && c + V <= n) {
                union { u32x4 v; T e[V]; } x, y;
                x.v = *(const u32x4 *)(p + c);
                plus_one<DT, V>(x.e, y.e);
                *(u32x4 *)(p + c) = y.v;
            } else {
                for (int v = 0; v < V && c + v < n; ++v) {
                    T y;
                    plus_one<DT, 1>(&p[c + v], &y);
                    p[c + v] = y;
                }
            }
        }
    }
}

// The same where the rows follow one another without a gap: one 16-byte
// vector of the whole array per thread, whatever the rows' own alignment.
// Non-temporal where the array alone exceeds the last-level cache; below that
// a loop of stencil and refresh finds part of it there (FP64 star R=2, n =
// 3000: 63 us per turn, 70 non-temporal).  Measured on MI355X, rows -> flat:
// FP64 n = 16384 789 -> 658 us (6.5 TB/s), n = 8001 227 -> 157, n = 4001 57
// -> 45.
template <int DT, bool NT>
__global__ __launch_bounds__(256) void add_one_flat_kernel(void *buf, long long count)
{
    typedef typename DTypeTraits<DT>::T T;
    constexpr int V = DTypeTraits<DT>::V;
    T *p = (T *)buf;
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k < count / V) {
        union { u32x4 v; T e[V]; } x, y;
        x.v = NT ? __builtin_nontemporal_load((const u32x4 *)p + k) : ((const u32x4 *)p)[k];
        plus_one<DT, V>(x.e, y.e);
        if (NT) __builtin_nontemporal_store(y.v, (u32x4 *)p + k);
        else ((u32x4 *)p)[k] = y.v;
    } else if (k < count / V + count % V) {
        const long long c = count / V * V + (k - count / V);  // the elements behind the last vector
        T y;
        plus_one<DT, 1>(&p[c], &y);
        p[c] = y;
    }
}

// in += 1, `times` times over, a vector of a row at a time (VEC: rows on
// 16-byte boundaries; the vector over column n by element).  Bound by HBM, one
// read and one write of the array, while the additions take less than those:
// FP64 n = 30000 on MI355X 2.4 ms for 10 (6.1 TB/s), 2.7 for 100.
template <int DT, bool VEC>
__global__ __launch_bounds__(256) void add_times_kernel(void *buf, int n, long long pitch, int times)
{
    typedef typename DTypeTraits<DT>::T T;
    constexpr int V = VEC ? DTypeTraits<DT>::V : 1;
    for (int row = blockIdx.y; row < n; row += gridDim.y) {
        T *p = (T *)buf + (long long)row * pitch;
        for (int c = (blockIdx.x * 256 + threadIdx.x) * V; c < n; c += gridDim.x * 256 * V) {
            const bool whole = c + V <= n;
            union { u32x4 v; T e[V]; } x;
            if (VEC && whole) {
                x.v = __builtin_nontemporal_load((const u32x4 *)(p + c));
            } else {
#pragma unroll
                for (int v = 0; v < V; ++v) x.e[v] = p[c + v < n ? c + v : c];
            }
#pragma unroll 4
            for (int t = 0; t < times; ++t) {
                decltype(x) y;
                plus_one<DT, V>(x.e, y.e);
                x = y;
            }
            if (VEC && whole) {
                __builtin_nontemporal_store(x.v, (u32x4 *)(p + c));
            } else {
#pragma unroll
                for (int v = 0; v < V; ++v)
                    if (c + v < n) p[c + v] = x.e[v];
            }
        }
    }
}

static int launch_add_times(int dtype, int n, long long pitch, void *in, int times, hipStream_t s)
{
    const bool vec = ((uintptr_t)in | (unsigned long long)pitch * dtype_size(dtype)) % 16 == 0;
    const int span = 256 * (vec ? vec_width(dtype) : 1);
    const dim3 grid((unsigned)std::min(1024, (n + span - 1) / span), (unsigned)std::min(n, 65535));
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, in, n, pitch, times); };
    switch (dtype) {
    case F64: vec ? launch(add_times_kernel<F64, true>) : launch(add_times_kernel<F64, false>); break;
    case F32: vec ? launch(add_times_kernel<F32, true>) : launch(add_times_kernel<F32, false>); break;
    default: vec ? launch(add_times_kernel<BF16, true>) : launch(add_times_kernel<BF16, false>); break;
    }
    return check_hip(hipGetLastError(), "refresh launch");
}

static long long add_flat_threads(int dtype, long long count)
{
    return count / vec_width(dtype) + count % vec_width(dtype);
}

template <int DT>
static int launch_add_flat(long long count, void *in, hipStream_t s)
{
    const long long threads = add_flat_threads(DT, count);
    const dim3 blocks((unsigned)((threads + 255) / 256));
    const bool nt = count * (long long)sizeof(typename DTypeTraits<DT>::T) > kLastLevelCache;
    if (nt) hipLaunchKernelGGL((add_one_flat_kernel<DT, true>), blocks, dim3(256), 0, s, in, count);
    else hipLaunchKernelGGL((add_one_flat_kernel<DT, false>), blocks, dim3(256), 0, s, in, count);
    return check_hip(hipGetLastError(), "add launch");
}

static int launch_add(int dtype, int n, long long pitch, void *in, hipStream_t s)
{
    if (!valid_dtype(dtype)) return set_error(PRK_EINVAL, "unknown dtype %d", dtype);
    if (n < 1 || pitch < n || !in) return set_error(PRK_EINVAL, "bad grid (n=%d pitch=%lld)", n, pitch);
    const bool vec = ((uintptr_t)in % 16 == 0) && ((pitch * dtype_size(dtype)) % 16 == 0);
    const int V = vec_width(dtype);
    // A launch holds fewer than 2^32 threads: larger grids (FP64 from n =
    // 92682 on) go row by row, which has a bounded launch.
    const long long count = (long long)n * n;
    const bool launchable = add_flat_threads(dtype, count) <= (1ll << 32) - 256;
    // Aligned rows of an array that the L2s hold, but not beside the out of
    // the stencil before it, go row by row too: with that stencil (FP64 star
    // R=1) n = 2000 28.6 us, flat 29.6; n = 700 10.0, flat 9.0.
    const long long bytes = count * (long long)dtype_size(dtype);
    const bool l2_rows = vec && bytes > (6ll << 20) && bytes <= kL2s;
    if (pitch == n && (uintptr_t)in % 16 == 0 && launchable && !l2_rows) {
        return dtype == F64 ? launch_add_flat<F64>(count, in, s)
               : dtype == F32 ? launch_add_flat<F32>(count, in, s)
                              : launch_add_flat<BF16>(count, in, s);
    }
    const unsigned bx = std::min<unsigned>(8, (unsigned)((n + 256 * V - 1) / (256 * V)));
    dim3 grid(bx, std::min(n, 65535));
    switch (dtype) {
    case F64:
        if (vec) hipLaunchKernelGGL((add_one_kernel<F64, true>), grid, dim3(256), 0, s, in, n, pitch);
        else hipLaunchKernelGGL((add_one_kernel<F64, false>), grid, dim3(256), 0, s, in, n, pitch);
        break;
    case F32:
        if (vec) hipLaunchKernelGGL((add_one_kernel<F32, true>), grid, dim3(256), 0, s, in, n, pitch);
        else hipLaunchKernelGGL((add_one_kernel<F32, false>), grid, dim3(256), 0, s, in, n, pitch);
        break;
    default:
        if (vec) hipLaunchKernelGGL((add_one_kernel<BF16, true>), grid, dim3(256), 0, s, in, n, pitch);
        else hipLaunchKernelGGL((add_one_kernel<BF16, false>), grid, dim3(256), 0, s, in, n, pitch);
        break;
    }
    return check_hip(hipGetLastError(), "add launch");
}

// ---------------------------------------------------------------------------
// Initial values
// ---------------------------------------------------------------------------
// Initial values of the lane's V columns of one row in 16-byte stores (VEC:
// rows on 16-byte boundaries; the vector over column n by element), or of
// one column.  Bound by its stores in FP64 and by the generator's 64-bit
// multiplies in BF16.  Measured on MI355X, by element -> by vector: n = 16384
// FP64 717 -> 680 us, FP32 331 -> 308, BF16 324 -> 268; n = 9999 FP32 161 ->
// 155.
template <int DT, bool VEC>
__global__ __launch_bounds__(256) void init_kernel(int kind, uint64_t seed, int n, long long pitch,
                                                   void *in, void *out)
{
    typedef typename DTypeTraits<DT>::T T;
    constexpr int V = VEC ? DTypeTraits<DT>::V : 1;
    for (int row = blockIdx.y; row < n; row += gridDim.y) {
        T *pi = (T *)in + (long long)row * pitch;
        T *po = out ? (T *)out + (long long)row * pitch : nullptr;
        for (int c = (blockIdx.x * 256 + threadIdx.x) * V; c < n; c += gridDim.x * 256 * V) {
            const uint64_t state = seeded_state(seed, (uint64_t)row * (uint64_t)n + c);
            union { u32x4 v; T e[V]; } x;
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const double val = kind == PRK_INIT_ANALYTIC ? (double)(row + (c + v))
                                                             : seeded_of_state(state + v * kSeedStep);
                if constexpr (DT == BF16) x.e[v] = f32_to_bf16((float)val);
                else x.e[v] = (T)val;
            }
            if (VEC && c + V <= n) {
                *(u32x4 *)(pi + c) = x.v;
                if (po) *(u32x4 *)(po + c) = u32x4{0u, 0u, 0u, 0u};
            } else {
#pragma unroll
                for (int v = 0; v < V; ++v)
                    if (c + v < n) {
                        pi[c + v] = x.e[v];
                        if (po) po[c + v] = (T)0;
                    }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// L1 norm: compensated per-thread sums (Neumaier), double-double combination
// across the block and, in a second single-block pass, across blocks in a
// fixed order, so the result does not depend on scheduling.
// ---------------------------------------------------------------------------
struct DD {
    double hi, lo;
};

__device__ inline DD dd_add(DD a, DD b)
{
#pragma clang fp contract(off)
    const double s = a.hi + b.hi;
    const double bb = s - a.hi;
    const double e = (a.hi - (s - bb)) + (b.hi - bb);
    const double lo = e + a.lo + b.lo;
    const double hi = s + lo;
    return DD{hi, lo - (hi - s)};
}

constexpr int kNormThreads = 256;
static_assert(sizeof(DD) * kNormBlocks == kNormPartialsBytes, "norm partials layout");

// Rows in 16-byte vectors (VEC: rows on 16-byte boundaries; columns outside
// the interior count as 0), kNormAhead of them loaded at a time, or by
// element.  Bound by HBM where the vectors are; one element per load had a
// wave wait for 512 bytes at a time.  Measured on MI355X with the result's
// way back, by element -> by vector: n = 16384 FP64 637 -> 381 us, FP32 568
// -> 212, BF16 524 -> 180; n = 30000 FP64 2038 -> 1185 (6.07 TB/s).
constexpr int kNormAhead = 4;

template <int DT, bool VEC>
__global__ __launch_bounds__(kNormThreads) void norm_partial_kernel(const void *out, int n,
                                                                    long long pitch, int R, DD *partials)
{
#pragma clang fp contract(off)
    typedef typename DTypeTraits<DT>::T T;
    constexpr int V = VEC ? DTypeTraits<DT>::V : 1;
    constexpr int SPAN = kNormThreads * V;
    const T *o = (const T *)out;
    NormSum ns;
    union Vec { u32x4 v; T e[V]; };
    const int first = R / V * V;  // column of the row's first vector
    for (int i = R + blockIdx.x; i < n - R; i += gridDim.x) {
        const T *row = o + (long long)i * pitch;
        for (int c = first + (int)threadIdx.x * V; c < n - R; c += kNormAhead * SPAN) {
            Vec x[kNormAhead];
#pragma unroll
            for (int k = 0; k < kNormAhead; ++k) {
                const int ck = c + k * SPAN;
                if constexpr (VEC) x[k].v = *(const u32x4 *)(row + (ck < n - R ? ck : c));
                else x[k].e[0] = row[ck < n - R ? ck : c];
            }
#pragma unroll
            for (int k = 0; k < kNormAhead; ++k)
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    const int cv = c + k * SPAN + v;
                    double a;
                    if constexpr (DT == F64) a = x[k].e[v];
                    else a = (double)to_f32<T>(x[k].e[v]);
                    ns.add(cv >= R && cv < n - R ? a : 0.0);
                }
        }
    }
    __shared__ DD red[kNormThreads];
    red[threadIdx.x] = DD{ns.sum, ns.comp};
    __syncthreads();
    for (int s = kNormThreads / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] = dd_add(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0) partials[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(kNormThreads) void norm_final_kernel(const DD *partials, int nparts,
                                                                  double active, double *result)
{
#pragma clang fp contract(off)
    __shared__ DD red[kNormThreads];
    DD acc{0.0, 0.0};
    for (int k = threadIdx.x; k < nparts; k += kNormThreads) acc = dd_add(acc, partials[k]);
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = kNormThreads / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] = dd_add(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0) result[0] = (red[0].hi + red[0].lo) / active;
}

// Per-device workspace for the norm, allocated once: partials, and the result
// in pinned host memory, which the last kernel writes (a copy of 8 bytes back
// is a third of a small grid's norm: n = 1000 FP64 32 us with it, 24 without).
struct NormWorkspace {
    DD *partials = nullptr;
    double *result = nullptr, *d_result = nullptr;  // host and device address
};
static std::mutex g_ws_mutex;
static std::vector<NormWorkspace> g_ws;

static int norm_workspace(NormWorkspace **ws)
{
    int dev = 0;
    int rc = check_hip(hipGetDevice(&dev), "hipGetDevice");
    if (rc) return rc;
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    if ((int)g_ws.size() <= dev) g_ws.resize(dev + 1);
    NormWorkspace &w = g_ws[dev];
    if (!w.partials) {
        void *p = nullptr, *h = nullptr, *d = nullptr;
        rc = check_hip(hipMalloc(&p, sizeof(DD) * kNormBlocks), "norm workspace");
        if (!rc) rc = check_hip(hipHostMalloc(&h, 64, hipHostMallocDefault), "norm result");
        if (!rc) rc = check_hip(hipHostGetDevicePointer(&d, h, 0), "norm result");
        if (rc) {
            if (h) (void)hipHostFree(h);
            if (p) (void)hipFree(p);
            return rc;
        }
        w.partials = (DD *)p;
        w.result = (double *)h;
        w.d_result = (double *)d;
    }
    *ws = &w;
    return PRK_OK;
}

// Blocks of the norm's first pass (one partial each): one per interior row,
// at most kNormBlocks.
static int norm_blocks(int n, int radius)
{
    return (int)std::max<long long>(1, std::min<long long>(kNormBlocks, (long long)n - 2 * radius));
}

int enqueue_l1norm(int dtype, int n, long long pitch, int radius, const void *out, double *d_result,
                   DD *partials, hipStream_t s)
{
    const long long w = n - 2 * radius;
    const int blocks = norm_blocks(n, radius);
    const bool vec = ((uintptr_t)out | (unsigned long long)pitch * dtype_size(dtype)) % 16 == 0;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kNormThreads), 0, s, out, n, pitch, radius, partials);
    };
    switch (dtype) {
    case F64: vec ? launch(norm_partial_kernel<F64, true>) : launch(norm_partial_kernel<F64, false>); break;
    case F32: vec ? launch(norm_partial_kernel<F32, true>) : launch(norm_partial_kernel<F32, false>); break;
    default: vec ? launch(norm_partial_kernel<BF16, true>) : launch(norm_partial_kernel<BF16, false>); break;
    }
    hipLaunchKernelGGL(norm_final_kernel, dim3(1), dim3(kNormThreads), 0, s, (const DD *)partials, blocks,
                       (double)(w * w), d_result);
    return check_hip(hipGetLastError(), "norm launch");
}

// ---------------------------------------------------------------------------
// HBM calibration
// ---------------------------------------------------------------------------
// One 16-byte vector per thread and one short-lived workgroup per 4 KiB, with
// non-temporal hints: the fastest streaming shape measured on MI355X.
__global__ __launch_bounds__(256) void triad_kernel(long long len, double scalar, double *A,
                                                    const double *B, const double *C)
{
    typedef double d2 __attribute__((ext_vector_type(2)));
    const long long nv = len / 2;
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k < nv) {
        d2 a = __builtin_nontemporal_load(&((d2 *)A)[k]);
        const d2 b = __builtin_nontemporal_load(&((const d2 *)B)[k]);
        const d2 c = __builtin_nontemporal_load(&((const d2 *)C)[k]);
        a += b + scalar * c;
        __builtin_nontemporal_store(a, &((d2 *)A)[k]);
    }
    if (k == 0 && (len & 1)) A[len - 1] += B[len - 1] + scalar * C[len - 1];
}

// The sweep's two read and two write streams, with no stencil between them
// (in through the cache as the sweep reads it, out and the stores
// non-temporal: the fastest of the hint combinations measured on MI355X).
__global__ __launch_bounds__(256) void stream_mix_kernel(long long len, const double *in, double *in_next,
                                                         double *out)
{
    typedef double d2 __attribute__((ext_vector_type(2)));
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k < len / 2) {
        const d2 x = ((const d2 *)in)[k];
        d2 o = __builtin_nontemporal_load(&((d2 *)out)[k]);
        o += x;
        __builtin_nontemporal_store(x + 1.0, &((d2 *)in_next)[k]);
        __builtin_nontemporal_store(o, &((d2 *)out)[k]);
    }
    if (k == 0 && (len & 1)) {
        in_next[len - 1] = in[len - 1] + 1.0;
        out[len - 1] += in[len - 1];
    }
}

__global__ __launch_bounds__(256) void copy_kernel(long long nvec, u32x4 *dst, const u32x4 *src)
{
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k < nvec) __builtin_nontemporal_store(__builtin_nontemporal_load(&src[k]), &dst[k]);
}

// Copy in a chosen shape: a workgroup's chunk is VPL rows of 256 vectors
// (lane t takes vector t of each row), all VPL loads issued before the
// stores; chunks are taken in turn by `gridDim.x` workgroups.
template <int VPL, bool NT>
__global__ __launch_bounds__(256) void copy_shape_kernel(long long nvec, u32x4 *dst, const u32x4 *src)
{
    const long long chunk = 256LL * VPL;
    for (long long base = (long long)blockIdx.x * chunk; base < nvec; base += (long long)gridDim.x * chunk) {
        u32x4 v[VPL];
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
            const long long k = base + j * 256 + threadIdx.x;
            if (k < nvec) v[j] = NT ? __builtin_nontemporal_load(&src[k]) : src[k];
        }
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
            const long long k = base + j * 256 + threadIdx.x;
            if (k < nvec) {
                if (NT) __builtin_nontemporal_store(v[j], &dst[k]);
                else dst[k] = v[j];
            }
        }
    }
}

template <int VPL>
static void launch_copy_shape(int nt, unsigned blocks, long long nvec, u32x4 *dst, const u32x4 *src, hipStream_t s)
{
    if (nt) hipLaunchKernelGGL((copy_shape_kernel<VPL, true>), dim3(blocks), dim3(256), 0, s, nvec, dst, src);
    else hipLaunchKernelGGL((copy_shape_kernel<VPL, false>), dim3(blocks), dim3(256), 0, s, nvec, dst, src);
}

// ---------------------------------------------------------------------------
// The norm's partials in a static device array, for the allocation-free
// entry point.  In host code `scratch` names a host-side stand-in, not device
// memory: kernels get the device address looked up for the current device
// (each device holds its own copy of the array).
// ---------------------------------------------------------------------------
constexpr int kScratchPartials = kNormBlocks;  // 16 KiB per device
static __device__ __align__(256) DD scratch[kScratchPartials];
constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[kMaxDevices];  // device address of `scratch`, per device

static int scratch_address(void **ptr)
{
    int dev = 0;
    int rc = check_hip(hipGetDevice(&dev), "hipGetDevice");
    if (rc) return rc;
    if (dev < 0 || dev >= kMaxDevices) return set_error(PRK_EINVAL, "device %d beyond the %d supported", dev, kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        rc = check_hip(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "norm scratch address");
        if (rc) return rc;
        if (!p) return set_error(PRK_EHIP, "norm scratch address is null");
        g_scratch_ptr[dev] = p;
    }
    *ptr = g_scratch_ptr[dev];
    return PRK_OK;
}

int l1norm_async(int dtype, int n, long long pitch, int radius, const void *out, double *d_result, void *partials,
                 hipStream_t s)
{
    if (!valid_dtype(dtype)) return set_error(PRK_EINVAL, "unknown dtype %d", dtype);
    if (n < 1 || pitch < n || !out || !d_result || !partials || radius < 1 || 2 * radius + 1 > n)
        return set_error(PRK_EINVAL, "bad norm arguments (n=%d radius=%d)", n, radius);
    return enqueue_l1norm(dtype, n, pitch, radius, out, d_result, (DD *)partials, s);
}

// ---------------------------------------------------------------------------
// Crash backtraces.  With the handlers installed, a fatal signal in any
// thread (a host fault in the server's worker thread, say) first writes the
// faulting thread's native frames to stderr, then the handler that was
// there before (Python's faulthandler under pytest, or the default action)
// runs.  Only async-signal-safe calls are made in the handler; backtrace()
// is called once at install so that its first use, which may load libgcc,
// is not in a handler.
// ---------------------------------------------------------------------------
constexpr int kCrashSignals[] = {SIGSEGV, SIGBUS, SIGILL, SIGFPE, SIGABRT};
constexpr int kNumCrashSignals = (int)(sizeof(kCrashSignals) / sizeof(kCrashSignals[0]));
struct sigaction g_prev_action[kNumCrashSignals];
bool g_crash_installed = false;
std::mutex g_crash_mu;

void crash_write(const char *s) { (void)!write(2, s, strlen(s)); }

void crash_handler(int sig)
{
    char digits[12], num[12];
    int nd = 0, k = 0;
    for (int v = sig; v > 0 || nd == 0; v /= 10) digits[nd++] = (char)('0' + v % 10);
    while (nd) num[k++] = digits[--nd];
    num[k] = 0;
    crash_write("prk: fatal signal ");
    crash_write(num);
    crash_write(", native frames of the faulting thread:\n");
    void *frames[64];
    backtrace_symbols_fd(frames, backtrace(frames, 64), 2);
    for (int i = 0; i < kNumCrashSignals; ++i)
        if (kCrashSignals[i] == sig) sigaction(sig, &g_prev_action[i], nullptr);
    raise(sig);  // delivered to the previous handler once this one returns
}

}  // namespace prk

using namespace prk;

// ---------------------------------------------------------------------------
// extern "C"
// ---------------------------------------------------------------------------
extern "C" {

int prk_crash_backtrace(int enable)
{
    std::lock_guard<std::mutex> lock(g_crash_mu);
    if (enable && !g_crash_installed) {
        void *f[1];
        (void)backtrace(f, 1);
        struct sigaction sa;
        std::memset(&sa, 0, sizeof sa);
        sa.sa_handler = crash_handler;
        sigemptyset(&sa.sa_mask);
        for (int i = 0; i < kNumCrashSignals; ++i)
            if (sigaction(kCrashSignals[i], &sa, &g_prev_action[i]) != 0) {
                for (int j = 0; j < i; ++j) sigaction(kCrashSignals[j], &g_prev_action[j], nullptr);
                return set_error(PRK_EINVAL, "sigaction failed for signal %d", kCrashSignals[i]);
            }
        g_crash_installed = true;
    } else if (!enable && g_crash_installed) {
        for (int i = 0; i < kNumCrashSignals; ++i) sigaction(kCrashSignals[i], &g_prev_action[i], nullptr);
        g_crash_installed = false;
    }
    return PRK_OK;
}

const char *prk_last_error(void) { return g_last_error.c_str(); }
int prk_abi_version(void) { return PRK_STENCIL_ABI_VERSION; }

int prk_set_rows_per_wave(int rows)
{
    if (rows < 0) return set_error(PRK_EINVAL, "rows per wave must be >= 0");
    g_rows_per_wave = rows;
    return PRK_OK;
}

int prk_set_sweep_variant(int variant)
{
    if (variant < -1 || variant >= kSweepVariants)
        return set_error(PRK_EINVAL, "sweep variant must be -1..%d", kSweepVariants - 1);
    g_variant_override = variant;
    return PRK_OK;
}

int prk_set_sweep_order(int order, int wgs_per_cu)
{
    if (order < -1 || order > 7 || wgs_per_cu < -1 || wgs_per_cu > 16)
        return set_error(PRK_EINVAL, "order must be -1..7 and wgs_per_cu -1..16 (-1: tuned)");
    g_order = order;
    g_wgs_per_cu = wgs_per_cu;
    return PRK_OK;
}

int prk_stencil(int pattern, int radius, int n, int t, const double *in, double *out)
{
    if (t < 1) return set_error(PRK_EINVAL, "tile size must be >= 1, got %d", t);
    SweepPlan p;
    int rc = plan_sweep(pattern, radius, F64, n, n, in, nullptr, out, 0, &p);
    if (rc) return rc;
    return launch_sweep(p, in, nullptr, out, 0);
}

#define PRK_DROPIN(name, pat, r)                                            \
    int name(int n, int t, const double *in, double *out)                   \
    {                                                                       \
        return prk_stencil(pat, r, n, t, in, out);                          \
    }
PRK_DROPIN(prk_star1, STAR, 1)
PRK_DROPIN(prk_star2, STAR, 2)
PRK_DROPIN(prk_star3, STAR, 3)
PRK_DROPIN(prk_star4, STAR, 4)
PRK_DROPIN(prk_star5, STAR, 5)
PRK_DROPIN(prk_grid1, GRID, 1)
PRK_DROPIN(prk_grid2, GRID, 2)
PRK_DROPIN(prk_grid3, GRID, 3)
PRK_DROPIN(prk_grid4, GRID, 4)
PRK_DROPIN(prk_grid5, GRID, 5)
#undef PRK_DROPIN

int prk_add(int n, int t, double *in)
{
    if (t < 1) return set_error(PRK_EINVAL, "tile size must be >= 1, got %d", t);
    return launch_add(F64, n, n, in, 0);
}

int prk_add_ex(int dtype, int n, long long pitch, void *in, void *stream)
{
    return launch_add(dtype, n, pitch, in, (hipStream_t)stream);
}

int prk_sweep(int pattern, int radius, int dtype, int n, long long pitch, const void *in, void *in_next,
              void *out, void *stream)
{
    if (!in_next) return set_error(PRK_EINVAL, "fused sweep needs in_next");
    SweepPlan p;
    int rc = plan_sweep(pattern, radius, dtype, n, pitch, in, in_next, out, 0, &p);
    if (rc) return rc;
    return launch_sweep(p, in, in_next, out, (hipStream_t)stream);
}

int prk_sweep_slab(int pattern, int radius, int dtype, int n, int row0, int rows, long long pitch,
                   const void *in, void *in_next, void *out, void *stream)
{
    if (!in_next) return set_error(PRK_EINVAL, "fused sweep needs in_next");
    const bool inside = row0 >= 0 && rows >= 1 && row0 < n && rows <= n - row0;
    const int top = inside ? std::min(radius, row0) : 0, bot = inside ? std::min(radius, n - row0 - rows) : 0;
    SweepPlan p;
    int rc = plan_sweep(pattern, radius, dtype, n, pitch, in, in_next, out, 0, &p, inside ? top + rows + bot : 0);
    if (rc) return rc;
    if (!inside)
        return set_error(PRK_EINVAL, "slab of rows [%d, %lld) is not inside the %d rows of the grid", row0,
                         (long long)row0 + rows, n);
    // Local row 0 is global row row0 - top.  The first R local rows are halo
    // rows or frame rows (top < R only when row0 < R), and so are the last R,
    // so the outputs, global rows [max(row0, R), min(row0+rows, n-R)), are
    // local rows [R, nrows-R) as for a whole grid (empty when nrows < 2R+1).
    p.span.nrows = top + rows + bot;
    p.span.upd_lo = top;
    p.span.upd_hi = top + rows;
    return launch_sweep(p, in, in_next, out, (hipStream_t)stream);
}

int prk_stencil_ex(int pattern, int radius, int dtype, int n, long long pitch, const void *in, void *out,
                   void *stream)
{
    SweepPlan p;
    int rc = plan_sweep(pattern, radius, dtype, n, pitch, in, nullptr, out, 0, &p);
    if (rc) return rc;
    return launch_sweep(p, in, nullptr, out, (hipStream_t)stream);
}

int prk_init(int init, uint64_t seed, int dtype, int n, long long pitch, void *in, void *out, void *stream)
{
    if (init != PRK_INIT_ANALYTIC && init != PRK_INIT_SEEDED)
        return set_error(PRK_EINVAL, "unknown init kind %d", init);
    if (!valid_dtype(dtype)) return set_error(PRK_EINVAL, "unknown dtype %d", dtype);
    if (n < 1 || pitch < n || !in) return set_error(PRK_EINVAL, "bad grid (n=%d pitch=%lld)", n, pitch);
    const bool vec =
        ((uintptr_t)in | (uintptr_t)out | (unsigned long long)pitch * dtype_size(dtype)) % 16 == 0;
    const int span = 256 * (vec ? vec_width(dtype) : 1);
    const dim3 grid(std::min(1024, (n + span - 1) / span), std::min(n, 65535));
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, (hipStream_t)stream, init, seed, n, pitch, in, out);
    };
    switch (dtype) {
    case F64: vec ? launch(init_kernel<F64, true>) : launch(init_kernel<F64, false>); break;
    case F32: vec ? launch(init_kernel<F32, true>) : launch(init_kernel<F32, false>); break;
    default: vec ? launch(init_kernel<BF16, true>) : launch(init_kernel<BF16, false>); break;
    }
    return check_hip(hipGetLastError(), "init launch");
}

int prk_l1norm(int dtype, int n, long long pitch, int radius, const void *out, double *norm, void *stream)
{
    if (!valid_dtype(dtype)) return set_error(PRK_EINVAL, "unknown dtype %d", dtype);
    if (n < 1 || pitch < n || !out || !norm || radius < 1 || 2 * radius + 1 > n)
        return set_error(PRK_EINVAL, "bad norm arguments (n=%d radius=%d)", n, radius);
    NormWorkspace *ws = nullptr;
    int rc = norm_workspace(&ws);
    if (rc) return rc;
    // the workspace is shared per device: one blocking norm at a time
    static std::mutex norm_mu;
    std::lock_guard<std::mutex> lock(norm_mu);
    hipStream_t s = (hipStream_t)stream;
    rc = enqueue_l1norm(dtype, n, pitch, radius, out, ws->d_result, ws->partials, s);
    if (!rc) rc = check_hip(hipStreamSynchronize(s), "norm sync");
    if (!rc) *norm = *(volatile double *)ws->result;
    return rc;
}

int prk_l1norm_noalloc(int dtype, int n, long long pitch, int radius, const void *out, double *d_norm, void *stream)
{
    if (!valid_dtype(dtype)) return set_error(PRK_EINVAL, "unknown dtype %d", dtype);
    if (n < 1 || pitch < n || !out || !d_norm || radius < 1 || 2 * radius + 1 > n)
        return set_error(PRK_EINVAL, "bad norm arguments (n=%d radius=%d)", n, radius);
    const int blocks = norm_blocks(n, radius);
    if (blocks > kScratchPartials)
        return set_error(PRK_EINVAL, "norm of n=%d needs %d partials; the static scratch holds %d", n, blocks,
                         kScratchPartials);
    void *ptr = nullptr;
    int rc = scratch_address(&ptr);
    if (rc) return rc;
    return enqueue_l1norm(dtype, n, pitch, radius, out, d_norm, (DD *)ptr, (hipStream_t)stream);
}

// The two events of a thread's prk_run calls, made once per thread and device
// and given back when the thread ends.  prk_run returns only once its last
// event has passed, so a call finds them idle.
struct RunEvents {
    int device = -1;
    hipEvent_t e[2] = {nullptr, nullptr};
    void release()
    {
        for (hipEvent_t &x : e) {
            if (x) (void)hipEventDestroy(x);
            x = nullptr;
        }
        device = -1;
    }
    ~RunEvents() { release(); }
    int get()
    {
        int dev = 0;
        int rc = check_hip(hipGetDevice(&dev), "hipGetDevice");
        if (rc || dev == device) return rc;
        release();
        for (hipEvent_t &x : e)
            if (!rc) rc = check_hip(hipEventCreate(&x), "event create");
        if (rc) release();
        else device = dev;
        return rc;
    }
};
static thread_local RunEvents t_run_events;

int prk_run(int pattern, int radius, int dtype, int n, long long pitch, int iterations, void *buf0, void *buf1,
            void *out, void *stream, int *final_in_buf, double *avg_seconds)
{
    if (iterations < 1) return set_error(PRK_EINVAL, "iterations must be >= 1, got %d", iterations);
    if (!buf1 || buf0 == buf1) return set_error(PRK_EINVAL, "run needs two distinct in buffers");
    SweepPlan p;
    int rc = plan_sweep(pattern, radius, dtype, n, pitch, buf0, buf1, out, 0, &p);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    if ((rc = t_run_events.get())) return rc;
    const hipEvent_t e0 = t_run_events.e[0], e1 = t_run_events.e[1];
    // The sweeps run in `passes` passes over the grid (pass.hpp) of nearly
    // equal length.  The final in must end in the buffer that one sweep per
    // pass would leave it in, so the number of passes is odd or even as the
    // number of sweeps is: an even number of iterations takes one pass, an odd
    // one a pass and its last sweep alone.  The other buffer must hold the in
    // before the final one, as after a sweep alone; after a pass the refreshes
    // that the pass made on it are made in the buffer itself (one read and one
    // write of the grid, where another sweep would take four).  Measured
    // against two passes and a sweep: star R=2 FP64 with init and norm, n =
    // 1000, 10 iterations 81 -> 56 us.  A tiling override asks for the sweep
    // kernel itself: one sweep per pass then.
    const bool overridden = g_rows_per_wave > 0 || g_variant_override >= 0 || g_order >= 0 || g_wgs_per_cu >= 0;
    int alone = 1, passes = iterations;
    if (!overridden && pass_built(pattern, radius, dtype) && (p.mode != MODE_ELEM || dtype == BF16)) {
        const auto fit = [](long long sweeps) {
            const int k = (int)((sweeps + kMaxPassSweeps - 1) / kMaxPassSweeps);
            return k + (int)((k ^ sweeps) & 1);
        };
        const long long all = (long long)iterations + 1;
        const int joined = fit(all), apart = fit(iterations), least = pass_min_sweeps(pattern, radius, dtype);
        if (joined < apart && all / joined >= least) {
            alone = 0;
            passes = joined;
        } else if (iterations / apart >= least) {
            passes = apart;
        }
    }
    const bool in_passes = passes + alone < (long long)iterations + 1;
    const long long timed = (long long)iterations + 1 - (in_passes ? 0 : 1);
    void *bufs[2] = {buf0, buf1};
    int cur = 0;
    if (in_passes) {
        // A process's first run would otherwise load its code between the events
        // (0.6 ms, measured on a first run of n = 1000 whose passes take 20 us).
        rc = launch_pass(p, 0, false, buf0, buf1, out, s);
        p.load_only = true;
        if (rc == PRK_OK && alone) rc = launch_sweep(p, buf0, buf1, out, s);
        p.load_only = false;
    } else {
        rc = launch_sweep(p, buf0, buf1, out, s);
        cur = 1;
    }
    if (rc == PRK_OK) rc = check_hip(hipEventRecord(e0, s), "event record");
    long long left = in_passes ? timed - alone : timed;
    int sweeps = 1;
    for (int it = 0; it < passes && rc == PRK_OK; ++it) {
        sweeps = (int)(left / (passes - it));  // spread over the passes left
        rc = sweeps == 1 ? launch_sweep(p, bufs[cur], bufs[cur ^ 1], out, s)
                         : launch_pass(p, sweeps, it == 0, bufs[cur], bufs[cur ^ 1], out, s);
        left -= sweeps;
        cur ^= 1;
    }
    if (rc == PRK_OK && in_passes && alone) {
        rc = launch_sweep(p, bufs[cur], bufs[cur ^ 1], out, s);
        cur ^= 1;
    } else if (rc == PRK_OK && in_passes) {
        rc = launch_add_times(dtype, n, pitch, bufs[cur ^ 1], sweeps - 1, s);
    }
    if (rc == PRK_OK) rc = check_hip(hipEventRecord(e1, s), "event record");
    if (rc == PRK_OK) rc = check_hip(hipEventSynchronize(e1), "event sync");
    float ms = 0.0f;
    if (rc == PRK_OK) rc = check_hip(hipEventElapsedTime(&ms, e0, e1), "event elapsed");
    if (rc) {
        t_run_events.release();  // a failed run may leave them recorded
        return rc;
    }
    if (final_in_buf) *final_in_buf = cur;
    if (avg_seconds) *avg_seconds = 1e-3 * (double)ms / (double)timed;
    return PRK_OK;
}

int prk_triad(long long len, double scalar, double *A, const double *B, const double *C, void *stream)
{
    if (len < 1 || !A || !B || !C) return set_error(PRK_EINVAL, "bad triad arguments");
    if (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) % 16)
        return set_error(PRK_EINVAL, "triad needs 16-byte aligned arrays");
    const long long nv = len / 2;
    if ((nv + 255) / 256 >= (1LL << 32)) return set_error(PRK_EINVAL, "triad length too large");
    const unsigned blocks = (unsigned)std::max<long long>(1, (nv + 255) / 256);
    hipLaunchKernelGGL(triad_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, len, scalar, A, B, C);
    return check_hip(hipGetLastError(), "triad launch");
}

int prk_stream_mix(long long len, const double *in, double *in_next, double *out, void *stream)
{
    if (len < 1 || !in || !in_next || !out || in == in_next || in == out || in_next == out)
        return set_error(PRK_EINVAL, "stream mix needs three separate arrays of len >= 1");
    if (((uintptr_t)in | (uintptr_t)in_next | (uintptr_t)out) % 16)
        return set_error(PRK_EINVAL, "stream mix needs 16-byte aligned arrays");
    const long long nv = len / 2;
    if ((nv + 255) / 256 >= (1LL << 32)) return set_error(PRK_EINVAL, "stream mix length too large");
    const unsigned blocks = (unsigned)std::max<long long>(1, (nv + 255) / 256);
    hipLaunchKernelGGL(stream_mix_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, len, in, in_next, out);
    return check_hip(hipGetLastError(), "stream mix launch");
}

int prk_copy_shape(long long bytes, void *dst, const void *src, int vpl, int nt, int blocks, void *stream)
{
    if (bytes < 16 || bytes % 16 || !dst || !src || ((uintptr_t)dst | (uintptr_t)src) % 16)
        return set_error(PRK_EINVAL, "copy needs a positive multiple of 16 bytes, 16-byte aligned");
    if (vpl != 1 && vpl != 2 && vpl != 4 && vpl != 8) return set_error(PRK_EINVAL, "vpl must be 1, 2, 4 or 8");
    if (nt != 0 && nt != 1) return set_error(PRK_EINVAL, "nt must be 0 or 1");
    if (blocks < 0) return set_error(PRK_EINVAL, "blocks must be >= 0");
    const long long nvec = bytes / 16;
    const long long chunks = (nvec + 256LL * vpl - 1) / (256LL * vpl);
    if (chunks >= (1LL << 31)) return set_error(PRK_EINVAL, "copy too large");
    const unsigned grid = blocks > 0 ? (unsigned)std::min<long long>(blocks, chunks) : (unsigned)chunks;
    hipStream_t s = (hipStream_t)stream;
    switch (vpl) {
    case 1: launch_copy_shape<1>(nt, grid, nvec, (u32x4 *)dst, (const u32x4 *)src, s); break;
    case 2: launch_copy_shape<2>(nt, grid, nvec, (u32x4 *)dst, (const u32x4 *)src, s); break;
    case 4: launch_copy_shape<4>(nt, grid, nvec, (u32x4 *)dst, (const u32x4 *)src, s); break;
    default: launch_copy_shape<8>(nt, grid, nvec, (u32x4 *)dst, (const u32x4 *)src, s); break;
    }
    return check_hip(hipGetLastError(), "copy launch");
}

int prk_copy(long long bytes, void *dst, const void *src, void *stream)
{
    if (bytes < 16 || bytes % 16 || !dst || !src || ((uintptr_t)dst | (uintptr_t)src) % 16)
        return set_error(PRK_EINVAL, "copy needs a positive multiple of 16 bytes, 16-byte aligned");
    const long long nv = bytes / 16;
    if ((nv + 255) / 256 >= (1LL << 32)) return set_error(PRK_EINVAL, "copy too large");
    const unsigned blocks = (unsigned)((nv + 255) / 256);
    hipLaunchKernelGGL(copy_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, nv, (u32x4 *)dst,
                       (const u32x4 *)src);
    return check_hip(hipGetLastError(), "copy launch");
}

}  // extern "C"
