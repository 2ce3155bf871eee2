// Several sweeps in one pass over the grid.
//
// The driver's loop is out += S(in), in += 1, again and again, and the
// refresh is pointwise: the input of sweep t at a point is that point's own
// initial value after t refreshes.  So a wave that holds the window of its
// output points (their columns and rows and R on each side) can run any
// number of sweeps on it without reading a neighbour again: per sweep it
// forms every sum from the window, adds it to out, and refreshes the whole
// window, halo included.  Every operation of every sweep is done, on the
// operands and in the order of the sweep kernel (sweep.hpp), with out and
// the window rounded to the storage type after each sweep, so results are
// bitwise those of T separate sweeps (FP64: see tap_f64); what goes away is
// their traffic, 2 reads and 2 writes of the grid per pass instead of per
// sweep.
//
// What bounds it: the VALU, not HBM.  Per point and sweep the FP64 star R=2
// takes 8 operations for the sum, one for out and (M+2R)/M + 2R/V = 4 for
// the window (M = 4 rows, V = 2 columns per lane), 13 in all, and runs at
// 92 % of the rate at which a loop of FP64 fmas issues on MI355X.  Measured
// per sweep at n = 16384 over 50 sweeps, sweep kernel -> passes: FP64 star
// R=2 1410 -> 112 us, star R=5 1532 -> 362, grid R=2 1408 -> 249, grid R=3
// 1705 -> 615; FP32 star R=2 715 -> 55, grid R=3 739 -> 170, grid R=5 1014
// -> 397; BF16 star R=2 403 -> 102, star R=8 494 -> 396, grid R=2 406 -> 204.
// Two vectors per lane (fewer halo columns to refresh) gave the FP64 star R=3
// 5 % over 50 sweeps and cost every pass twice its loading and storing time.
//
// Mapping.  A lane owns V columns (16 bytes) of M output rows and keeps
// their window in registers: (M+2R) x (V+2R) values, for the stars without
// the corners nothing reads.  M is the largest that leaves room for two or
// more waves per SIMD (pass_rows).  A group of M rows is loaded straight
// from global memory, one 16-byte buffer load per row and vector: the waves
// of a workgroup take row groups below one another, so the rows their
// windows share come from L1 and L2, and with T sweeps of arithmetic per
// load nothing would be gained by parking rows in LDS (no LDS is used).
#pragma once

#include "sweep.hpp"

namespace prk {

// Rows per wave group; 0: no pass kernel (the grid stencils whose window
// does not fit the registers; their single sweep is bound by its arithmetic,
// not by HBM, so a pass would gain nothing).
template <int DT, int P, int R>
constexpr int pass_rows()
{
    if (P == STAR) return DT == F64 ? (R <= 5 ? 4 : 2) : DT == F32 ? (R <= 6 ? 4 : 2) : (R <= 3 ? 4 : 2);
    if (DT == F64) return R <= 2 ? 4 : R <= 4 ? 2 : 0;
    if (DT == F32) return R <= 3 ? 4 : R <= 5 ? 2 : 0;
    return R <= 2 ? 2 : 0;
}

template <int DT, int P, int R>
constexpr bool pass_ok() { return pass_rows<DT, P, R>() > 0; }

// Sweeps from which a pass beats that many sweeps on their own: loading a
// wide window takes longer than the two sweeps save (n = 16384, two sweeps:
// FP32 grid R=5 1074 us each in a pass, 870 alone; BF16 star R=7 485, 450;
// with three 746 and 409).
constexpr int pass_min_sweeps(int pattern, int radius, int dtype)
{
    return (pattern == GRID && ((dtype == F64 && radius >= 3) || (dtype == F32 && radius >= 5))) ||
                   (dtype == BF16 && radius >= 7)
               ? 3
               : 2;
}

template <int DT, int... I>
constexpr bool pass_built_dtype(int pattern, int radius, std::integer_sequence<int, I...>)
{
    constexpr bool star[] = {pass_ok<DT, STAR, I + 1>()...}, grid[] = {pass_ok<DT, GRID, I + 1>()...};
    return (pattern == STAR ? star : grid)[radius - 1];
}

// Whether a valid stencil has a pass kernel.
inline bool pass_built(int pattern, int radius, int dtype)
{
    typedef std::make_integer_sequence<int, kMaxRadius> Radii;
    return dtype == F64 ? pass_built_dtype<F64>(pattern, radius, Radii{})
           : dtype == F32 ? pass_built_dtype<F32>(pattern, radius, Radii{})
                          : pass_built_dtype<BF16>(pattern, radius, Radii{});
}

constexpr bool power_of_two(double w)
{
    double a = w < 0 ? -w : w;
    if (a == 0.0) return false;
    while (a < 1.0) a = a * 2.0;
    while (a > 1.0) a = a * 0.5;
    return a == 1.0;
}

// Tap K of one FP64 sum, in the generator's order.  A product by a power of
// two is exact unless it falls below the normal range, so there the multiply
// and the add are one fma with the same result (FMA).  No product falls that
// low for a value the library refreshed (in + 1) or seeded itself, which is 0
// or at least 2^-53 in magnitude; the first sweep over a caller's values
// multiplies and adds.
template <int P, int R, int M, int V, bool FMA, int K>
__device__ inline void pass_tap_f64(const double (&w)[M + 2 * R][V + 2 * R], double (&s)[M][V])
{
#pragma clang fp contract(off)
    constexpr Tap t = Stencil<P, R>::taps.t[K];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const double x = w[m + R + t.di][v + R + t.dj];
            if constexpr (K == 0)
                s[m][v] = x * t.w;
            else if constexpr (FMA && power_of_two(t.w))
                s[m][v] = __builtin_fma(x, t.w, s[m][v]);
            else
                s[m][v] = s[m][v] + x * t.w;
        }
}

template <int P, int R, int M, int V, bool FMA, size_t... I>
__device__ inline void pass_taps_f64(const double (&w)[M + 2 * R][V + 2 * R], double (&s)[M][V],
                                     std::index_sequence<I...>)
{
    (pass_tap_f64<P, R, M, V, FMA, (int)I>(w, s), ...);
}

// The reduced-precision sums of one output row: the pairs of the stars, the
// ring sums of the grids (operand for operand those of sweep.hpp).
template <int R, int M, int V, int K>
__device__ inline void pass_pair(const float (&w)[M + 2 * R][V + 2 * R], float (&acc)[M][V])
{
#pragma clang fp contract(off)
    constexpr Tap t = Stencil<STAR, R>::pairs.t[K];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const float d = w[m + R + t.di][v + R + t.dj] - w[m + R - t.di][v + R - t.dj];
            if constexpr (K == 0)
                acc[m][v] = (float)t.w * d;
            else
                acc[m][v] = __builtin_fmaf((float)t.w, d, acc[m][v]);
        }
}

template <int R, int M, int V, size_t... I>
__device__ inline void pass_pairs(const float (&w)[M + 2 * R][V + 2 * R], float (&acc)[M][V],
                                  std::index_sequence<I...>)
{
    (pass_pair<R, M, V, (int)I>(w, acc), ...);
}

template <int R, int M, int V, int J>
__device__ inline void pass_rings(const float (&w)[M + 2 * R][V + 2 * R], int m, float (&vs)[V + 2 * R],
                                  float (&acc)[V])
{
    ring_step<R, V, R, J>(w[m + R + J], w[m + R - J], vs, acc);
    if constexpr (J < R) pass_rings<R, M, V, J + 1>(w, m, vs, acc);
}

// x rounded to the storage type, as the type the sums are formed in.
template <int DT, int N, typename C>
__device__ inline void round_storage(C (&x)[N])
{
    if constexpr (DT == BF16) {
        bf16_t h[N];
        from_f32_vec<N>(x, h);
#pragma unroll
        for (int i = 0; i < N; ++i) x[i] = bf16_to_f32(h[i]);
    }
}

// One 16-byte vector of row r at byte offset off (kOOB: zeros).  ALIGNED:
// rows on 16-byte boundaries and the row resource a whole number of vectors.
// Otherwise FP64 and FP32 rows still take one 16-byte load where the vector
// lies inside the row (buffer loads need no more than 4-byte alignment) and
// the vectors over either end, and BF16 rows, are read by element.
template <int DT, bool ALIGNED, int AUX>
__device__ inline u32x4 pass_load(__amdgpu_buffer_rsrc_t r, int col, int n)
{
    typedef typename DTypeTraits<DT>::T T;
    constexpr int V = DTypeTraits<DT>::V, ES = (int)sizeof(T);
    if constexpr (ALIGNED) return bload16<AUX>(r, (unsigned)(col * ES));  // col < 0 wraps out of range
    union { u32x4 v; T e[V]; } x;
    const bool whole = ES >= 4 && col >= 0 && col + V <= n;
    if (whole) {
        x.v = bload16<AUX>(r, (unsigned)(col * ES));
    } else {
#pragma unroll
        for (int v = 0; v < V; ++v)
            x.e[v] = bload_elem<T, AUX>(r, col + v >= 0 && col + v < n ? (unsigned)((col + v) * ES) : kOOB);
    }
    return x.v;
}

// Elements [lo, hi) of one vector at column col.
template <int DT, bool ALIGNED, int AUX>
__device__ inline void pass_store(__amdgpu_buffer_rsrc_t r, int col, int lo, int hi, const u32x4 &val)
{
    typedef typename DTypeTraits<DT>::T T;
    constexpr int V = DTypeTraits<DT>::V, ES = (int)sizeof(T);
    if ((ALIGNED || ES >= 4) && col >= lo && col + V <= hi) {
        bstore16<AUX>(r, (unsigned)(col * ES), val);
    } else {
        union { u32x4 v; T e[V]; } x;
        x.v = val;
#pragma unroll
        for (int v = 0; v < V; ++v)
            bstore_elem<T, AUX>(r, col + v >= lo && col + v < hi ? (unsigned)((col + v) * ES) : kOOB, x.e[v]);
    }
}

// Compensated sum of |x| (Neumaier): the lane's share of an L1 norm.
struct NormSum {
    double sum = 0.0, comp = 0.0;
    __device__ inline void add(double x)
    {
#pragma clang fp contract(off)
        const double a = fabs(x), t = sum + a;
        comp += fabs(sum) >= a ? (sum - t) + a : (a - t) + sum;
        sum = t;
    }
};

// `sweeps` sweeps of rows [r0, r1) and the lane's V columns at cm of an
// n x n grid: in is read, in_next gets in after `sweeps` refreshes (columns
// below st_cols), out is updated on the interior.  `first`: out holds
// nothing yet and starts from zeros, frame included (columns below st_cols).
// `last`: adds |out| over the lane's interior points to `norm`.  `any`: in
// may hold any values (otherwise refreshed or seeded ones, pass_tap_f64).
template <int DT, int P, int R, bool ALIGNED>
__device__ inline void pass_tile(const void *in_, void *in_next_, void *out_, long long pitch, int n, int cm, int r0,
                                 int r1, int sweeps, int st_cols, bool first, bool last, bool any, NormSum &norm)
{
#pragma clang fp contract(off)
    typedef typename DTypeTraits<DT>::T T;
    typedef std::conditional_t<DT == F64, double, float> C;
    constexpr int M = pass_rows<DT, P, R>(), V = DTypeTraits<DT>::V, ES = (int)sizeof(T);
    constexpr int W = V + 2 * R, NH = (R + V - 1) / V;  // window width, halo vectors per side
    const T *in = (const T *)in_;
    T *in_next = (T *)in_next_, *out = (T *)out_;
    const unsigned row_bytes = (unsigned)(pitch * ES);
    union Vec { u32x4 v; T e[V]; };

#pragma unroll 1
    for (int o = r0; o < r1; o += M) {
        C w[M + 2 * R][W], acc_out[M][V];
#pragma unroll
        for (int k = 0; k < M + 2 * R; ++k) {
            const int row = o - R + k;
            const bool ok = row >= 0 && row < n;  // uniform
            const __amdgpu_buffer_rsrc_t r = row_rsrc(in + (long long)(ok ? row : 0) * pitch, ok ? row_bytes : 0u);
            const bool wide = P == GRID || (k >= R && k < R + M);  // rows whose halo columns are read
#pragma unroll
            for (int q = -NH; q <= NH; ++q) {
                if (q != 0 && !wide) continue;
                Vec x;
                x.v = pass_load<DT, ALIGNED, 0>(r, cm + q * V, n);
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    const int i = R + q * V + v;
                    if (i < 0 || i >= W) continue;
                    if constexpr (DT == F64) w[k][i] = x.e[v];
                    else w[k][i] = to_f32<T>(x.e[v]);
                }
            }
        }
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const bool ok = !first && o + m >= R && o + m < n - R;  // uniform
            const __amdgpu_buffer_rsrc_t r = row_rsrc(out + (long long)(ok ? o + m : 0) * pitch, ok ? row_bytes : 0u);
            Vec x;
            x.v = pass_load<DT, ALIGNED, 2>(r, cm, n);
#pragma unroll
            for (int v = 0; v < V; ++v) {
                if constexpr (DT == F64) acc_out[m][v] = x.e[v];
                else acc_out[m][v] = to_f32<T>(x.e[v]);
            }
        }

#pragma unroll 1
        for (int t = 0; t < sweeps; ++t) {
            C s[M][V];
            if constexpr (DT == F64) {
                typedef std::make_index_sequence<Stencil<P, R>::taps.count> Taps;
                if (any && t == 0) pass_taps_f64<P, R, M, V, false>(w, s, Taps{});
                else pass_taps_f64<P, R, M, V, true>(w, s, Taps{});
            } else if constexpr (P == STAR) {
                pass_pairs<R, M, V>(w, s, std::make_index_sequence<Stencil<P, R>::pairs.count>{});
            } else {
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    float vs[W];
#pragma unroll
                    for (int i = 0; i < W; ++i) vs[i] = w[m + R][i];
                    pass_rings<R, M, V, 1>(w, m, vs, s[m]);
                }
            }
#pragma unroll
            for (int m = 0; m < M; ++m) {
#pragma unroll
                for (int v = 0; v < V; ++v) acc_out[m][v] = acc_out[m][v] + s[m][v];
                round_storage<DT, V>(acc_out[m]);
            }
#pragma unroll
            for (int k = 0; k < M + 2 * R; ++k) {
                if (P == GRID || (k >= R && k < R + M)) {
#pragma unroll
                    for (int i = 0; i < W; ++i) w[k][i] = w[k][i] + (C)1;
                    round_storage<DT, W>(w[k]);
                } else {
                    C c[V];
#pragma unroll
                    for (int v = 0; v < V; ++v) c[v] = w[k][R + v] + (C)1;
                    round_storage<DT, V>(c);
#pragma unroll
                    for (int v = 0; v < V; ++v) w[k][R + v] = c[v];
                }
            }
        }

#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int row = o + m;
            if (row >= r1) break;  // uniform
            const bool inner_row = row >= R && row < n - R;
            if (last && inner_row) {
#pragma unroll
                for (int v = 0; v < V; ++v)
                    if (cm + v >= R && cm + v < n - R) norm.add((double)acc_out[m][v]);
            }
            if (first) {
#pragma unroll
                for (int v = 0; v < V; ++v)
                    acc_out[m][v] = inner_row && cm + v >= R && cm + v < n - R ? acc_out[m][v] : (C)0;
            }
            Vec x, y;
            if constexpr (DT == F64) {
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    x.e[v] = w[R + m][R + v];
                    y.e[v] = acc_out[m][v];
                }
            } else {
                C c[V];
#pragma unroll
                for (int v = 0; v < V; ++v) c[v] = w[R + m][R + v];
                from_f32_vec<V>(c, x.e);
                from_f32_vec<V>(acc_out[m], y.e);
            }
            pass_store<DT, ALIGNED, 2>(row_rsrc(in_next + (long long)row * pitch, row_bytes), cm, 0, st_cols, x.v);
            if (first)
                pass_store<DT, ALIGNED, 2>(row_rsrc(out + (long long)row * pitch, row_bytes), cm, 0, st_cols, y.v);
            else if (inner_row)
                pass_store<DT, ALIGNED, 2>(row_rsrc(out + (long long)row * pitch, row_bytes), cm, R, n - R, y.v);
        }
    }
}

struct PassArgs {
    const void *in;
    void *in_next;
    void *out;
    long long pitch;
    int n;
    int nstrips;  // ceil(n / 64V)
    int rows;     // rows per wave, a multiple of M
    int sweeps;
    int any;      // in may hold any values
};

// A workgroup is four waves on row blocks below one another of one strip of
// 64*V columns; workgroups run along the strips of a row band first.
template <int DT, int P, int R, bool ALIGNED>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) void pass_kernel(PassArgs a)
{
    constexpr int V = DTypeTraits<DT>::V;
    const int band = blockIdx.x / a.nstrips, strip = blockIdx.x - band * a.nstrips;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int r0 = (band * kWavesPerBlock + wave) * a.rows;
    if (r0 >= a.n) return;
    NormSum unused;
    pass_tile<DT, P, R, ALIGNED>(a.in, a.in_next, a.out, a.pitch, a.n, (strip * 64 + lane) * V, r0,
                                 min(r0 + a.rows, a.n), a.sweeps, a.n, false, false, a.any, unused);
}

}  // namespace prk
