// Batched solves: many independent solves (grids of any size, star/grid,
// radius 1..8, their own iteration counts) in a few launches.
//
// A solve is a sequence of stages over its tiles: stage 0 initialises in,
// stages 1..K+1 are its K+1 sweeps, stage K+2 computes the L1 norm partials
// and stage K+3 reduces them.  Where the stencil has a pass kernel
// (pass.hpp) one pass takes pass_sweeps sweeps: a solve then goes through
// stages 1, 1 + pass_sweeps, 1 + 2 pass_sweeps, ..., the first pass starts
// out from zeros and the last one leaves the norm partials, so stage K+2
// falls away (batch_next_stage).  Pass p reads buffer p%2 and writes buffer
// (p+1)%2.  A tile is one wavefront's share of a stage: 64*V columns of a
// block of rows, processed by the same pass_tile() or wave_tile() as a
// single grid, so a solve's arithmetic does not depend on what else is in
// the launch.
//
// Solves are grouped in classes of one (storage type, pattern, radius), each
// with its own kernel.  One launch is one round: at most one stage of each
// solve, so its tiles are independent (a table gives each workgroup its
// solve, stage and tiles); stage order within a solve comes from launch
// order.  No wave ever waits on another.  (A persistent form, one launch
// whose waves took tiles from queues and waited on per-solve counters, hung
// on MI355X; it was removed and the host refuses PRK_BATCH_PERSISTENT.)
#pragma once

#include <algorithm>

#include "pass.hpp"
#include "prk_stencil.h"
#include "sweep.hpp"

namespace prk {

constexpr int kBatchMaxRadius = kMaxRadius;  // batched and served solves: radii 1..8

// Row pitch (elements) of the grids the library allocates itself (batched,
// served and one-grid-per-launch solves): rows padded to 128 bytes, so that
// every row starts on a cache line.  With rows padded only to 16 bytes, a
// wave's 1 KiB row segment straddles nine lines whenever n is not a multiple
// of 128 bytes: measured on MI355X, batches of equal FP32 grids ran 15-20 %
// slower at n = 600, 1025, 1100, 2100 than at n = 512, 1024, 2048, and
// 11-17 % faster with 128-byte rows (no change at the aligned sizes).
inline long long lib_pitch(int n, int dtype)
{
    const long long per = 128 / (long long)dtype_size(dtype);
    return ((long long)n + per - 1) / per * per;
}

struct DDv {
    double hi, lo;
};

// 32-byte aligned (128 bytes): every workgroup reads its grid's entry with
// scalar loads at the start of a tile.
struct alignas(32) BGrid {
    void *buf0, *buf1, *out;
    long long pitch;         // elements, 128-byte multiple (lib_pitch); padding may be written
    int n, pattern, radius, dtype;
    int iters;               // K: the solve runs K+1 sweeps
    int pass_sweeps;         // sweeps of one pass (the last may have fewer)
    int rows;                // rows per tile
    int strips;              // ceil(n / 64V)
    int ntiles;              // strips * ceil(n / rows)
    int init_kind;
    int pass_rows;           // rows per tile of a pass
    int pass_tiles;          // strips * ceil(n / pass_rows)
    int npartials;           // norm partials: pass_tiles, or ntiles without a pass kernel
    unsigned long long seed;
    DDv *partials;           // the norm partials
    double *norm;            // result: L1 norm / (n-2R)^2
};

__device__ inline DDv dd_add_dev(DDv a, DDv b)
{
#pragma clang fp contract(off)
    const double s = a.hi + b.hi;
    const double bb = s - a.hi;
    const double e = (a.hi - (s - bb)) + (b.hi - bb);
    const double lo = e + a.lo + b.lo;
    const double hi = s + lo;
    return DDv{hi, lo - (hi - s)};
}

// Fixed-order butterfly over the 64 lanes: every lane ends with the total.
__device__ inline DDv wave_reduce_dd(DDv v)
{
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
        DDv o;
        o.hi = __shfl_xor(v.hi, m, 64);
        o.lo = __shfl_xor(v.lo, m, 64);
        // combine in lane order so both partners compute the same value
        const bool low = (__lane_id() & m) == 0;
        v = low ? dd_add_dev(v, o) : dd_add_dev(o, v);
    }
    return v;
}

// Stage 0: in = initial values over the tile (padding columns 0), and out = 0
// if the first sweep does not set it (OUT).
template <int DT, bool OUT>
__device__ inline void init_tile(const BGrid &g, int c0, int r0, int r1, int lane)
{
    typedef typename DTypeTraits<DT>::T T;
    constexpr int V = DTypeTraits<DT>::V, ES = (int)sizeof(T);
    const unsigned row_bytes = (unsigned)(g.pitch * ES);
    const int cm = c0 + lane * V;
    uint64_t state = seeded_state(g.seed, (uint64_t)r0 * (uint64_t)g.n + cm);
    for (int r = r0; r < r1; ++r, state += (uint64_t)g.n * kSeedStep) {
        union { u32x4 v; T e[V]; } x, z;
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const int c = cm + v;
            double val = 0.0;
            if (c < g.n) val = g.init_kind == 0 ? (double)(r + c) : seeded_of_state(state + v * kSeedStep);
            if constexpr (DT == F64) {
                x.e[v] = val;
                z.e[v] = 0.0;
            } else if constexpr (DT == F32) {
                x.e[v] = (float)val;
                z.e[v] = 0.0f;
            } else {
                x.e[v] = f32_to_bf16((float)val);
                z.e[v] = 0;
            }
        }
        const unsigned off = (unsigned)(cm * ES);
        bstore16<0>(row_rsrc((T *)g.buf0 + (long long)r * g.pitch, row_bytes), off, x.v);
        if constexpr (OUT) bstore16<0>(row_rsrc((T *)g.out + (long long)r * g.pitch, row_bytes), off, z.v);
    }
}

// Stage K+2: compensated partial L1 sum of the tile's interior points.
template <int DT>
__device__ inline DDv norm_tile(const BGrid &g, int c0, int r0, int r1, int lane)
{
    typedef typename DTypeTraits<DT>::T T;
    constexpr int V = DTypeTraits<DT>::V, ES = (int)sizeof(T);
    const unsigned row_bytes = (unsigned)(g.pitch * ES);
    const int cm = c0 + lane * V;
    const int R = g.radius;
    double sum = 0.0, comp = 0.0;
    for (int r = max(r0, R); r < min(r1, g.n - R); ++r) {
        union { u32x4 v; T e[V]; } x;
        x.v = bload16<1>(row_rsrc((const T *)g.out + (long long)r * g.pitch, row_bytes), (unsigned)(cm * ES));
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const int c = cm + v;
            if (c >= R && c < g.n - R) {
                double a;
                if constexpr (DT == F64) a = x.e[v];
                else if constexpr (DT == F32) a = (double)x.e[v];
                else a = (double)bf16_to_f32(x.e[v]);
                a = fabs(a);
                const double t = sum + a;
                if (fabs(sum) >= a) comp += (sum - t) + a;
                else comp += (a - t) + sum;
                sum = t;
            }
        }
    }
    return wave_reduce_dd(DDv{sum, comp});
}

// Sweeps of one pass at most: in a batch, where a pass's traffic is already
// small beside the arithmetic of this many; in the server, whose requests
// take turns round by round and whose windows are a few rounds long.
constexpr int kBatchPassSweeps = 64;
constexpr int kServerPassSweeps = 6;

// Rows of a batch's pass tiles: one group of rows per wave.  A pass loads
// every group's window anew, so taller tiles save nothing but the partials,
// and they leave small batches with few waves.  Measured on MI355X, 4, 8 and
// 16 rows: 512 mixed solves of n up to 2048 6.71, 6.65, 6.74 ms; 300 of n up
// to 300 0.34, 0.57, 0.89 ms; 64 of n up to 2048 1.56, 1.65, 1.85 ms.
constexpr int kBatchPassRows = 4;

__device__ inline void pass_tile_at(const BGrid &g, int tile, int &strip, int &r0)
{
    const int nrb = g.pass_tiles / g.strips;
    strip = tile / nrb;
    r0 = (tile - strip * nrb) * g.pass_rows;
}

// The pass that starts with sweep k, over pass tile `tile` (tiles run down
// the strips: the waves of a workgroup share the rows their windows share).
template <int DT, int P, int R>
__device__ inline void pass_stage(const BGrid &g, int k, int tile, int lane)
{
    constexpr int V = DTypeTraits<DT>::V;
    const int p = k / g.pass_sweeps, sweeps = min(g.pass_sweeps, g.iters + 1 - k);
    int strip, r0;
    pass_tile_at(g, tile, strip, r0);
    const bool last = k + sweeps > g.iters;
    NormSum ns;
    pass_tile<DT, P, R, true>((p & 1) ? g.buf1 : g.buf0, (p & 1) ? g.buf0 : g.buf1, g.out, g.pitch, g.n,
                              (strip * 64 + lane) * V, r0, min(r0 + g.pass_rows, g.n), sweeps, (int)g.pitch, k == 0,
                              last, false, ns);
    if (last) {
        const DDv part = wave_reduce_dd(DDv{ns.sum, ns.comp});
        if (lane == 0) g.partials[tile] = part;
    }
}

// Sweep k as a stage of its own.
template <int DT, int P, int R>
__device__ inline void sweep_tile(const BGrid &g, int k, int c0, int r0, int r1, typename DTypeTraits<DT>::T *ring,
                                  int lane)
{
    const void *in = (k & 1) ? g.buf1 : g.buf0;
    void *nx = (k & 1) ? g.buf0 : g.buf1;
    // the grids are the library's own: out's frame may be rewritten with
    // the values it holds (FRAME_REWRITE)
    wave_tile<DT, P, R, true, MODE_VEC, 4, 1, 1, false>(in, nx, g.out, g.pitch, g.n, whole_grid(g.n), c0, r0, r1, 1,
                                                        ring, lane);
}

// ---------------------------------------------------------------------------
// Round form.  One launch = one round.  Every workgroup of the launch has a
// work entry (solve, stage, first tile) and its four waves run four
// consecutive tiles of that stage.
// ---------------------------------------------------------------------------
struct RWork {
    int grid;
    int stage;
    int tile0;
};

struct RoundArgs {
    const BGrid *grids;
    const RWork *work;  // one entry per workgroup
};

// The final norm of a solve from its partials, by one wave.
__device__ inline void final_norm(const BGrid &g, int lane)
{
    DDv acc{0.0, 0.0};
    for (int k = lane; k < g.npartials; k += 64) acc = dd_add_dev(acc, g.partials[k]);
    acc = wave_reduce_dd(acc);
    const long long wd = g.n - 2 * g.radius;
    if (lane == 0) *g.norm = (acc.hi + acc.lo) / (double)(wd * wd);
}

// One kernel per (storage type, pattern, radius): each keeps the registers
// and LDS ring its own stencil needs.
template <int DT, int P, int R>
__global__ __launch_bounds__(kThreads) void batch_round_kernel(RoundArgs a)
{
    typedef SweepGeom<DT, R> G;
    typedef typename G::T T;
    constexpr int SW = G::SW;
    constexpr bool PASS = pass_ok<DT, P, R>();
    constexpr int kRing = PASS ? 1 : G::S * G::LR;  // passes use no LDS
    __shared__ __attribute__((aligned(16))) T lds[kWavesPerBlock][kRing];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const RWork wk = a.work[blockIdx.x];
    const BGrid &g = a.grids[wk.grid];
    const int norm_stage = g.iters + 2;
    const int tile = wk.tile0 + wave;
    if (wk.stage == norm_stage + 1) {
        if (wave == 0) final_norm(g, lane);
        return;
    }
    if constexpr (PASS) {
        if (wk.stage > 0) {
            if (tile < g.pass_tiles) pass_stage<DT, P, R>(g, wk.stage - 1, tile, lane);
            return;
        }
    }
    if (tile >= g.ntiles) return;
    const int rb = tile / g.strips;
    const int c0 = (tile - rb * g.strips) * SW;
    const int r0 = rb * g.rows;
    const int r1 = min(r0 + g.rows, g.n);
    if constexpr (PASS) {
        init_tile<DT, false>(g, c0, r0, r1, lane);
    } else if (wk.stage == 0) {
        init_tile<DT, true>(g, c0, r0, r1, lane);
    } else if (wk.stage < norm_stage) {
        sweep_tile<DT, P, R>(g, wk.stage - 1, c0, r0, r1, lds[wave], lane);
    } else {
        const DDv part = norm_tile<DT>(g, c0, r0, r1, lane);
        if (lane == 0) g.partials[tile] = part;
    }
}

// Host helpers shared by the batch and the server (batch.hip).
int batch_class_of(const prk_solve &s);  // (dtype, pattern, radius) class index
constexpr int kBatchClasses = 3 * 2 * kBatchMaxRadius;
// The solve's sweeps, how many of them a pass takes (passes of equal length,
// the last perhaps shorter) and a pass's tiles.  Without a pass kernel each
// sweep is a stage over the solve's ordinary tiles.
inline void batch_set_passes(BGrid &g, const prk_solve &s, int max_sweeps, int rows)
{
    const int sweeps = s.iterations + 1;
    const int passes = pass_built(s.pattern, s.radius, s.dtype) ? (sweeps + max_sweeps - 1) / max_sweeps : sweeps;
    g.dtype = s.dtype;
    g.iters = s.iterations;
    g.pass_sweeps = (sweeps + passes - 1) / passes;
    g.pass_rows = rows;
    g.pass_tiles = g.strips * ((g.n + rows - 1) / rows);
    g.npartials = pass_built(s.pattern, s.radius, s.dtype) ? g.pass_tiles : g.ntiles;
}
inline bool batch_has_passes(const BGrid &g) { return pass_built(g.pattern, g.radius, g.dtype); }
// The buffer (0 or 1) that holds the final in.
inline int batch_final_buf(const BGrid &g) { return ((g.iters + g.pass_sweeps) / g.pass_sweeps) & 1; }
inline int batch_last_stage(const BGrid &g) { return g.iters + 3; }
inline int batch_next_stage(const BGrid &g, int stage)
{
    if (stage < 1 || stage > g.iters + 1) return stage + 1;
    const int next = std::min(stage + g.pass_sweeps, g.iters + 2);
    return next == g.iters + 2 && batch_has_passes(g) ? g.iters + 3 : next;
}
// Tiles of a stage.
inline int batch_stage_tiles(const BGrid &g, int stage)
{
    if (stage == batch_last_stage(g)) return 1;
    return stage > 0 && batch_has_passes(g) ? g.pass_tiles : g.ntiles;
}
int batch_launch_round(int cls, const RoundArgs &a, unsigned blocks, hipStream_t s);
int batch_validate_solve(const prk_solve &s);

// Error of a reduced-precision result x (FP32 or BF16, pitch xp) against the
// same solve in FP64 y (pitch yp) over the interior R <= i, j < n-R:
// out[0] = max |x-y|, out[1] = sum |x-y|, out[2] = sum (x-y)^2,
// out[3] = sum y^2, each summed in a fixed order (kErrBlocks partials of
// four doubles in `partials`, then one block), on stream s.
constexpr int kErrBlocks = 256;
int error_vs_f64_launch(int dtype, const void *x, long long xp, const double *y, long long yp, int n, int R,
                        double *partials, double *out, hipStream_t s);

}  // namespace prk
