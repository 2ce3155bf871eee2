// Matrix transpose for gfx950: one iteration is B += A^T, A += 1
// (Cxx11/transpose.cc:118-131; the HIP driver's transposeNoBankConflict,
// Cxx11/transpose-hip.cc:64-87), both matrices order x order FP64, row-major.
//
// Mapping.  A workgroup owns one tile of A.  It reads the tile's rows of A
// with 16-byte buffer loads, all of them issued before the first is used,
// writes A + 1 back to the same addresses, and parks the tile in LDS (rows
// padded by one element so that reading a column spreads over the banks).
// Then it issues the loads of the matching rows of B, waits for the others'
// share of the tile, adds the tile's columns to B and stores it.  Every element
// of A and B is read once and written once: 32 bytes per element, the
// algorithmic traffic of the reference's Rate (4 * 8 * order^2 bytes).  What
// bounds it is HBM, at the rate the tiles' short row segments reach
// (launch_transpose).
// Edges: rows and columns beyond `order` are out-of-range buffer offsets
// (reads give 0, writes are dropped).  Where order is odd, rows start on
// 8-byte boundaries, which the 16-byte accesses take as they are; the tiles
// that hold a row's last column, whose vector would run past the row, move
// single elements.  Large matrices with such rows have a kernel of 8-byte
// accesses.
//
// Values stay integers below 2^53 (order^2 * (iterations + 1) plus the
// added ones), so every sum is exact and results equal the reference's bit
// for bit in any order of operations.
#include <hip/hip_runtime.h>

#include <mutex>
#include <vector>

#include "prk_internal.hpp"
#include "prk_stencil.h"
#include "sweep.hpp"

namespace prk {
namespace {

struct TransposeArgs {
    double *A;
    double *B;
    int order;
    int ntr, ntc;  // tiles down / across A
    int mode;      // tile order: 0 row-major, 1 column-major, 2 groups of 8 tile rows
};

// Workgroup -> tile (tr, tc) of A.  Mode 2 walks groups of eight tile rows
// column by column, so the workgroups in flight read eight row bands of A
// and write eight adjacent column bands of each B row band.
__device__ inline void tile_of_transpose(const TransposeArgs &a, int b, int &tr, int &tc)
{
    if (a.mode == 1) {
        tc = b / a.ntr;
        tr = b - tc * a.ntr;
    } else if (a.mode == 2) {
        const int per = 8 * a.ntc;            // tiles in a full group
        const int g = b / per, k = b - g * per;
        const int rows = min(8, a.ntr - g * 8);  // tile rows in this group
        tc = k / rows;
        tr = g * 8 + (k - tc * rows);
    } else {
        tr = b / a.ntc;
        tc = b - tr * a.ntc;
    }
}

// Two neighbouring elements; SPLIT: as single ones, without the second
// where `last` (offsets of kOOB and above, up to the 95 MB a tile spans, are
// out of range).
template <int AUX, bool SPLIT>
__device__ inline u32x4 load2(__amdgpu_buffer_rsrc_t r, unsigned off, bool last)
{
    if constexpr (!SPLIT) return bload16<AUX>(r, off);
    union { u32x4 v; double d[2]; } x;
    x.d[0] = bload_elem<double, AUX>(r, off);
    x.d[1] = bload_elem<double, AUX>(r, last ? kOOB : off + 8u);
    return x.v;
}

template <int AUX, bool SPLIT>
__device__ inline void store2(__amdgpu_buffer_rsrc_t r, unsigned off, bool last, const u32x4 &v)
{
    if constexpr (!SPLIT) {
        bstore16<AUX>(r, off, v);
    } else {
        union { u32x4 v; double d[2]; } x;
        x.v = v;
        bstore_elem<double, AUX>(r, off, x.d[0]);
        bstore_elem<double, AUX>(r, last ? kOOB : off + 8u, x.d[1]);
    }
}

// Non-temporal accesses of a tile.  NT_A: the stores of A alone, and B's rows
// are loaded behind the barrier, after A's stores.
enum { NT_NONE, NT_STORES, NT_A, NT_ALL };

// One TR x TC tile of A (TR rows, TC columns) on NTH threads.
template <int TR, int TC, int NTH, int NT, bool SPLIT>
__device__ inline void transpose_tile(const TransposeArgs &a, int tr, int tc, double (*tile)[TC + 1])
{
    constexpr int LPR1 = TC / 2, RPP1 = NTH / LPR1, NP1 = TR / RPP1;  // A rows
    constexpr int LPR2 = TR / 2, RPP2 = NTH / LPR2, NP2 = TC / RPP2;  // B rows
    static_assert(NP1 >= 1 && NP2 >= 1 && RPP1 * NP1 == TR && RPP2 * NP2 == TC, "tile shape");
    constexpr int AUX_LD = NT == NT_ALL ? 2 : 0;
    constexpr int AUX_ST_A = NT == NT_NONE ? 0 : 2, AUX_ST_B = NT == NT_A ? 0 : AUX_ST_A;
    const int order = a.order;
    const unsigned row_bytes = (unsigned)order * 8u;
    union V { u32x4 v; double d[2]; };
    // One resource per matrix, the rows of the tile (at most 256 rows of
    // 46340 elements: 95 MB), so that it is the same in every lane; rows past
    // the last lie beyond its range, columns past the last are moved there.
    const __amdgpu_buffer_rsrc_t ra =
        row_rsrc(a.A + (long long)tr * TR * order, (unsigned)min(TR, order - tr * TR) * row_bytes);
    const __amdgpu_buffer_rsrc_t rb =
        row_rsrc(a.B + (long long)tc * TC * order, (unsigned)min(TC, order - tc * TC) * row_bytes);
    // this thread's elements: of A, rows tr*TR + p*RPP1 + ar, columns ac and
    // ac + 1 of the tile; of B, rows tc*TC + p*RPP2 + br, columns bc, bc + 1
    const int ar = threadIdx.x / LPR1, ac = (threadIdx.x - ar * LPR1) * 2;
    const int br = threadIdx.x / LPR2, bc = (threadIdx.x - br * LPR2) * 2;
    const unsigned off_a = tc * TC + ac < order ? ar * row_bytes + (unsigned)(tc * TC + ac) * 8u : kOOB;
    const unsigned off_b = tr * TR + bc < order ? br * row_bytes + (unsigned)(tr * TR + bc) * 8u : kOOB;
    const unsigned step_a = RPP1 * row_bytes, step_b = RPP2 * row_bytes;
    // the last column's second element would be the next row's first
    const bool last_a = tc * TC + ac + 1 >= order, last_b = tr * TR + bc + 1 >= order;

    V x[NP1], y[NP2];
#pragma unroll
    for (int p = 0; p < NP1; ++p) x[p].v = load2<AUX_LD, SPLIT>(ra, off_a + p * step_a, last_a);
#pragma unroll
    for (int p = 0; p < NP1; ++p) {
        V z;
        z.d[0] = x[p].d[0] + 1.0;
        z.d[1] = x[p].d[1] + 1.0;
        tile[p * RPP1 + ar][ac] = x[p].d[0];
        tile[p * RPP1 + ar][ac + 1] = x[p].d[1];
        store2<AUX_ST_A, SPLIT>(ra, off_a + p * step_a, last_a, z.v);
    }
    if (NT == NT_A) __syncthreads();
#pragma unroll
    for (int p = 0; p < NP2; ++p) y[p].v = load2<AUX_LD, SPLIT>(rb, off_b + p * step_b, last_b);
    if (NT != NT_A) __syncthreads();
#pragma unroll
    for (int p = 0; p < NP2; ++p) {
        y[p].d[0] = y[p].d[0] + tile[bc][p * RPP2 + br];
        y[p].d[1] = y[p].d[1] + tile[bc + 1][p * RPP2 + br];
        store2<AUX_ST_B, SPLIT>(rb, off_b + p * step_b, last_b, y[p].v);
    }
}

// ODD: order is odd; the tiles that hold the last column of A or B split
// their vectors.
template <int TR, int TC, int NTH, int NT, bool ODD>
__global__ __launch_bounds__(NTH) void transpose_kernel(TransposeArgs a)
{
    __shared__ double tile[TR][TC + 1];
    int tr, tc;
    tile_of_transpose(a, blockIdx.x, tr, tc);
    if (ODD && ((tc + 1) * TC > a.order || (tr + 1) * TR > a.order))
        transpose_tile<TR, TC, NTH, NT, true>(a, tr, tc, tile);
    else
        transpose_tile<TR, TC, NTH, NT, false>(a, tr, tc, tile);
}

// One 64 x 64 tile of A in 8-byte accesses, non-temporal stores, a resource
// for each row (one for the tile took 1 to 5 % longer above order 13000: 18473
// 2341 us, 2390; 14497 1632, 1715).
__global__ __launch_bounds__(256) void transpose_kernel_8b(TransposeArgs a)
{
    constexpr int T = 64, RPP = 4, NP = T / RPP;  // four rows at a time
    __shared__ double tile[T][T + 1];
    int tr, tc;
    tile_of_transpose(a, blockIdx.x, tr, tc);
    const int order = a.order;
    const unsigned row_bytes = (unsigned)order * 8u;
    const int r = threadIdx.x / T, c = threadIdx.x - r * T;
    const unsigned off_a = tc * T + c < order ? (unsigned)(tc * T + c) * 8u : kOOB;
    const unsigned off_b = tr * T + c < order ? (unsigned)(tr * T + c) * 8u : kOOB;
    __amdgpu_buffer_rsrc_t rs[NP];
    double x[NP];
    auto load = [&](const double *m, int row0, unsigned off) {
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const int row = row0 + p * RPP + r;
            const bool ok = row < order;
            rs[p] = row_rsrc(m + (long long)(ok ? row : 0) * order, ok ? row_bytes : 0u);
            x[p] = bload_elem<double, 0>(rs[p], off);
        }
    };
    load(a.A, tr * T, off_a);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        tile[p * RPP + r][c] = x[p];
        bstore_elem<double, 2>(rs[p], off_a, x[p] + 1.0);
    }
    __syncthreads();
    load(a.B, tc * T, off_b);
#pragma unroll
    for (int p = 0; p < NP; ++p) bstore_elem<double, 2>(rs[p], off_b, x[p] + tile[c][p * RPP + r]);
}

// One 128 x 128 tile of A on 1024 threads, in two halves through 66 KiB of
// LDS, so that both matrices move in 1 KiB row segments (the 64 x 128 tile
// writes B in 512-byte segments) and two workgroups fit on a CU.  Each
// thread loads 16 doubles of A (eight 16-byte loads, rows p*16 + t/64,
// columns 2(t%64), 2(t%64)+1 of the tile) and writes A + 1 back at once.
// Half h = 0, 1: the threads holding tile columns [64h, 64h+64) park them in
// LDS (128 rows x 64 columns, rows padded by one element); after a barrier
// every thread adds four 16-byte pieces of B rows 64h + q*16 + t/64 (tile
// rows 2(t%64), 2(t%64)+1 as B columns) and stores them; a barrier ends the
// half before the LDS is reused.
template <int NT>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(8))) void transpose_kernel_2h(TransposeArgs a)
{
    constexpr int T = 128, H = 64, NTH = 1024, RPP = NTH / 64;  // 16 A rows per pass
    constexpr int AUX_ST = NT ? 2 : 0;
    __shared__ double half[T][H + 1];

    int tr, tc;
    tile_of_transpose(a, blockIdx.x, tr, tc);
    const int order = a.order;
    const unsigned row_bytes = (unsigned)order * 8u;
    union V { u32x4 v; double d[2]; };
    // lr: the wave's index, uniform (row resources stay in scalar registers)
    const int lr = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l2 = (threadIdx.x & 63) * 2;

    // A: tile rows p*16 + lr, columns l2, l2+1
    V x[T / RPP];
    {
        const int c = tc * T + l2;
        const unsigned off = c < order ? (unsigned)c * 8u : kOOB;
        __amdgpu_buffer_rsrc_t rs[T / RPP];
#pragma unroll
        for (int p = 0; p < T / RPP; ++p) {
            const int r = tr * T + p * RPP + lr;
            const bool ok = r < order;
            rs[p] = row_rsrc(a.A + (long long)(ok ? r : 0) * order, ok ? row_bytes : 0u);
            x[p].v = bload16<0>(rs[p], off);
        }
#pragma unroll
        for (int p = 0; p < T / RPP; ++p) {
            V y;
            y.d[0] = x[p].d[0] + 1.0;
            y.d[1] = x[p].d[1] + 1.0;
            bstore16<AUX_ST>(rs[p], off, y.v);
        }
    }
    // B rows tc*T + 64h + q*16 + lr, columns tr*T + l2, l2+1
    const int cb = tr * T + l2;
    const unsigned offb = cb < order ? (unsigned)cb * 8u : kOOB;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if ((l2 >> 6) == h) {
#pragma unroll
            for (int p = 0; p < T / RPP; ++p) {
                half[p * RPP + lr][l2 - H * h] = x[p].d[0];
                half[p * RPP + lr][l2 - H * h + 1] = x[p].d[1];
            }
        }
        __syncthreads();
        V b[H / RPP];
        __amdgpu_buffer_rsrc_t rs[H / RPP];
#pragma unroll
        for (int q = 0; q < H / RPP; ++q) {
            const int y = tc * T + H * h + q * RPP + lr;
            const bool ok = y < order;
            rs[q] = row_rsrc(a.B + (long long)(ok ? y : 0) * order, ok ? row_bytes : 0u);
            b[q].v = bload16<0>(rs[q], offb);
        }
#pragma unroll
        for (int q = 0; q < H / RPP; ++q) {
            const int j = q * RPP + lr;  // column of the half
            b[q].d[0] = b[q].d[0] + half[l2][j];
            b[q].d[1] = b[q].d[1] + half[l2 + 1][j];
            bstore16<AUX_ST>(rs[q], offb, b[q].v);
        }
        __syncthreads();
    }
}

// A = 0, 1, ..., order^2 - 1 (row-major), B = 0 (Cxx11/transpose.cc:110-112).
__global__ __launch_bounds__(256) void transpose_init_kernel(double *A, double *B, long long nn)
{
    for (long long k = (long long)blockIdx.x * 256 + threadIdx.x; k < nn; k += (long long)gridDim.x * 256) {
        A[k] = (double)k;
        B[k] = 0.0;
    }
}

// Partial sums of |B[j][i] - ((i*order + j)(K+1) + K(K+1)/2)| in a fixed order
// (Cxx11/transpose.cc:137-146).
constexpr int kChkBlocks = 1024;
constexpr int kChkThreads = 256;

__global__ __launch_bounds__(kChkThreads) void transpose_check_kernel(const double *B, int order, int iterations,
                                                                     double *partials)
{
#pragma clang fp contract(off)
    const double addit = (iterations + 1.0) * (iterations / 2.0);
    const long long nn = (long long)order * order;
    double s = 0.0;
    for (long long k = (long long)blockIdx.x * kChkThreads + threadIdx.x; k < nn;
         k += (long long)kChkBlocks * kChkThreads) {
        const long long j = k / order, i = k - j * order;  // k = j*order + i
        const double ref = (double)(i * order + j) * (1.0 + iterations) + addit;
        s += fabs(B[k] - ref);
    }
    __shared__ double red[kChkThreads];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = kChkThreads / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) partials[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(kChkThreads) void transpose_check_final(const double *partials, double *out)
{
    __shared__ double red[kChkThreads];
    double s = 0.0;
    for (int k = threadIdx.x; k < kChkBlocks; k += kChkThreads) s += partials[k];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = kChkThreads / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0];
}

std::mutex g_chk_mu;
std::vector<double *> g_chk_ws;  // per device: kChkBlocks partials + 1 result

int check_workspace(double **ws)
{
    int dev = 0;
    int rc = check_hip(hipGetDevice(&dev), "hipGetDevice");
    if (rc) return rc;
    std::lock_guard<std::mutex> lock(g_chk_mu);
    if ((int)g_chk_ws.size() <= dev) g_chk_ws.resize(dev + 1, nullptr);
    if (!g_chk_ws[dev]) {
        void *p = nullptr;
        rc = check_hip(hipMalloc(&p, sizeof(double) * (kChkBlocks + 1)), "transpose check workspace");
        if (rc) return rc;
        g_chk_ws[dev] = (double *)p;
    }
    *ws = g_chk_ws[dev];
    return PRK_OK;
}

int transpose_args(int order, const double *A, const double *B)
{
    if (order < 1) return set_error(PRK_EINVAL, "matrix order must be positive, got %d", order);
    if (order > 46340) return set_error(PRK_EINVAL, "matrix order %d too large (overflow risk)", order);
    if (!A || !B) return set_error(PRK_EINVAL, "null matrix pointer");
    if (A == B) return set_error(PRK_EINVAL, "A and B must be separate matrices");
    if ((uintptr_t)A % 8 || (uintptr_t)B % 8) return set_error(PRK_EINVAL, "matrices must be 8-byte aligned");
    return PRK_OK;
}

int g_tr_shape = -1, g_tr_mode = -1;  // -1: the defaults below

template <int TR, int TC, int NTH = 256>
int launch_shape(TransposeArgs a, int nt, hipStream_t s)
{
    a.ntr = (a.order + TR - 1) / TR;
    a.ntc = (a.order + TC - 1) / TC;
    const unsigned blocks = (unsigned)a.ntr * (unsigned)a.ntc;
    // NT_ALL: one workgroup per CU of the 64 x 128 tiles (more than half of
    // its LDS each)
    constexpr size_t lds = sizeof(double) * TR * (TC + 1), half = 80u * 1024u;
    const size_t dyn = nt == NT_ALL && lds > half / 2 && lds < half ? half + 4096u - lds : 0;
    if (a.order & 1)
        hipLaunchKernelGGL((transpose_kernel<TR, TC, NTH, NT_NONE, true>), dim3(blocks), dim3(NTH), 0, s, a);
    else if (nt == NT_ALL)
        hipLaunchKernelGGL((transpose_kernel<TR, TC, NTH, NT_ALL, false>), dim3(blocks), dim3(NTH), dyn, s, a);
    else if (nt == NT_STORES)
        hipLaunchKernelGGL((transpose_kernel<TR, TC, NTH, NT_STORES, false>), dim3(blocks), dim3(NTH), 0, s, a);
    else if (nt == NT_A)
        hipLaunchKernelGGL((transpose_kernel<TR, TC, NTH, NT_A, false>), dim3(blocks), dim3(NTH), 0, s, a);
    else
        hipLaunchKernelGGL((transpose_kernel<TR, TC, NTH, NT_NONE, false>), dim3(blocks), dim3(NTH), 0, s, a);
    return check_hip(hipGetLastError(), "transpose launch");
}

int launch_8b(TransposeArgs a, hipStream_t s)
{
    a.ntr = (a.order + 63) / 64;
    a.ntc = a.ntr;
    const unsigned blocks = (unsigned)a.ntr * (unsigned)a.ntc;
    hipLaunchKernelGGL(transpose_kernel_8b, dim3(blocks), dim3(256), 0, s, a);
    return check_hip(hipGetLastError(), "transpose launch");
}

int launch_2h(TransposeArgs a, hipStream_t s)
{
    a.ntr = (a.order + 127) / 128;
    a.ntc = a.ntr;
    const unsigned blocks = (unsigned)a.ntr * (unsigned)a.ntc;
    hipLaunchKernelGGL(transpose_kernel_2h<1>, dim3(blocks), dim3(1024), 0, s, a);
    return check_hip(hipGetLastError(), "transpose launch");
}

// The rule, with times on MI355X in us at each order:
//  - Up to 1024, 32 x 64 tiles: enough workgroups for the chip (order 512:
//    2.7, 64 x 128 tiles 4.2; 1000: 5.7 against 6.4; at 1400 they lose, 11.2
//    against 9.4).
//  - Up to 4096 64 x 128 tiles, loads and stores through the caches: both
//    matrices stay in the 256 MB of the last one (order 2000: 19; 4096: 79,
//    93 non-temporal; 64 x 64 tiles in 8-byte accesses at 3001: 56, these 48).
//    64 x 64 tiles between 1409 and 1600 and between 2497 and 2560, where the
//    others come to little more than one or three workgroups for each CU
//    (order 1495, 288 of them: 16.5, 64 x 64 14.0; 1450 14.7, 13.5; 2505
//    38.4, 36.2; a little over two or four they stay ahead: 2101 27.9, 28.7;
//    2901 49.6, 51.6).
//  - Above, the same tiles, and only the stores non-temporal.  Rows on 64-byte
//    boundaries share no cache line between tiles, so from 4800 on their loads
//    are non-temporal too, with one workgroup at a time on a CU: order 32768
//    6005 (two workgroups 6150, only the stores non-temporal 6540), 16384 1490
//    (1520, 1630), 9000 529 (533, 598), 4808 150 (151 the stores alone).  Other
//    rows lose by non-temporal loads (10002 817, 787).  32 x 32 tiles without hints
//    take them in between, but by where the rows fall on the memory's channels:
//    18 % faster at 21050, 18 % slower at 24006.
//  - Up to 5200 the last-level cache holds much of what the tiles above leave:
//    B's stores stay in it, and its loads wait for A's stores (4450 110, with
//    B's non-temporal and its loads up front 121; 4590 121, 137; 4098 90.8,
//    90.7; 5178 190, 191; above, the others are the faster: 7004 363, 352).
//  - Odd orders and matrices off 16-byte boundaries: 64 x 64 tiles in 8-byte
//    accesses (order 12289 1091, 64 x 128 1251).
int launch_transpose(int order, double *A, double *B, hipStream_t s)
{
    TransposeArgs a{A, B, order, 0, 0, g_tr_mode < 0 ? 0 : g_tr_mode};
    const uintptr_t ptrs = (uintptr_t)A | (uintptr_t)B;
    const bool aligned = order % 2 == 0 && ptrs % 16 == 0;
    if (order > 4096 && !aligned) return launch_8b(a, s);
    const bool lines = order % 8 == 0 && ptrs % 64 == 0;
    const int nt = order <= 4096 ? NT_NONE : lines && order >= 4800 ? NT_ALL : order <= 5200 ? NT_A : NT_STORES;
    const bool few = (order > 1408 && order <= 1600) || (order > 2496 && order <= 2560);
    const int shape = order <= 1024 ? 3 : few ? 0 : 2;
    switch (g_tr_shape < 0 ? shape : g_tr_shape) {
    case 1: return launch_shape<128, 64>(a, nt, s);
    case 2: return launch_shape<64, 128>(a, nt, s);
    case 3: return launch_shape<32, 64>(a, nt, s);
    case 4: return launch_shape<128, 128, 1024>(a, nt, s);
    case 5: return launch_shape<32, 256>(a, nt, s);
    case 6: return launch_shape<256, 32>(a, nt, s);
    case 7: return launch_shape<64, 128, 512>(a, nt, s);
    case 8:
        if (aligned) return launch_2h(a, s);
        return launch_shape<64, 64>(a, nt, s);
    default: return launch_shape<64, 64>(a, nt, s);
    }
}

}  // namespace
}  // namespace prk

using namespace prk;

extern "C" {

int prk_transpose(int order, int tile, double *A, double *B)
{
    (void)tile;  // a tiling hint in the reference; results do not depend on it
    int rc = transpose_args(order, A, B);
    if (rc) return rc;
    return launch_transpose(order, A, B, nullptr);
}

int prk_transpose_ex(int order, double *A, double *B, void *stream)
{
    int rc = transpose_args(order, A, B);
    if (rc) return rc;
    return launch_transpose(order, A, B, (hipStream_t)stream);
}

int prk_set_transpose_variant(int shape, int mode)
{
    if (shape < -1 || shape > 8 || mode < -1 || mode > 2)
        return set_error(PRK_EINVAL, "transpose shape must be -1..8 and tile order -1..2");
    g_tr_shape = shape;
    g_tr_mode = mode;
    return PRK_OK;
}

int prk_transpose_init(int order, double *A, double *B, void *stream)
{
    int rc = transpose_args(order, A, B);
    if (rc) return rc;
    const long long nn = (long long)order * order;
    const unsigned blocks = (unsigned)std::min<long long>((nn + 255) / 256, 16384);
    hipLaunchKernelGGL(transpose_init_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, A, B, nn);
    return check_hip(hipGetLastError(), "transpose init launch");
}

int prk_transpose_run(int order, int iterations, double *A, double *B, void *stream_, double *avg_seconds)
{
    hipStream_t stream = (hipStream_t)stream_;
    int rc = transpose_args(order, A, B);
    if (rc) return rc;
    if (iterations < 1) return set_error(PRK_EINVAL, "iterations must be >= 1");
    hipEvent_t e0 = nullptr, e1 = nullptr;
    rc = check_hip(hipEventCreate(&e0), "event");
    if (!rc) rc = check_hip(hipEventCreate(&e1), "event");
    for (int it = 0; it <= iterations && !rc; ++it) {
        if (it == 1) rc = check_hip(hipEventRecord(e0, stream), "event record");
        if (!rc) rc = launch_transpose(order, A, B, stream);
    }
    if (!rc) rc = check_hip(hipEventRecord(e1, stream), "event record");
    if (!rc) rc = check_hip(hipEventSynchronize(e1), "event sync");
    float ms = 0.0f;
    if (!rc) rc = check_hip(hipEventElapsedTime(&ms, e0, e1), "event time");
    if (!rc && avg_seconds) *avg_seconds = (double)ms * 1e-3 / iterations;
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    return rc;
}

int prk_transpose_check(int order, int iterations, const double *B, double *abserr, void *stream_)
{
    hipStream_t stream = (hipStream_t)stream_;
    if (order < 1 || !B || !abserr || iterations < 0) return set_error(PRK_EINVAL, "bad transpose check arguments");
    double *ws = nullptr;
    int rc = check_workspace(&ws);
    if (rc) return rc;
    // the workspace is shared per device: one blocking check at a time
    static std::mutex check_mu;
    std::lock_guard<std::mutex> lock(check_mu);
    hipLaunchKernelGGL(transpose_check_kernel, dim3(kChkBlocks), dim3(kChkThreads), 0, stream, B, order, iterations,
                       ws);
    hipLaunchKernelGGL(transpose_check_final, dim3(1), dim3(kChkThreads), 0, stream, (const double *)ws,
                       ws + kChkBlocks);
    rc = check_hip(hipGetLastError(), "transpose check launch");
    if (rc) return rc;
    rc = check_hip(hipMemcpyAsync(abserr, ws + kChkBlocks, sizeof(double), hipMemcpyDeviceToHost, stream),
                   "transpose check copy");
    if (!rc) rc = check_hip(hipStreamSynchronize(stream), "transpose check sync");
    return rc;
}

}  // extern "C"
