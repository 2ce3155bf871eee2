// Instantiation and launch of the sweep kernel for one storage dtype.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstdint>

#include "pass.hpp"
#include "prk_internal.hpp"
#include "sweep.hpp"

namespace prk {

// Loads a kernel's code on the current device, so that a later launch does not
// wait for it: asked for once per device (the answer takes 4 us).
template <auto kernel>
int load_code()
{
    static std::atomic<uint64_t> loaded{0};
    int dev = 0;
    int rc = check_hip(hipGetDevice(&dev), "hipGetDevice");
    const uint64_t bit = dev < 64 ? uint64_t(1) << dev : 0;
    if (rc || (loaded.load(std::memory_order_relaxed) & bit)) return rc;
    hipFuncAttributes attr;
    rc = check_hip(hipFuncGetAttributes(&attr, (const void *)kernel), "kernel load");
    if (!rc) loaded.fetch_or(bit, std::memory_order_relaxed);
    return rc;
}

template <int DT, int P, int R, bool FUSE, int MODE, int PF, int NT, bool RW = false>
int launch_one(const SweepPlan &p, const void *in, void *in_next, void *out, hipStream_t s)
{
    typedef SweepGeom<DT, R> G;
    SweepArgs a;
    a.in = in;
    a.in_next = in_next;
    a.out = out;
    a.pitch = p.pitch;
    a.n = p.n;
    a.span = p.span;
    a.rows_per_wave = p.rows_per_wave;
    a.nstrips = (p.n + G::SW - 1) / G::SW;
    a.ngroups = (a.nstrips + kWavesPerBlock - 1) / kWavesPerBlock;
    a.nrowblocks = (p.span.nrows + p.rows_per_wave - 1) / p.rows_per_wave;
    a.ntiles = a.ngroups * a.nrowblocks;
    a.pad_writable = p.pad_writable ? 1 : 0;
    a.order = p.order;
    unsigned blocks;
    if (p.order == 1) {
        a.chunk = 0;
        blocks = (unsigned)a.ntiles;
    } else if (p.order >= 3) {
        a.chunk = (a.ngroups + 7) / 8 * 8;
        blocks = (unsigned)a.chunk * (unsigned)a.nrowblocks;
    } else if (p.order == 2) {
        a.chunk = (a.ngroups + 7) / 8;
        blocks = 8u * (unsigned)a.chunk * (unsigned)a.nrowblocks;
    } else {
        a.chunk = (a.ntiles + 7) / 8;
        blocks = 8u * (unsigned)a.chunk;
    }
    // Extra dynamic LDS caps the workgroups resident per CU (occupancy knob).
    constexpr size_t kLdsPerCu = 160u * 1024u;
    const size_t lds_cap = p.wgs_per_cu > 0 ? kLdsPerCu / (unsigned)p.wgs_per_cu : 0;
    constexpr size_t lds_bytes = RW ? 0 : sweep_lds_bytes<DT, P, R>();
    size_t dyn = lds_cap > lds_bytes ? lds_cap - lds_bytes : 0;
    // The edge stash of the LDS-ring whole-vector sweeps lives at the start
    // of the dynamic LDS: in the occupancy padding when it is large enough,
    // else in kStashBytes added to it where that leaves the workgroups per CU
    // as they were (at most 8: 32 waves per CU), else not at all (edge waves
    // store their straddling vectors at once).  Its flush addresses
    // kStashRows rows of out from one resource, which must stay below the
    // out-of-range offset.
    a.stash = 0;
    if (!RW && vec_stores(MODE) &&
        (long long)kStashRows * p.pitch * (long long)sizeof(typename G::T) < (long long)kOOB) {
        if (dyn >= kStashBytes) {
            a.stash = 1;
        } else {
            const size_t wgs_before = std::min<size_t>(8, kLdsPerCu / std::max<size_t>(lds_bytes + dyn, 1));
            const size_t wgs_after = kLdsPerCu / (lds_bytes + kStashBytes);
            if (wgs_after >= wgs_before) {
                dyn = kStashBytes;
                a.stash = 1;
            }
        }
    }
    if (p.load_only) {
        if constexpr (RW) return load_code<sweep_rw_kernel<DT, P, R, FUSE, MODE, PF, NT>>();
        else return load_code<sweep_kernel<DT, P, R, FUSE, MODE, PF, NT>>();
    }
    if constexpr (RW)
        hipLaunchKernelGGL((sweep_rw_kernel<DT, P, R, FUSE, MODE, PF, NT>), dim3(blocks), dim3(kThreads), dyn, s, a);
    else
        hipLaunchKernelGGL((sweep_kernel<DT, P, R, FUSE, MODE, PF, NT>), dim3(blocks), dim3(kThreads), dyn, s, a);
    return check_hip(hipGetLastError(), "sweep launch");
}

// The fused sweep of aligned rows is the hot path: it is instantiated for
// every pipeline depth / cache policy the tuner chooses from (radii beyond
// the reference's 5: one, two rows in flight with non-temporal stores).  Four
// rows in flight (variant 8) made FP64 star R=2 at n=30000 1.3-1.8 % faster
// than three at 6- and 8-row blocks on MI355X (alternating runs on one box),
// and slower at 12 and 16 rows.
template <int DT, int P, int R>
int launch_pr(const SweepPlan &p, const void *in, void *in_next, void *out, hipStream_t s)
{
    const bool fuse = in_next != nullptr;
    if (fuse && p.mode == MODE_VEC) {
        const int v = p.variant;
        if (v < 0 || v >= kSweepVariants) return set_error(PRK_EINVAL, "unknown sweep variant %d", v);
        if constexpr (R > kRefMaxRadius) {
            return launch_one<DT, P, R, true, MODE_VEC, 2, 1>(p, in, in_next, out, s);
        } else {
            if constexpr (reg_window_ok<DT, P, R>()) {
                if (v == 6) return launch_one<DT, P, R, true, MODE_VEC, 2, 1, true>(p, in, in_next, out, s);
                if (v == 7) return launch_one<DT, P, R, true, MODE_VEC, 3, 1, true>(p, in, in_next, out, s);
            }
            switch (v) {
            case 0: return launch_one<DT, P, R, true, MODE_VEC, 1, 0>(p, in, in_next, out, s);
            case 1: return launch_one<DT, P, R, true, MODE_VEC, 2, 0>(p, in, in_next, out, s);
            case 2: return launch_one<DT, P, R, true, MODE_VEC, 3, 0>(p, in, in_next, out, s);
            case 3: return launch_one<DT, P, R, true, MODE_VEC, 1, 1>(p, in, in_next, out, s);
            case 4: case 6: return launch_one<DT, P, R, true, MODE_VEC, 2, 1>(p, in, in_next, out, s);
            case 8: return launch_one<DT, P, R, true, MODE_VEC, 4, 1>(p, in, in_next, out, s);
            default: return launch_one<DT, P, R, true, MODE_VEC, 3, 1>(p, in, in_next, out, s);
            }
        }
    }
    // The other forms take the rows in flight and the non-temporal stores of the
    // default fused sweep where the call's arrays are past the caches or lie in
    // the L2s together; between (`cached`) their stores go through the caches.
    // Measured on MI355X, us, FP64 star R=2 unless said otherwise, in a loop on
    // one grid / on three in turn:
    //  - unfused, then in += 1: n = 1200 16.7 / 17.2, non-temporal 18.2 / 19.7;
    //    n = 2300 40.2 / 40.4, 40.2 / 40.8; n = 3000 - / 75.6, - / 63.6 (three
    //    pairs no longer fit the last-level cache); n = 700 10.1 / 10.6, 9.4 /
    //    10.6; n = 16384 1146, 1071.
    //  - fused, ragged rows: FP64 inside the last-level cache takes element
    //    stores (n = 2301 31.0, vectors 32.3, non-temporal ones 33.3; n = 4001
    //    102, 91.8, 85.9; three grids in turn lose 4 to 14 % by it between 2301
    //    and 3201, and are still as fast as before the vectors), FP32 grid R=4
    //    vectors (n = 4001 50.2, non-temporal 60.7, element stores 49.1; star
    //    R=4, n = 1801 14.2, 15.3, 15.7), so does BF16 (stencils' mean at 4001
    //    7 % over non-temporal).  The widest grids are bound by their
    //    arithmetic, and the vectors' registers cost more than their stores
    //    save (FP64 grid R=8, n = 6501 809, vectors 849; FP32 grid R=8, n = 8001
    //    402, 444).
    //  - fused, rows off 16 bytes: FP64 inside the last-level cache by element
    //    (n = 3101 56.4, vectors 57.9, non-temporal 62.3).
    constexpr int PF = R > kRefMaxRadius ? 2 : 3;
    const long long bytes = (fuse ? 3 : 2) * (long long)p.span.nrows * p.pitch * (long long)sizeof(typename SweepGeom<DT, R>::T);
    const bool fits = bytes <= kLastLevelCache;
    const bool cached = fuse ? fits && bytes > (20ll << 20) : bytes > (12ll << 20) && bytes <= kLastLevelCache / 3;
    if (fuse) {
        if (p.mode == MODE_RAGGED) {
            constexpr bool wide = P == GRID && R >= (DT == F64 ? 8 : DT == F32 ? 6 : kMaxRadius + 1);
            if constexpr (DT == F64) {
                if (wide || fits) return launch_one<DT, P, R, true, MODE_LOADS, kPrefetch, 0>(p, in, in_next, out, s);
            } else if constexpr (wide) {
                return launch_one<DT, P, R, true, MODE_LOADS, kPrefetch, 0>(p, in, in_next, out, s);
            } else {
                if (cached) return launch_one<DT, P, R, true, MODE_RAGGED, PF, 0>(p, in, in_next, out, s);
            }
            if constexpr (!wide) return launch_one<DT, P, R, true, MODE_RAGGED, PF, 1>(p, in, in_next, out, s);
        }
        if (p.mode == MODE_DWORD && !(DT == F64 && fits))
            return launch_one<DT, P, R, true, MODE_DWORD, PF, 1>(p, in, in_next, out, s);
        return launch_one<DT, P, R, true, MODE_ELEM, kPrefetch, 0>(p, in, in_next, out, s);
    }
    if (p.mode == MODE_ELEM) return launch_one<DT, P, R, false, MODE_ELEM, kPrefetch, 0>(p, in, in_next, out, s);
    if (cached) {
        if (p.mode == MODE_VEC) return launch_one<DT, P, R, false, MODE_VEC, kPrefetch, 0>(p, in, in_next, out, s);
        if (p.mode == MODE_RAGGED) return launch_one<DT, P, R, false, MODE_RAGGED, kPrefetch, 0>(p, in, in_next, out, s);
        return launch_one<DT, P, R, false, MODE_DWORD, kPrefetch, 0>(p, in, in_next, out, s);
    }
    if (p.mode == MODE_VEC) return launch_one<DT, P, R, false, MODE_VEC, PF, 1>(p, in, in_next, out, s);
    if (p.mode == MODE_RAGGED) return launch_one<DT, P, R, false, MODE_RAGGED, PF, 1>(p, in, in_next, out, s);
    return launch_one<DT, P, R, false, MODE_DWORD, PF, 1>(p, in, in_next, out, s);
}

template <int DT>
int launch_dtype(const SweepPlan &p, const void *in, void *in_next, void *out, hipStream_t s)
{
    if (p.pattern == STAR) {
        switch (p.radius) {
        case 1: return launch_pr<DT, STAR, 1>(p, in, in_next, out, s);
        case 2: return launch_pr<DT, STAR, 2>(p, in, in_next, out, s);
        case 3: return launch_pr<DT, STAR, 3>(p, in, in_next, out, s);
        case 4: return launch_pr<DT, STAR, 4>(p, in, in_next, out, s);
        case 5: return launch_pr<DT, STAR, 5>(p, in, in_next, out, s);
        case 6: return launch_pr<DT, STAR, 6>(p, in, in_next, out, s);
        case 7: return launch_pr<DT, STAR, 7>(p, in, in_next, out, s);
        case 8: return launch_pr<DT, STAR, 8>(p, in, in_next, out, s);
        }
    } else {
        switch (p.radius) {
        case 1: return launch_pr<DT, GRID, 1>(p, in, in_next, out, s);
        case 2: return launch_pr<DT, GRID, 2>(p, in, in_next, out, s);
        case 3: return launch_pr<DT, GRID, 3>(p, in, in_next, out, s);
        case 4: return launch_pr<DT, GRID, 4>(p, in, in_next, out, s);
        case 5: return launch_pr<DT, GRID, 5>(p, in, in_next, out, s);
        case 6: return launch_pr<DT, GRID, 6>(p, in, in_next, out, s);
        case 7: return launch_pr<DT, GRID, 7>(p, in, in_next, out, s);
        case 8: return launch_pr<DT, GRID, 8>(p, in, in_next, out, s);
        }
    }
    return set_error(PRK_ENOSTENCIL, "no stencil for pattern %d radius %d", p.pattern, p.radius);
}

// One pass of `sweeps` sweeps (pass.hpp), where pass_built.  With sweeps == 0
// nothing is launched: the kernel's code is loaded, so that a later launch
// does not wait for it.
template <int DT, int P, int R>
int launch_pass_pr(const SweepPlan &p, int sweeps, bool any, const void *in, void *in_next, void *out, hipStream_t s)
{
    if constexpr (pass_ok<DT, P, R>()) {
        constexpr int V = SweepGeom<DT, R>::V;
        PassArgs a;
        a.in = in;
        a.in_next = in_next;
        a.out = out;
        a.pitch = p.pitch;
        a.n = p.n;
        a.nstrips = (p.n + 64 * V - 1) / (64 * V);
        a.rows = pass_rows<DT, P, R>();
        a.sweeps = sweeps;
        a.any = any;
        const int per_block = a.rows * kWavesPerBlock;
        const unsigned blocks = (unsigned)a.nstrips * (unsigned)((p.n + per_block - 1) / per_block);
        const auto kernel =
            p.mode == MODE_VEC || p.mode == MODE_RAGGED ? pass_kernel<DT, P, R, true> : pass_kernel<DT, P, R, false>;
        if (sweeps == 0) {
            const int rc = load_code<pass_kernel<DT, P, R, true>>();
            return rc ? rc : load_code<pass_kernel<DT, P, R, false>>();
        }
        hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kThreads), 0, s, a);
        return check_hip(hipGetLastError(), "pass launch");
    } else {
        return set_error(PRK_EINVAL, "no pass kernel for pattern %d radius %d", P, R);
    }
}

template <int DT>
int launch_pass_dtype(const SweepPlan &p, int sweeps, bool any, const void *in, void *in_next, void *out, hipStream_t s)
{
    switch (p.pattern * 8 + p.radius) {
    case 1: return launch_pass_pr<DT, STAR, 1>(p, sweeps, any, in, in_next, out, s);
    case 2: return launch_pass_pr<DT, STAR, 2>(p, sweeps, any, in, in_next, out, s);
    case 3: return launch_pass_pr<DT, STAR, 3>(p, sweeps, any, in, in_next, out, s);
    case 4: return launch_pass_pr<DT, STAR, 4>(p, sweeps, any, in, in_next, out, s);
    case 5: return launch_pass_pr<DT, STAR, 5>(p, sweeps, any, in, in_next, out, s);
    case 6: return launch_pass_pr<DT, STAR, 6>(p, sweeps, any, in, in_next, out, s);
    case 7: return launch_pass_pr<DT, STAR, 7>(p, sweeps, any, in, in_next, out, s);
    case 8: return launch_pass_pr<DT, STAR, 8>(p, sweeps, any, in, in_next, out, s);
    case 9: return launch_pass_pr<DT, GRID, 1>(p, sweeps, any, in, in_next, out, s);
    case 10: return launch_pass_pr<DT, GRID, 2>(p, sweeps, any, in, in_next, out, s);
    case 11: return launch_pass_pr<DT, GRID, 3>(p, sweeps, any, in, in_next, out, s);
    case 12: return launch_pass_pr<DT, GRID, 4>(p, sweeps, any, in, in_next, out, s);
    case 13: return launch_pass_pr<DT, GRID, 5>(p, sweeps, any, in, in_next, out, s);
    case 14: return launch_pass_pr<DT, GRID, 6>(p, sweeps, any, in, in_next, out, s);
    case 15: return launch_pass_pr<DT, GRID, 7>(p, sweeps, any, in, in_next, out, s);
    case 16: return launch_pass_pr<DT, GRID, 8>(p, sweeps, any, in, in_next, out, s);
    }
    return set_error(PRK_ENOSTENCIL, "no stencil for pattern %d radius %d", p.pattern, p.radius);
}

}  // namespace prk
