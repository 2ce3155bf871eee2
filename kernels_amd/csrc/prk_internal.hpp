// Internal declarations shared by the translation units of libprkstencil.so.
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "prk_common.hpp"
#include "prk_stencil.h"

namespace prk {

// Thread-local last-error message behind prk_last_error().
int set_error(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));
void clear_error();
int check_hip(hipError_t e, const char *what);

// Geometry of one sweep launch.
struct SweepPlan {
    int dtype, pattern, radius, n;  // n: columns (and rows, for a whole grid)
    RowSpan span;                   // rows read and written (prk_common.hpp)
    long long pitch;
    int rows_per_wave;
    int mode;           // MODE_* (sweep.hpp)
    int variant;        // pipeline depth / cache policy of the fused vector sweep
    bool pad_writable;  // columns n..pitch-1 may be overwritten
    int order;          // workgroup -> tile order (sweep.hpp tile_of)
    int wgs_per_cu;     // occupancy cap, 0 = none
    bool load_only = false;  // launch_sweep loads the kernel's code and launches nothing
};

// Number of fused-sweep variants: 0..5 the LDS-ring sweep (pipeline depth
// 1..3 x temporal / non-temporal), 6 and 7 the register-window sweep of the
// FP32/BF16 forms at R <= 3 (depth 2 and 3, non-temporal; elsewhere they run
// as 4 and 5), 8 the LDS-ring sweep at depth 4, non-temporal.
constexpr int kSweepVariants = 9;
inline bool register_window_variant(int variant, int radius, int dtype)
{
    return (variant == 6 || variant == 7) && dtype != F64 && radius <= 3;
}

// The L1 norm's first pass leaves one double-double partial per block, at
// most kNormBlocks of them, in a device buffer of kNormPartialsBytes.
constexpr int kNormBlocks = 1024;
constexpr size_t kNormPartialsBytes = 2 * sizeof(double) * kNormBlocks;

// L1 norm into a device double, enqueued on s, with the caller's partials
// buffer (kNormPartialsBytes of device memory, in use until the norm is done).
int l1norm_async(int dtype, int n, long long pitch, int radius, const void *out, double *d_result, void *partials,
                 hipStream_t s);

// Tiling a sweep of this shape uses: tuned entry, nearest tuned size, or the
// built-in default (autotune.hip).  nrows: rows of the array, n of a whole grid.
prk_tuning choose_tuning(int pattern, int radius, int dtype, int n, int nrows);
prk_tuning heuristic_tuning(int pattern, int radius, int dtype, int n, int nrows);

// Fills the launch geometry; rows_per_wave <= 0 picks automatically, for an
// array of nrows rows (0: a whole grid).
int plan_sweep(int pattern, int radius, int dtype, int n, long long pitch, const void *in,
               const void *in_next, const void *out, int rows_per_wave, SweepPlan *plan, int nrows = 0);

// Enqueue one sweep (in_next == nullptr: unfused).
int launch_sweep(const SweepPlan &p, const void *in, void *in_next, void *out, hipStream_t s);
int launch_sweep_f64(const SweepPlan &p, const void *in, void *in_next, void *out, hipStream_t s);
int launch_sweep_f32(const SweepPlan &p, const void *in, void *in_next, void *out, hipStream_t s);
int launch_sweep_bf16(const SweepPlan &p, const void *in, void *in_next, void *out, hipStream_t s);

// Enqueue one pass of `sweeps` sweeps over a whole grid (pass.hpp): in_next
// gets in after that many refreshes.  Only where pass_built.  With sweeps == 0
// the kernel's code is loaded and nothing launched.
int launch_pass(const SweepPlan &p, int sweeps, bool any, const void *in, void *in_next, void *out, hipStream_t s);
int launch_pass_f64(const SweepPlan &p, int sweeps, bool any, const void *in, void *in_next, void *out, hipStream_t s);
int launch_pass_f32(const SweepPlan &p, int sweeps, bool any, const void *in, void *in_next, void *out, hipStream_t s);
int launch_pass_bf16(const SweepPlan &p, int sweeps, bool any, const void *in, void *in_next, void *out, hipStream_t s);

constexpr long long kLastLevelCache = 256ll << 20, kL2s = 32ll << 20;  // bytes (the L2s of eight dies)

// Sweeps of one pass at most: keeps a launch's time and the loss from an
// interrupted one bounded (star R=2 FP64 at n = 30000: 256 sweeps take about
// 0.1 s).
constexpr int kMaxPassSweeps = 256;

}  // namespace prk
