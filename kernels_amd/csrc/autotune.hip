// Autotuner for the fused sweep: for a (pattern, radius, dtype, n) it times
// every candidate tiling on the device -- pipeline variant (depth 1..4 rows,
// temporal or non-temporal streams, and for the FP32/BF16 forms at R <= 3
// the register-window sweep), row-block height per wavefront and
// resident workgroups per CU -- and records the fastest in a process-wide
// table that plan_sweep() consults.  The table can be saved to and loaded
// from a text file.  Tiling never changes results, only speed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "prk_internal.hpp"
#include "sweep.hpp"

namespace prk {

namespace {

typedef std::tuple<int, int, int, int> Key;  // pattern, radius, dtype, n
std::mutex g_mu;
std::map<Key, prk_tuning> g_table;

const int kCandVariants[] = {1, 2, 4, 5, 6, 7, 8};
const int kCandWgs[] = {2, 3, 4};
const int kCandRows[] = {4, 6, 8, 12, 16, 24, 32, 48, 64};
// Row blocks beyond 32 only for R >= 4, where the 2R rows each block re-reads
// are a large share (star R=8 FP64: 48 rows 3 % faster than 24); below that
// they never won and would only lengthen the search.
constexpr int kTallRowsMinRadius = 4;
constexpr int kFinalists = 4;  // candidates timed again in the second stage

}  // namespace

// Measured defaults on MI355X: a 3-row non-temporal pipeline, and by size (a
// slab's turns of the chip counted by its own rows: by the whole grid's, FP32
// star R=3, n = 3001, one of eight slabs took 16.2 us instead of 8.0):
//  - Large whole grids take the row blocks and workgroups per CU that were
//    fastest at n = 16384 for each stencil and no slower anywhere above the
//    line: the HBM-bound sweeps want two workgroups per CU, those with longer
//    row steps as many as fit.  Slabs of as many points take them from R = 6
//    on (BF16 star R=8, n = 22000, half of the rows: 471 -> 414 us), the
//    others lose (FP32 star R=5 641 -> 670), as do those of fewer points (BF16
//    grid R=7, n = 18000, an eighth: 198 -> 236; not the FP64 star R=8, whose
//    height is the same, n = 13000, a quarter: 307 -> 270).  Against the rule
//    below for the middle: FP64 star R=8 1683 -> 1547 us; FP32 star R=5 797 ->
//    730, grid R=5 1010 -> 901; BF16 star R=1 404 -> 380, grid R=6 942 -> 853.
//    Stencils whose best at 16384 lost elsewhere keep the middle's (FP64 star
//    R=5, 8 rows and four workgroups: n = 10000 484 -> 465 us, but 11000 684
//    -> 723, 27000 4103 -> 4291).  The FP64 grids of R = 3..7 and the FP32
//    grid R=5, which are bound by their arithmetic, take theirs at every size
//    (FP64 grid R=5, n = 5000: 272 -> 213).
//  - In the middle one height per radius, growing so that the 2R halo rows
//    each block re-reads stay a small share, and two workgroups per CU (four
//    in BF16): what was fastest at 16384 loses up to 15 % between 2000 and
//    8000, where the turns of the chip count (FP64 star R=5, n = 6000: 203 us,
//    8 rows 220).
//  - An array of more than one and less than three (BF16: two) turns of two
//    workgroups per CU takes the height that fills its turns best, the last
//    one of which may be nearly empty, against the share of halo rows (FP64
//    grid R=8, n = 2600: 24 rows 175 us, 32 rows 156; the FP32 grid R=5, four
//    workgroups per CU, keeps its 32: n = 4800 76 us, 24 rows 90).  The
//    middle's height stays unless another fills the turns clearly better, a
//    lower one much better (FP64 star R=8, n = 2800: 24 rows 63.9 us, 12 rows,
//    by this measure 14 % better, 65.5), and where what lies past the last
//    whole turn is the last row of tiles alone, a short one: that costs
//    nothing (FP32 grid R=6, n = 7000, half of the rows, 1029 workgroups of 24
//    rows: 111 us, one and a half turns of 32 rows 135).  Stars and grids of R
//    <= 2 keep 8 rows.
//  - Where that is no more than one turn, the time is that of one wave going
//    down its h + 2R rows, and lower tiles are faster until the chip is full:
//    the lowest that give one workgroup per CU or two.  Two on a CU take 9/7
//    of the time per row of one; less where a row is one long chain of
//    arithmetic, which a second wave hides (medians over n = 300..3000: BF16
//    star R=3 1.19, FP32 grid R=4 1.14, BF16 grid R=3 1.13, star R=5 1.11,
//    FP32 grid R=6 1.03, FP64 grid R=8 1.07).  8 rows (BF16 12) -> the rule:
//    FP64 star R=2, n = 150 6.5 -> 3.5 us, n = 512 7.0 -> 4.2, n = 1000 8.3 ->
//    8.1, grid R=5, n = 512 14.6 -> 6.9; FP32 star R=2, n = 1000 7.9 -> 5.5;
//    BF16 grid R=3, n = 1000 15.1 -> 8.4, star R=2, n = 2000 10.5 -> 9.2.
prk_tuning heuristic_tuning(int pattern, int radius, int dtype, int n, int nrows)
{
    static const signed char kRows[3][2][kMaxRadius] = {
        {{8, 8, 12, 16, 24, 24, 12, 24}, {8, 8, 12, 24, 32, 48, 48, 24}},
        {{8, 8, 12, 12, 12, 24, 24, 24}, {8, 8, 12, 16, 32, 48, 48, 48}},
        {{8, 8, 12, 12, 12, 12, 24, 24}, {12, 12, 12, 32, 32, 32, 32, 32}}};
    static const signed char kWgs[3][2][kMaxRadius] = {
        {{2, 2, 2, 2, 2, 2, 4, 4}, {2, 2, 4, 4, 4, 4, 4, 2}},
        {{2, 2, 2, 2, 2, 2, 2, 2}, {2, 2, 2, 2, 4, 4, 4, 4}},
        {{2, 2, 2, 4, 4, 4, 4, 4}, {2, 3, 4, 4, 4, 4, 4, 4}}};
    const int d = dtype == F32 || dtype == BF16 ? dtype : F64, p = pattern == GRID ? 1 : 0;
    const int R = std::max(1, std::min(radius, kMaxRadius));
    prk_tuning t;
    t.variant = 5;
    t.order = 1;
    int rows = d == BF16 ? 12 : R <= 2 ? 8 : R == 3 ? 12 : R == 4 ? 16 : 24;
    t.wgs_per_cu = d == BF16 ? 4 : 2;
    // BF16 sweeps of R <= 3 lose by theirs below 16000 (grid R=2, n = 15000:
    // 332 -> 349 us; 18000 485 -> 461), the wider ones gain from 12000 on.
    const int line = d == F64 ? 8000 : d == BF16 && R <= 3 ? 16000 : 12000;
    const bool arithmetic = p == 1 && ((d == F64 && R >= 3 && R <= 7) || (d == F32 && R == 5));
    const int lanes = d == F64 ? 128 : d == F32 ? 256 : 512;  // columns of a strip
    constexpr long long kTurn = 512;  // workgroups
    const long long groups = std::max(1, ((n + lanes - 1) / lanes + kWavesPerBlock - 1) / kWavesPerBlock);
    auto tiles = [&](int h) { return groups * ((nrows + h - 1) / h); };
    const bool wgs_alone = d == F64 && p == 0 && R == 8 && n >= line && tiles(rows) >= 3 * kTurn;  // the middle's height
    const bool large = wgs_alone || ((long long)n * nrows >= (long long)line * line && (nrows == n || R >= 6));
    if (large || arithmetic) {
        rows = kRows[d][p][R - 1];
        t.wgs_per_cu = kWgs[d][p][R - 1];
    }
    // a second workgroup on a CU adds nothing to the FP64 grid R=8, and the
    // FP32 grid R=5 has four
    const long long lap = d == F64 && p == 1 && R == 8 ? kTurn / 2 : kTurn;
    const long long over = (tiles(rows) - 1) % lap + 1;  // workgroups of the last turn
    const bool short_turn = over <= groups && 3 * ((nrows - 1) % rows + 1) <= 2 * rows;
    if ((R >= 3 || d == BF16) && tiles(rows) > kTurn && tiles(rows) < (d == BF16 ? 2 : 3) * kTurn && !short_turn &&
        !(arithmetic && d == F32)) {
        static const int kHeights[] = {8, 12, 16, 24, 32};
        auto score = [&](int h) {  // share of its turns that the grid fills, times the share of rows that are no halo
            const long long t = tiles(h), turns = (t + lap - 1) / lap;
            return (double)t / (double)(turns * lap) * h / (h + 0.6 * R);
        };
        const int middle = rows;
        const double stay = score(middle);
        double best = 0.0;
        for (int h : kHeights) {
            if (d == BF16 && h > 16) break;  // its row steps are long: 24 and 32 rows lose however they fill
            if (!arithmetic && score(h) < (h < middle ? 1.25 : h > middle ? 1.05 : 1.0) * stay) continue;
            if (score(h) > best) {
                best = score(h);
                rows = h;
            }
        }
    }
    if (tiles(rows) <= kTurn) {
        auto lowest = [&](long long wgs) {  // height of at most that many workgroups, or of one tile per group
            const long long blocks = std::max(1ll, wgs / groups);
            return (int)((nrows + blocks - 1) / blocks);
        };
        const int h2 = lowest(kTurn), h1 = lowest(kTurn / 2);
        const bool chains = p == 1 && R >= (d == F64 ? 8 : d == F32 ? 5 : 4);
        int two = 9, one = 7;
        if (chains) two = 20, one = 19;
        else if (d == BF16 && R >= 2 && (p == 1 || (R >= 3 && R <= 5))) two = 12, one = 11;
        else if ((d == BF16 && p == 0 && R == 2) || (d == F32 && p == 1 && R == 4)) two = 8, one = 7;
        rows = std::min(rows, one * (h1 + 2 * R) <= two * (h2 + 2 * R) ? h1 : h2);
    }
    t.rows_per_wave = std::max(1, std::min(rows, n));
    t.gbs = 0.0;
    return t;
}

prk_tuning choose_tuning(int pattern, int radius, int dtype, int n, int nrows)
{
    {
        std::lock_guard<std::mutex> lock(g_mu);
        auto it = g_table.find(Key(pattern, radius, dtype, n));
        if (it != g_table.end()) return it->second;
        // nearest tuned size of the same stencil and dtype within a factor 1.5
        const prk_tuning *best = nullptr;
        double bestd = std::log(1.5);
        for (const auto &kv : g_table) {
            if (std::get<0>(kv.first) != pattern || std::get<1>(kv.first) != radius ||
                std::get<2>(kv.first) != dtype)
                continue;
            const double d = std::fabs(std::log((double)std::get<3>(kv.first) / n));
            if (d <= bestd) {
                bestd = d;
                best = &kv.second;
            }
        }
        if (best) {
            prk_tuning t = *best;
            t.rows_per_wave = std::max(1, std::min(t.rows_per_wave, n));
            return t;
        }
    }
    return heuristic_tuning(pattern, radius, dtype, n, nrows);
}

}  // namespace prk

using namespace prk;

extern "C" {

int prk_tuning_get(int pattern, int radius, int dtype, int n, prk_tuning *t)
{
    if (!t) return set_error(PRK_EINVAL, "null tuning");
    *t = choose_tuning(pattern, radius, dtype, n, n);
    return PRK_OK;
}

int prk_tuning_set(int pattern, int radius, int dtype, int n, const prk_tuning *t)
{
    if (!t || t->variant < 0 || t->variant >= kSweepVariants || t->rows_per_wave < 1 || t->wgs_per_cu < 0 ||
        t->wgs_per_cu > 16 || t->order < 0 || t->order > 7)
        return set_error(PRK_EINVAL, "bad tuning");
    std::lock_guard<std::mutex> lock(g_mu);
    g_table[Key(pattern, radius, dtype, n)] = *t;
    return PRK_OK;
}

int prk_tuning_clear(void)
{
    std::lock_guard<std::mutex> lock(g_mu);
    g_table.clear();
    return PRK_OK;
}

int prk_tuning_save(const char *path)
{
    FILE *f = path ? std::fopen(path, "w") : nullptr;
    if (!f) return set_error(PRK_EINVAL, "cannot write %s", path ? path : "(null)");
    std::lock_guard<std::mutex> lock(g_mu);
    std::fprintf(f, "# pattern radius dtype n variant rows_per_wave wgs_per_cu order gbs\n");
    for (const auto &kv : g_table)
        std::fprintf(f, "%d %d %d %d %d %d %d %d %.1f\n", std::get<0>(kv.first), std::get<1>(kv.first),
                     std::get<2>(kv.first), std::get<3>(kv.first), kv.second.variant, kv.second.rows_per_wave,
                     kv.second.wgs_per_cu, kv.second.order, kv.second.gbs);
    std::fclose(f);
    return PRK_OK;
}

int prk_tuning_load(const char *path)
{
    FILE *f = path ? std::fopen(path, "r") : nullptr;
    if (!f) return set_error(PRK_EINVAL, "cannot read %s", path ? path : "(null)");
    char line[256];
    int loaded = 0;
    while (std::fgets(line, sizeof line, f)) {
        if (line[0] == '#') continue;
        int p, r, d, n;
        prk_tuning t;
        if (std::sscanf(line, "%d %d %d %d %d %d %d %d %lf", &p, &r, &d, &n, &t.variant, &t.rows_per_wave,
                        &t.wgs_per_cu, &t.order, &t.gbs) == 9 &&
            prk_tuning_set(p, r, d, n, &t) == PRK_OK)
            ++loaded;
    }
    std::fclose(f);
    return loaded;
}

}  // extern "C"

namespace {

// The search on three caller grids of n rows at `pitch` (contents
// overwritten), on stream s; records the winner in the table.
int autotune_on(int pattern, int radius, int dtype, int n, long long pitch, void *b0, void *b1, void *out, int reps,
                hipStream_t s, prk_tuning *best)
{
    const size_t es = dtype_size(dtype);
    void *bufs[2] = {b0, b1};
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = check_hip(hipEventCreate(&e0), "autotune event");
    if (rc == PRK_OK) rc = check_hip(hipEventCreate(&e1), "autotune event");
    if (rc == PRK_OK) rc = prk_init(PRK_INIT_ANALYTIC, 0, dtype, n, pitch, b0, out, s);
    const double bytes_iter = 2.0 * es * (double)n * n + 2.0 * es * (double)(n - 2 * radius) * (n - 2 * radius);
    int cur = 0;
    // Time `r` sweeps of one tiling (after one untimed sweep); GB/s or < 0.
    auto time_tiling = [&](const prk_tuning &t, int r, double *gbs) -> int {
        SweepPlan p;
        int e = plan_sweep(pattern, radius, dtype, n, pitch, b0, b1, out, t.rows_per_wave, &p);
        if (e) return e;
        p.variant = t.variant;
        p.wgs_per_cu = t.wgs_per_cu;
        p.order = t.order;
        p.rows_per_wave = t.rows_per_wave;
        e = launch_sweep(p, bufs[cur], bufs[cur ^ 1], out, s);  // warm-up
        cur ^= 1;
        if (!e) e = check_hip(hipEventRecord(e0, s), "event");
        for (int k = 0; k < r && !e; ++k) {
            e = launch_sweep(p, bufs[cur], bufs[cur ^ 1], out, s);
            cur ^= 1;
        }
        if (!e) e = check_hip(hipEventRecord(e1, s), "event");
        if (!e) e = check_hip(hipEventSynchronize(e1), "event sync");
        float ms = 0.0f;
        if (!e) e = check_hip(hipEventElapsedTime(&ms, e0, e1), "event time");
        *gbs = (!e && ms > 0.0f) ? bytes_iter * r / (ms * 1e-3) / 1e9 : -1.0;
        return e;
    };
    // Stage 1: every candidate, `reps` sweeps each.
    std::vector<prk_tuning> cands;
    for (int v : kCandVariants) {
        // beyond the reference's radii one variant is built (see launch_pr);
        // 6 and 7 exist only where the register-window sweep applies
        if (radius > kRefMaxRadius && v != 4) continue;
        if (v >= 6 && !register_window_variant(v, radius, dtype)) continue;
        for (int w : kCandWgs) {
            for (int rows : kCandRows) {
                if (rc != PRK_OK) break;
                if (rows > n || (rows > 32 && radius < kTallRowsMinRadius)) continue;
                prk_tuning t{v, rows, w, 1, 0.0};
                rc = time_tiling(t, reps, &t.gbs);
                if (rc == PRK_OK && t.gbs > 0.0) cands.push_back(t);
            }
        }
    }
    // Stage 2: the fastest few again, over four times as many sweeps, twice
    // each in turn; a short sample alone picks noise as often as a tiling.
    std::sort(cands.begin(), cands.end(), [](const prk_tuning &a, const prk_tuning &b) { return a.gbs > b.gbs; });
    if (cands.size() > (size_t)kFinalists) cands.resize(kFinalists);
    std::vector<double> sum(cands.size(), 0.0);
    for (int pass = 0; pass < 2 && rc == PRK_OK; ++pass)
        for (size_t i = 0; i < cands.size() && rc == PRK_OK; ++i) {
            double g = 0.0;
            rc = time_tiling(cands[i], 4 * reps, &g);
            sum[i] += g;
        }
    prk_tuning top{};
    top.gbs = -1.0;
    for (size_t i = 0; i < cands.size() && rc == PRK_OK; ++i)
        if (sum[i] / 2 > top.gbs) {
            top = cands[i];
            top.gbs = sum[i] / 2;
        }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (rc) return rc;
    if (top.gbs <= 0.0) return set_error(PRK_EINVAL, "no tiling candidate fits n=%d", n);
    rc = prk_tuning_set(pattern, radius, dtype, n, &top);
    if (rc) return rc;
    if (best) *best = top;
    return PRK_OK;
}

}  // namespace

extern "C" {

int prk_autotune(int pattern, int radius, int dtype, int n, int reps, prk_tuning *best)
{
    if (reps < 1) return set_error(PRK_EINVAL, "reps must be >= 1");
    if (dtype != PRK_F64 && dtype != PRK_F32 && dtype != PRK_BF16) return set_error(PRK_EINVAL, "unknown dtype %d", dtype);
    if (n < 1) return set_error(PRK_EINVAL, "bad n %d", n);
    const size_t es = dtype_size(dtype);
    const long long pitch = ((long long)n * (long long)es + 15) / 16 * 16 / (long long)es;
    const size_t bytes = (size_t)n * (size_t)pitch * es;
    void *buf[3] = {nullptr, nullptr, nullptr};
    int rc = PRK_OK;
    for (int k = 0; k < 3 && rc == PRK_OK; ++k) rc = check_hip(hipMalloc(&buf[k], bytes), "autotune alloc");
    hipStream_t s = nullptr;
    if (rc == PRK_OK) rc = check_hip(hipStreamCreate(&s), "autotune stream");
    if (rc == PRK_OK) rc = autotune_on(pattern, radius, dtype, n, pitch, buf[0], buf[1], buf[2], reps, s, best);
    if (s) (void)hipStreamDestroy(s);
    for (void *b : buf)
        if (b) (void)hipFree(b);
    return rc;
}

int prk_autotune_buffers(int pattern, int radius, int dtype, int n, long long pitch, void *buf0, void *buf1,
                         void *out, int reps, void *stream, prk_tuning *best)
{
    if (reps < 1) return set_error(PRK_EINVAL, "reps must be >= 1");
    if (!buf0 || !buf1 || !out || buf0 == buf1 || buf0 == out || buf1 == out)
        return set_error(PRK_EINVAL, "autotune needs three separate grids");
    if (dtype != PRK_F64 && dtype != PRK_F32 && dtype != PRK_BF16) return set_error(PRK_EINVAL, "unknown dtype %d", dtype);
    if (n < 1 || pitch < n) return set_error(PRK_EINVAL, "bad grid (n=%d pitch=%lld)", n, pitch);
    return autotune_on(pattern, radius, dtype, n, pitch, buf0, buf1, out, reps, (hipStream_t)stream, best);
}

}  // extern "C"
