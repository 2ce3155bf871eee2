"""The work that users of this library have it do, as cases to be timed.

Kinds of cases, each through the package's public entry points:

  solve      the reference driver's whole path on one grid: initial values,
             iterations + 1 sweeps, L1 norm (init, run, l1norm)
  sweep      one fused sweep (out += S(in), in_next = in + 1) inside a
             program's own loop
  operators  the drop-in pair of the reference's loop, stencil then add, on
             dense FP64 grids
  slab       the fused sweep of one GPU's rows of a row-strip decomposition
  transpose  one iteration B += A^T, A += 1
  batch      many uneven solves in one batch, replayed: norms of all, grids
             of a few

Grids hold seeded uniform values in (-1, 1), the distribution the library's
seeded initial values have.
"""
from __future__ import annotations

import math
import random

import torch

import kernels_amd as K
from kernels_amd.batch import Batch

STAR, GRID = "star", "grid"
PATTERN = {STAR: 0, GRID: 1}
DTYPE = {"f64": 0, "f32": 1, "bf16": 2}
TORCH = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16}
SIZE = {"f64": 8, "f32": 4, "bf16": 2}
DEVICE = "cuda"


def listed() -> list[dict]:
    return [
        # The smallest call: a drop-in operator and its refresh on a grid of
        # a few tens of KiB, where launches are all the time there is.
        dict(name="operators_star1_n96", kind="operators", pattern=STAR, radius=1, n=96),
        # The drop-in operators as the reference's driver calls them, dense
        # rows of an odd length.
        dict(name="operators_star2_n4001", kind="operators", pattern=STAR, radius=2, n=4001),
        # The reference's own default-sized run: n=1000, 10 iterations.
        dict(name="solve_star2_f64_n1000", kind="solve", pattern=STAR, radius=2, dtype="f64", n=1000, iterations=10),
        # The headline run: n=30000, 100 iterations, the largest case.
        dict(name="solve_star2_f64_n30000", kind="solve", pattern=STAR, radius=2, dtype="f64", n=30000,
             iterations=100),
        # The radius/precision sweep's full-square stencil in FP32 storage.
        dict(name="solve_grid3_f32_n16384", kind="solve", pattern=GRID, radius=3, dtype="f32", n=16384,
             iterations=50),
        # One sweep of a program that does its own work between sweeps: the
        # half-width storage type at a middle radius.
        dict(name="sweep_star3_bf16_n16384", kind="sweep", pattern=STAR, radius=3, dtype="bf16", n=16384),
        # One sweep of a ragged grid (rows not a whole number of vectors).
        dict(name="sweep_star1_f32_n9999", kind="sweep", pattern=STAR, radius=1, dtype="f32", n=9999),
        # The reference's widest operator, 110 taps.
        dict(name="sweep_grid5_f64_n16384", kind="sweep", pattern=GRID, radius=5, dtype="f64", n=16384),
        # One GPU's share of the headline grid on eight GPUs.
        dict(name="slab_star2_f64_n30000", kind="slab", pattern=STAR, radius=2, dtype="f64", n=30000, parts=8,
             part=3),
        # The suite's other bandwidth kernel at its benchmark size, and a
        # small odd order.
        dict(name="transpose_32768", kind="transpose", n=32768),
        dict(name="transpose_1999", kind="transpose", n=1999),
        # A parameter study: uneven grids n in [64, 2048], every radius 1..4,
        # both patterns, 1..50 iterations, a third of them in FP64.
        dict(name="batch_512", kind="batch", count=512, n_lo=64, n_hi=2048, iters_hi=50, f64_every=3),
    ]


def _log_uniform(rng: random.Random, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> dict:
    kind = rng.choices(("solve", "sweep", "operators", "slab", "transpose", "batch"), (4, 3, 2, 1, 1, 2))[0]
    pattern, radius = rng.choice((STAR, GRID)), rng.randint(1, 5)
    dtype = rng.choices(("f64", "f32", "bf16"), (4, 4, 2))[0]
    if kind == "solve":
        return dict(kind=kind, pattern=pattern, radius=radius, dtype=dtype, n=_log_uniform(rng, 64, 16384),
                    iterations=_log_uniform(rng, 1, 50))
    if kind == "sweep":
        # the stencils beyond the reference's radii too
        return dict(kind=kind, pattern=pattern, radius=rng.randint(1, 8), dtype=dtype,
                    n=_log_uniform(rng, 64, 24000))
    if kind == "operators":
        return dict(kind=kind, pattern=pattern, radius=radius, n=_log_uniform(rng, 64, 16384))
    if kind == "slab":
        parts = rng.choice((2, 4, 8))
        return dict(kind=kind, pattern=pattern, radius=radius, dtype=dtype, n=_log_uniform(rng, 512, 30000),
                    parts=parts, part=rng.randrange(parts))
    if kind == "transpose":
        return dict(kind=kind, n=_log_uniform(rng, 64, 24000))
    lo = _log_uniform(rng, 32, 256)
    return dict(kind=kind, count=_log_uniform(rng, 16, 512), n_lo=lo, n_hi=_log_uniform(rng, 2 * lo, 2048),
                iters_hi=_log_uniform(rng, 2, 50), f64_every=rng.randint(2, 6))


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------
def _uniform(rows: int, cols: int, dtype: str, seed: int) -> torch.Tensor:
    """rows x cols values in (-1, 1), from the seed alone."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    x = torch.rand((rows, cols), generator=gen, device=DEVICE, dtype=torch.float64 if dtype == "f64" else torch.float32)
    return x.mul_(2.0).sub_(1.0).to(TORCH[dtype])


def _matrix(n: int, seed: int) -> torch.Tensor:
    """n x n whole numbers in FP64, as the transpose's own matrices hold."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    return torch.randint(0, 1 << 30, (n, n), generator=gen, device=DEVICE, dtype=torch.int32).to(torch.float64)


def _slab_rows(case: dict) -> tuple[int, int]:
    """First row and number of rows of the slab."""
    n, parts, part = case["n"], case["parts"], case["part"]
    lo, hi = n * part // parts, n * (part + 1) // parts
    return lo, hi - lo


def _slab_halo(case: dict) -> tuple[int, int]:
    row0, rows = _slab_rows(case)
    return min(case["radius"], row0), min(case["radius"], case["n"] - row0 - rows)


def _batch_solves(case: dict, seed: int) -> list[tuple]:
    """(pattern, radius, dtype, n, iterations, init, seed) of each solve.  The
    mix belongs to the case; the seed gives the grids' values."""
    rng = random.Random(case["count"] * 1000003 + case["n_lo"] * 1009 + case["n_hi"])
    out = []
    for k in range(case["count"]):
        n = _log_uniform(rng, case["n_lo"], case["n_hi"])
        out.append((rng.randint(0, 1), rng.randint(1, 4), 0 if k % case["f64_every"] == 0 else 1, n,
                    rng.randint(1, case["iters_hi"]), K.INIT_SEEDED, seed * 65537 + k))
    return out


_FETCHED = 4  # grids of a batch that are copied back


def _fetched(case: dict) -> list[int]:
    return [case["count"] * k // _FETCHED for k in range(_FETCHED)]


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "batch":
        return dict(case=case, batch=Batch(_batch_solves(case, seed)))
    n = case["n"]
    if kind == "transpose":
        return dict(case=case, A=_matrix(n, 2 * seed), B=_matrix(n, 2 * seed + 1))
    if kind == "operators":
        return dict(case=case, inp=_uniform(n, n, "f64", 2 * seed), out=_uniform(n, n, "f64", 2 * seed + 1))
    dt = DTYPE[case["dtype"]]
    if kind == "slab":
        row0, rows = _slab_rows(case)
        b = [K.alloc_slab(n, case["radius"], row0, rows, dt) for _ in range(3)]
    else:
        b = [K.alloc_grid(n, dt) for _ in range(3)]
    if kind != "solve":  # a solve sets its own initial values
        b[0].copy_(_uniform(b[0].shape[0], n, case["dtype"], 2 * seed))
        b[1].zero_()  # a slab's halo rows are not written
        b[2].copy_(_uniform(b[2].shape[0], n, case["dtype"], 2 * seed + 1))
    return dict(case=case, seed=seed, inp=b[0], nxt=b[1], out=b[2])


def run(state: dict):
    c = state["case"]
    kind = c["kind"]
    if kind == "batch":
        b = state["batch"]
        b.run(torch.cuda.current_stream().cuda_stream)
        norms = b.wait()
        return {"norms": norms, "grids": [b.output(i) for i in _fetched(c)]}
    if kind == "transpose":
        K.transpose(state["A"], state["B"])
        return {"A": state["A"], "B": state["B"]}
    pattern, radius = PATTERN[c["pattern"]], c["radius"]
    inp, out = state["inp"], state["out"]
    if kind == "operators":
        K.stencil(f"{c['pattern']}{radius}", c["n"], 32, inp, out)
        K.add(c["n"], 32, inp)
        return {"in": inp, "out": out}
    dt, nxt = DTYPE[c["dtype"]], state["nxt"]
    if kind == "sweep":
        K.sweep(pattern, radius, dt, inp, nxt, out)
        return {"in": nxt, "out": out}
    if kind == "slab":
        row0, rows = _slab_rows(c)
        K.sweep_slab(pattern, radius, dt, c["n"], row0, rows, inp, nxt, out)
        return {"in": nxt, "out": out}
    K.init(K.INIT_SEEDED, state["seed"], dt, inp, out)
    final, _ = K.run(pattern, radius, dt, c["iterations"], inp, nxt, out)
    norm = K.l1norm(dt, radius, out)
    return {"in": (inp, nxt)[final], "out": out, "norm": norm}


# --------------------------------------------------------------------------
# What a pass cannot do without: each input read once, each output written
# once, two operations per nonzero weight and point and one for the refresh.
# --------------------------------------------------------------------------
def _taps(pattern: str, radius: int) -> int:
    return 4 * radius if pattern == STAR else 4 * radius * radius + 2 * radius


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "batch":
        nbytes = flops = 0
        for pattern, radius, dtype, n, iters, _, _ in _batch_solves(case, 0):
            nbytes += 2 * (8, 4)[dtype] * n * n
            flops += (iters + 1) * (2 * _taps((STAR, GRID)[pattern], radius) + 1) * n * n
        return {"bytes": nbytes, "flops": flops}
    n = case["n"]
    if kind == "transpose":
        return {"bytes": 32 * n * n, "flops": 2 * n * n}
    radius = case["radius"]
    per = 2 * _taps(case["pattern"], radius) + 1
    inner = (n - 2 * radius) ** 2
    if kind == "operators":
        return {"bytes": 16 * n * n + 16 * inner, "flops": per * n * n}
    s = SIZE[case["dtype"]]
    if kind == "solve":
        return {"bytes": 2 * s * n * n, "flops": (case["iterations"] + 1) * per * n * n}
    if kind == "slab":
        row0, rows = _slab_rows(case)
        return {"bytes": K.slab_bytes_per_iter(n, radius, DTYPE[case["dtype"]], row0, rows), "flops": per * n * rows}
    return {"bytes": 2 * s * n * n + 2 * s * inner, "flops": per * n * n}


# --------------------------------------------------------------------------
# The same results in 64 bits, in plain torch
# --------------------------------------------------------------------------
def _weight(pattern: str, radius: int, a: int, b: int) -> float:
    """Weight of the point a columns and b rows away."""
    if a == 0 and b == 0:
        return 0.0
    sign = lambda x: 1.0 if x > 0 else -1.0  # noqa: E731
    if pattern == STAR:
        if a == 0 or b == 0:
            return sign(a + b) / (2.0 * abs(a + b) * radius)
        return 0.0
    m = max(abs(a), abs(b))
    if abs(a) < m:
        return sign(b) / (4 * m * (2 * m - 1) * radius)
    if abs(b) < m:
        return sign(a) / (4 * m * (2 * m - 1) * radius)
    return sign(a) / (4 * m * radius) if a == b else 0.0


def _stencil(x: torch.Tensor, pattern: str, radius: int) -> torch.Tensor:
    """S(x) on the points that have all their neighbours, in FP64."""
    rows, cols = x.shape
    s = torch.zeros((rows - 2 * radius, cols - 2 * radius), dtype=torch.float64, device=x.device)
    for a in range(-radius, radius + 1):
        for b in range(-radius, radius + 1):
            w = _weight(pattern, radius, a, b)
            if w != 0.0:
                s.add_(x[radius + b:rows - radius + b, radius + a:cols - radius + a], alpha=w)
    return s


def _seeded(n: int, seed: int, dtype: str) -> torch.Tensor:
    """2u - 1, u the top 53 bits of SplitMix64(seed, index) / 2^53, rounded
    once to the storage type, as FP64."""
    def signed(v: int) -> int:
        v &= (1 << 64) - 1
        return v - (1 << 64) if v >> 63 else v

    def shifted(z: torch.Tensor, k: int) -> torch.Tensor:  # logical right shift
        return (z >> k).bitwise_and_((1 << (64 - k)) - 1)

    out = torch.empty((n, n), dtype=torch.float64, device=DEVICE)
    step = max(1, (1 << 28) // n)
    for r in range(0, n, step):
        rows = min(step, n - r)
        z = torch.arange(r * n + 1, (r + rows) * n + 1, dtype=torch.int64, device=DEVICE)
        z.mul_(signed(0x9E3779B97F4A7C15)).add_(signed(seed))
        z.bitwise_xor_(shifted(z, 30)).mul_(signed(0xBF58476D1CE4E5B9))
        z.bitwise_xor_(shifted(z, 27)).mul_(signed(0x94D049BB133111EB))
        z.bitwise_xor_(shifted(z, 31))
        u = shifted(z, 11).to(torch.float64).mul_(2.0 ** -53)
        out[r:r + rows] = u.mul_(2.0).sub_(1.0).view(rows, n)
    return out if dtype == "f64" else out.to(TORCH[dtype]).to(torch.float64)


def _solved(pattern: str, radius: int, dtype: str, n: int, iterations: int, seed: int):
    """(out, in, norm) of a solve.  The weights sum to zero, so S(in + k) is
    S(in) and out is iterations + 1 times that."""
    x = _seeded(n, seed, dtype)
    inner = _stencil(x, pattern, radius).mul_(iterations + 1.0)
    norm = float(inner.abs().sum()) / (n - 2 * radius) ** 2
    out = torch.zeros((n, n), dtype=torch.float64, device=DEVICE)
    out[radius:n - radius, radius:n - radius] = inner
    return out, x.add_(iterations + 1.0), norm


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "batch":
        norms, grids, wanted = [], [], set(_fetched(case))
        for k, (pattern, radius, dtype, n, iters, _, s) in enumerate(_batch_solves(case, seed)):
            out, _, norm = _solved((STAR, GRID)[pattern], radius, ("f64", "f32")[dtype], n, iters, s)
            norms.append(norm)
            if k in wanted:
                grids.append(out)
        return {"norms": torch.tensor(norms, dtype=torch.float64), "grids": grids}
    n = case["n"]
    if kind == "transpose":
        A = _matrix(n, 2 * seed)
        return {"B": _matrix(n, 2 * seed + 1).add_(A.t()), "A": A.add_(1.0)}
    radius, pattern = case["radius"], case["pattern"]
    if kind == "solve":
        if case["dtype"] == "bf16":  # the rounding of in + k decides the result
            return None
        out, fin, norm = _solved(pattern, radius, case["dtype"], n, case["iterations"], seed)
        return {"in": fin, "out": out, "norm": norm}
    dtype = case.get("dtype", "f64")
    rows, top, bot = n, 0, 0
    if kind == "slab":
        rows = _slab_rows(case)[1]
        top, bot = _slab_halo(case)
        rows += top + bot
    x = _uniform(rows, n, dtype, 2 * seed).to(torch.float64)
    out = _uniform(rows, n, dtype, 2 * seed + 1).to(torch.float64)
    if rows > 2 * radius:
        out[radius:rows - radius, radius:n - radius] += _stencil(x, pattern, radius)
    x.add_(1.0)
    x[:top] = 0.0
    x[rows - bot:] = 0.0
    return {"in": x, "out": out}
