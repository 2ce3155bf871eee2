"""Several sweeps per pass (K.run) against the oracle, bit for bit.

Every stencil that has a pass kernel, in every storage type, at the sizes
where a pass can go wrong: the smallest grid, one strip of 64 lanes and the
column on either side of it, row groups that end inside the grid, rows that
are not on 16-byte boundaries, and odd and even numbers of sweeps (which set
the number of passes and the buffer that ends up with in).  Columns past n
and the frame of out must keep what they held."""
import numpy as np
import pytest
import torch

import kernels_amd as K
from tests._oracle import F64

pytestmark = pytest.mark.gpu

VEC = {0: 2, 1: 4, 2: 8}  # columns per lane
BITS = {8: np.uint64, 4: np.uint32, 2: np.uint16}


def host(t):
    torch.cuda.synchronize()
    if t.dtype == torch.bfloat16:
        return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)
    return t.contiguous().cpu().numpy()


def bits(a):
    return a.view(BITS[a.dtype.itemsize])


def stencils():
    return [(p, r) for p in (0, 1) for r in range(1, 9)]


@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("pattern,radius", stencils())
def test_run_bitwise(gpu, oracle, pattern, radius, dtype):
    strip = 64 * VEC[dtype]
    sizes = [(2 * radius + 1, None, 3), (strip - 1, None, 4), (strip, None, 2), (strip + 1, strip + 1, 5),
             (37 + radius, 37 + radius, 7)]
    for n, pitch, iters in sizes:
        print(f"pass p{pattern} r{radius} d{dtype} n={n} pitch={pitch} iterations={iters}", flush=True)
        pitch = pitch or K.default_pitch(n, dtype)
        base = [torch.full((n, pitch), 3.0, dtype=K.torch_dtype(dtype), device=gpu) for _ in range(3)]
        b0, b1, out = (b[:, :n] for b in base)
        K.init(K.INIT_SEEDED, 77 + n, dtype, b0, out)
        final, _ = K.run(pattern, radius, dtype, iters, b0, b1, out)
        assert final == (iters + 1) % 2
        if dtype == F64:
            ref_out, ref_in = oracle.run(pattern, radius, n, 32, iters, 1, 77 + n)
        else:
            ref_out, ref_in = oracle.run_lp(dtype, pattern, radius, n, iters, 1, 77 + n)
        assert np.array_equal(bits(host(out)), bits(ref_out)), (n, pitch, iters)
        assert np.array_equal(bits(host((b0, b1)[final])), bits(ref_in)), (n, pitch, iters)
        for b in base:
            assert bool((b[:, n:] == 3.0).all())


@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("n", [63, 300])
def test_frame_of_out_is_kept(gpu, dtype, n):
    b0, b1, out = (K.alloc_grid(n, dtype) for _ in range(3))
    K.init(K.INIT_SEEDED, 5, dtype, b0, out)
    out.fill_(7.0)
    K.run(K.STAR, 3, dtype, 4, b0, b1, out)
    o = out.float()
    assert bool((o[:3] == 7.0).all() and (o[-3:] == 7.0).all() and (o[:, :3] == 7.0).all() and (o[:, -3:] == 7.0).all())
    assert bool((o[3:-3, 3:-3] != 7.0).any())


def test_passes_equal_single_sweeps(gpu):
    # more sweeps than one pass holds: 300 sweeps are two passes; the same
    # run one sweep per pass (a tiling override) gives the same bits
    n, iters = 150, 300
    got = []
    for rows in (0, 8):
        K.check(K.lib().prk_set_rows_per_wave(rows))
        try:
            b0, b1, out = (K.alloc_grid(n, K.F64) for _ in range(3))
            K.init(K.INIT_SEEDED, 9, K.F64, b0, out)
            final, _ = K.run(K.GRID, 2, K.F64, iters, b0, b1, out)
            got.append((bits(host(out)), bits(host((b0, b1)[final]))))
        finally:
            K.check(K.lib().prk_set_rows_per_wave(0))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])


def test_first_run_is_timed_without_loading_code(gpu):
    """The time a fresh process reports for its first run is that of the
    sweeps.  Loading the pass kernel's code takes about 0.6 ms, 60 us for each
    of 10 sweeps, where a sweep by itself takes 9; the least of five processes
    is under 30."""
    import re
    import subprocess
    from pathlib import Path

    exe = Path(K.__file__).parent / "prk-stencil"
    times = []
    for _ in range(5):
        text = subprocess.run([str(exe), "10", "1000"], capture_output=True, text=True, timeout=60, check=True).stdout
        times.append(float(re.search(r"Avg time \(s\):\s*(\S+)", text).group(1)))
    assert min(times) < 30e-6, times


@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("pattern,radius", [(0, 1), (0, 2), (0, 4), (0, 8), (1, 1), (1, 2), (1, 3), (1, 4)])
def test_run_of_any_values(gpu, pattern, radius, dtype):
    """An even number of iterations runs sweep 0, which reads the caller's
    values, inside the pass.  Values whose products with the weights round
    below the normal range, and sums that lie there themselves, give the bits
    of sweeps one by one; so do ordinary and large ones, on an out that holds
    values already."""
    n = 64 * VEC[dtype] + 13
    tiny, big = (2.0**-1060, 2.0**900) if dtype == F64 else (2.0**-138, 2.0**100)
    td = K.torch_dtype(dtype)
    gen = torch.Generator(device=gpu).manual_seed(9)
    a, o = (torch.rand((n, n), generator=gen, device=gpu, dtype=torch.float64) * 2 - 1 for _ in range(2))
    a[: n // 2] *= tiny
    a[n // 2 + 20 : n // 2 + 24] *= big
    o[: n // 2] = 0.0
    for iters in (2, 10):
        print(f"any p{pattern} r{radius} d{dtype} n={n} iterations={iters}", flush=True)
        got, want = ([K.alloc_grid(n, dtype) for _ in range(3)] for _ in range(2))
        for g in (got, want):
            g[0].copy_(a.to(td))
            g[1].zero_()
            g[2].copy_(o.to(td))
        final, _ = K.run(pattern, radius, dtype, iters, *got)
        src, dst, out = want
        for _ in range(iters + 1):
            K.sweep(pattern, radius, dtype, src, dst, out)
            src, dst = dst, src
        assert final == (iters + 1) % 2
        assert np.array_equal(bits(host(got[2])), bits(host(out))), iters
        assert np.array_equal(bits(host(got[final])), bits(host(src))), iters
