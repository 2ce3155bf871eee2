"""Sweeps one call each (K.sweep, and stencil then add) with the default
tiling, against the oracle bit for bit.  K.run takes many sweeps per pass, so
these are the tests of the sweep kernels that a program's own loop runs."""
import numpy as np
import pytest
import torch

import kernels_amd as K
from tests._oracle import BF16, F32, F64

pytestmark = pytest.mark.gpu


def bits(a: np.ndarray) -> np.ndarray:
    return a.view({8: np.uint64, 4: np.uint32, 2: np.uint16}[a.dtype.itemsize])


def host(t: torch.Tensor) -> np.ndarray:
    torch.cuda.synchronize()
    if t.dtype == torch.bfloat16:
        return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)
    return t.contiguous().cpu().numpy()


def loop(pattern, radius, dtype, bufs, sweeps):
    """Sweeps over the ping-pong pair; returns the buffer that holds in."""
    src, dst, out = bufs
    for _ in range(sweeps):
        K.sweep(pattern, radius, dtype, src, dst, out)
        src, dst = dst, src
    return src


def band(oracle, dtype, pattern, radius, n, iters, seed, a, b):
    if dtype == F64:
        return oracle.band(pattern, radius, n, iters, 1, seed, a, b)
    return oracle.band_lp(dtype, pattern, radius, n, iters, 1, seed, a, b)


# ragged rows on both sides of the sizes at which the arrays leave the L2s (20
# MB) and the last-level cache (256 MB): each takes other stores
@pytest.mark.parametrize("dtype,n", [(F64, 905), (F64, 921), (F64, 3243), (F64, 3299), (F32, 1301), (F32, 1337),
                                     (F32, 4673), (F32, 4801), (BF16, 1833), (BF16, 1897), (BF16, 6663), (BF16, 6791)])
@pytest.mark.parametrize("pattern,radius", [(0, 2), (0, 6), (1, 3), (1, 7), (1, 8)])
def test_forms_by_size(gpu, oracle, dtype, n, pattern, radius):
    for pitch in (None, n):
        print(f"form p{pattern} r{radius} d{dtype} n={n} pitch={pitch}", flush=True)
        base = [torch.full((n, pitch or K.default_pitch(n, dtype)), 3.0, dtype=K.torch_dtype(dtype), device=gpu)
                for _ in range(3)]
        b0, b1, out = (b[:, :n] for b in base)
        K.init(K.INIT_SEEDED, 5, dtype, b0, out)
        loop(pattern, radius, dtype, (b0, b1, out), 1)
        for a, b in ((0, radius + 3), (n // 2, n // 2 + 9), (n - radius - 3, n)):
            assert np.array_equal(bits(host(out[a:b])), bits(band(oracle, dtype, pattern, radius, n, 0, 5, a, b))), (a, b)
        one = b0 + 1
        assert torch.equal(b1, one)
        unfused = torch.zeros_like(base[2])[:, :n]
        K.stencil_ex(pattern, radius, dtype, b0, unfused)
        assert torch.equal(unfused, out)
        K.check(K.lib().prk_add_ex(dtype, n, b0.stride(0), b0.data_ptr(), torch.cuda.current_stream().cuda_stream))
        assert torch.equal(b0, one)
        for b in base:
            assert bool((b[:, n:] == 3.0).all())


# the refresh alone and after a stencil takes rows or vectors of the array by its size
@pytest.mark.parametrize("n", [886, 888, 1144, 1146, 2048, 2050])
def test_refresh_by_size(gpu, n):
    t = torch.rand((n, n), generator=torch.Generator(device=gpu).manual_seed(n), device=gpu, dtype=torch.float64)
    want = t + 1.0
    K.add(n, 32, t)
    assert torch.equal(t, want)


@pytest.mark.parametrize("dtype", [F64, F32, BF16])
@pytest.mark.parametrize("pattern,radius", [(p, r) for p in (0, 1) for r in range(1, 9)])
def test_sweep_by_sweep_bitwise(gpu, oracle, pattern, radius, dtype):
    # whole vectors, ragged rows, and rows off 16 bytes, default tiling
    strip, sweeps = 64 * (2, 4, 8)[dtype], 5
    for n, pitch in ((2 * radius + 1, None), (strip, None), (strip + 1, None), (131 + radius, 131 + radius)):
        print(f"sweeps p{pattern} r{radius} d{dtype} n={n} pitch={pitch}", flush=True)
        bufs = [K.alloc_grid(n, dtype, pitch=pitch) for _ in range(3)]
        K.init(K.INIT_SEEDED, 31 + n, dtype, bufs[0], bufs[2])
        fin = loop(pattern, radius, dtype, bufs, sweeps)
        if dtype == F64:
            ref_out, ref_in = oracle.run(pattern, radius, n, 32, sweeps - 1, 1, 31 + n)
        else:
            ref_out, ref_in = oracle.run_lp(dtype, pattern, radius, n, sweeps - 1, 1, 31 + n)
        assert np.array_equal(bits(host(bufs[2])), bits(ref_out)), (n, pitch)
        assert np.array_equal(bits(host(fin)), bits(ref_in)), (n, pitch)


@pytest.mark.parametrize("dtype,pattern,radius", [(F64, 0, 4), (F64, 1, 3), (F32, 0, 4), (F32, 1, 2), (BF16, 0, 7)])
def test_sweeps_of_the_tuned_tiling(gpu, oracle, dtype, pattern, radius):
    # the tiling that the search recorded, without an override
    n, sweeps = 256, 3
    bufs = [K.alloc_grid(n, dtype) for _ in range(3)]
    try:
        tuned, got = K.autotune(pattern, radius, dtype, *bufs, reps=1), K.Tuning()
        K.check(K.lib().prk_tuning_get(pattern, radius, dtype, n, got))
        assert (got.variant, got.rows_per_wave) == (tuned.variant, tuned.rows_per_wave)
        K.init(K.INIT_SEEDED, 4, dtype, bufs[0], bufs[2])
        loop(pattern, radius, dtype, bufs, sweeps)
        assert np.array_equal(bits(host(bufs[2])), bits(band(oracle, dtype, pattern, radius, n, sweeps - 1, 4, 0, n)))
    finally:
        K.check(K.lib().prk_tuning_clear())


@pytest.mark.parametrize("dtype,n,pattern,radius", [(F64, 30000, 0, 2), (F64, 30000, 1, 2), (F64, 16384, 1, 5),
                                                    (F32, 30000, 0, 2), (BF16, 30000, 1, 3)])
def test_large_grid_sweeps_on_bands(gpu, oracle, dtype, n, pattern, radius):
    bufs, sweeps = [K.alloc_grid(n, dtype) for _ in range(3)], 2
    K.init(K.INIT_SEEDED, 42, dtype, bufs[0], bufs[2])
    loop(pattern, radius, dtype, bufs, sweeps)
    rng = np.random.default_rng(7)
    spans = [(0, radius + 4), (n - radius - 4, n)] + [(int(a), int(a) + 8) for a in rng.integers(0, n - 8, 6)]
    for rows in (8, 12, 32):  # across tile boundaries in the middle
        c = n // 2 // rows * rows
        spans.append((c - 3, c + 3))
    for a, b in spans:
        ref = band(oracle, dtype, pattern, radius, n, sweeps - 1, 42, a, b)
        assert np.array_equal(bits(host(bufs[2][a:b])), bits(ref)), (a, b)
