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
@pytest.mark.parametrize("n", [1144, 1146, 2048, 2050])
def test_refresh_by_size(gpu, n):
    t = torch.rand((n, n), generator=torch.Generator(device=gpu).manual_seed(n), device=gpu, dtype=torch.float64)
    want = t + 1.0
    K.add(n, 32, t)
    assert torch.equal(t, want)
