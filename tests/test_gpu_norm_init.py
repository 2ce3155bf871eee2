"""The L1 norm and the initial values at the edges of their vectors: n on
either side of a whole number of vectors and of the columns one block takes
at a time, every radius's first interior column, rows on 16-byte boundaries
and off them.  The norm's reference is an exact sum (math.fsum); columns
outside the interior hold NaN and infinities, which it must not see."""
import math

import numpy as np
import pytest
import torch

import kernels_amd as K

pytestmark = pytest.mark.gpu
MASK = (1 << 64) - 1


@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("n,radius,pad", [(3, 1, 0), (17, 8, 0), (18, 8, 1), (65, 3, 0), (511, 2, 1), (512, 1, 0),
                                          (513, 5, 0), (2047, 2, 0), (2049, 7, 0)])
def test_norm_is_the_exact_sum(gpu, dtype, n, radius, pad):
    for pitch in (K.default_pitch(n, dtype), n + pad):
        print(f"norm d{dtype} n={n} R={radius} pitch={pitch}", flush=True)
        gen = torch.Generator(device=gpu).manual_seed(n)
        base = torch.full((n, pitch), float("nan"), dtype=K.torch_dtype(dtype), device=gpu)
        g = base[:, :n]
        g.fill_(float("inf"))
        inner = slice(radius, n - radius)
        g[inner, inner] = (torch.rand((n - 2 * radius,) * 2, generator=gen, device=gpu) * 2 - 1).to(g.dtype)
        want = math.fsum(np.abs(g[inner, inner].double().cpu().numpy()).ravel()) / (n - 2 * radius) ** 2
        got = K.l1norm(dtype, radius, g)
        # the sum is right to far below a rounding; rounded once, divided once
        assert abs(got - want) <= 2.0 ** -51 * want, (got, want)


@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 511, 1025])
def test_seeded_initial_values(gpu, dtype, n):
    def value(seed, idx):
        z = (seed + (idx + 1) * 0x9E3779B97F4A7C15) & MASK
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & MASK
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & MASK
        return 2.0 * (((z ^ (z >> 31)) >> 11) * 2.0 ** -53) - 1.0

    seed = 0xFEDCBA9876543210
    for pitch in (K.default_pitch(n, dtype), n):
        print(f"init d{dtype} n={n} pitch={pitch}", flush=True)
        base = [torch.full((n, pitch), 3.0, dtype=K.torch_dtype(dtype), device=gpu) for _ in range(2)]
        a, out = (b[:, :n] for b in base)
        K.init(K.INIT_SEEDED, seed, dtype, a, out)
        rows = sorted({0, n // 2, n - 1})
        want = torch.tensor([[value(seed, r * n + c) for c in range(n)] for r in rows], dtype=torch.float64)
        if dtype == 2:
            want = want.float()  # rounded to FP32, then to BF16
        assert torch.equal(a[rows].cpu(), want.to(a.dtype))
        assert bool((out == 0).all())
        for b in base:
            assert bool((b[:, n:] == 3.0).all())
