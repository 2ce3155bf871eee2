"""Both in buffers of K.run, bit for bit those of sweeps one call each: the
final in and the in before it, whatever number of sweeps a pass takes."""
import numpy as np
import pytest
import torch

import kernels_amd as K
from tests._oracle import BF16, F32, F64
from tests.test_gpu_sweep_loop import bits, host, loop

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [F64, F32, BF16])
@pytest.mark.parametrize("n,pitch", [(64, None), (513, None), (131, 131), (301, 304)])
def test_both_in_buffers(gpu, dtype, n, pitch):
    # one and two sweeps per pass, sweep 0 in the pass and apart, two passes
    for pattern, radius, iters in ((0, 2, 1), (0, 2, 2), (1, 2, 3), (0, 1, 10), (1, 1, 11), (0, 3, 257), (1, 6, 4)):
        print(f"buffers p{pattern} r{radius} d{dtype} n={n} pitch={pitch} iterations={iters}", flush=True)
        pt = pitch or K.default_pitch(n, dtype)
        base = [[torch.full((n, pt), 3.0, dtype=K.torch_dtype(dtype), device=gpu) for _ in range(3)] for _ in range(2)]
        got, want = ([b[:, :n] for b in x] for x in base)
        for g in (got, want):
            K.init(K.INIT_SEEDED, 11, dtype, g[0], g[2])
        final, _ = K.run(pattern, radius, dtype, iters, *got)
        last = loop(pattern, radius, dtype, want, iters + 1)
        assert got[final].data_ptr() == got[(iters + 1) % 2].data_ptr() and last is want[final]
        for k in range(3):
            assert np.array_equal(bits(host(got[k])), bits(host(want[k]))), (k, iters)
        for b in base[0]:
            assert bool((b[:, n:] == 3.0).all())
