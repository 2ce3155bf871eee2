"""in += 1 against plain torch, bit for bit: whole and ragged numbers of
vectors, dense arrays (taken flat) and pitched ones, on 16-byte boundaries and
off them, and a dense array larger than the last-level cache."""
import pytest
import torch

import kernels_amd as K

pytestmark = pytest.mark.gpu


def add(dtype, n, pitch, t):
    K.check(K.lib().prk_add_ex(dtype, n, pitch, t.data_ptr(), torch.cuda.current_stream().cuda_stream))


@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("n", [1, 2, 3, 7, 31, 64, 65, 255, 1025])
def test_add_bitwise(gpu, dtype, n):
    gen = torch.Generator(device=gpu).manual_seed(n)
    for pitch in (n, n + 3, K.default_pitch(n, dtype)):
        for offset in (0, 1):
            print(f"add d{dtype} n={n} pitch={pitch} offset={offset}", flush=True)
            base = (torch.rand(n * pitch + 9, generator=gen, device=gpu) * 4 - 2).to(K.torch_dtype(dtype))
            want = base.clone()
            inner = want[offset:offset + n * pitch].view(n, pitch)[:, :n]
            inner += 1
            add(dtype, n, pitch, base[offset:])
            assert torch.equal(base, want)


def test_add_beyond_the_cache(gpu):
    n = 5801  # 269 MB of FP64, an odd number of elements
    t = torch.rand((n, n), generator=torch.Generator(device=gpu).manual_seed(1), device=gpu, dtype=torch.float64)
    want = t + 1.0
    K.add(n, 32, t)
    assert torch.equal(t, want)
