"""The flat cast at the edges of its workgroups' tiles (1024 elements) and at
every alignment, bit-exact, in one launch, with nothing written around it."""

import numpy as np
import pytest
import torch

import oracle
from test1_amd import _native, kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 8, 9, 15, 1016, 1017, 1023, 1024, 1025, 1031, 1032, 2048, 3 * 1024 + 5])
@pytest.mark.parametrize("src_off", [0, 1, 2, 3])
def test_cast_at_every_alignment(dev, n, src_off):
    rng = np.random.default_rng(n + src_off)
    bits = rng.integers(0, 1 << 32, n + src_off, dtype=np.uint64).astype(np.uint32)   # NaN, infinities, subnormals
    x = torch.from_numpy(bits.view(np.float32).copy())
    xs = x.to(dev)[src_off:]
    for dtype, ref in ((torch.bfloat16, oracle.cast_f32_bf16), (torch.float16, oracle.cast_f32_f16)):
        want = ref(x.numpy()[src_off:])
        for dst_off in range(8):
            out = torch.full((n + 32,), -1, dtype=torch.int16, device=dev)
            timer = kernels.KernelTimer() if dst_off % 2 else None
            kernels.cast_f32_16_(out[dst_off + 8:dst_off + 8 + n].view(dtype), xs, timer=timer)
            torch.cuda.synchronize()
            got = out.cpu().numpy().view(np.uint16)
            exp = np.full(n + 32, 0xFFFF, np.uint16)
            exp[dst_off + 8:dst_off + 8 + n] = want
            assert np.array_equal(got, exp), (dtype, dst_off)
            assert timer is None or timer.elapsed_ms() > 0.0


@pytest.mark.parametrize("past", [0, 7])
def test_largest_cast(dev, past):
    """2^33 elements and up to 7 more are the largest aligned cast; 8 more are refused."""
    n = (1 << 33) + past
    if torch.cuda.mem_get_info(dev)[0] < 8 * n:
        pytest.skip("needs 64 GiB of free GPU memory")
    src = torch.zeros(n + 8, device=dev)
    src[:1000] = torch.arange(1000, device=dev)
    src[n - 1000:n] = torch.arange(1000, device=dev)
    out = torch.full((n + 8,), -1, dtype=torch.int16, device=dev)
    kernels.cast_f32_16_(out[:n].view(torch.bfloat16), src[:n])
    want = torch.arange(1000, device=dev).bfloat16().view(torch.int16)
    assert torch.equal(out[:1000], want) and torch.equal(out[n - 1000:n], want) and bool((out[n:] == -1).all())
    assert not any(bool(part.any()) for part in out[1000:n - 1000].split(1 << 31))
    if past:
        with pytest.raises(_native.NativeError):
            kernels.cast_f32_16_(out[:n - past + 8].view(torch.bfloat16), src[:n - past + 8])
