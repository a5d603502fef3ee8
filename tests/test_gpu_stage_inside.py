"""Staging from inside a pinned allocation into the inside of a device one, at
any element, and again after the host has rewritten the master: bit for bit,
with the neighbours untouched."""

import numpy as np
import pytest
import torch

import oracle
from test1_amd import kernels
from test1_amd.pinned import pinned_empty

pytestmark = pytest.mark.gpu

# one element to several tiles of 16,384; the largest size that one kernel reads, and pieces through a buffer
SIZES = [1, 9, 16_384, 100_003, 1 << 22, (1 << 22) + 1]


def stage(entry, dst, src):
    if entry == "noalloc":
        kernels.stage_f32_bf16_noalloc_(dst, src)
    else:
        kernels.stage_f32_bf16_(dst, src, torch.empty(1 << 22, dtype=torch.float32, device=dst.device))


@pytest.mark.parametrize("entry", ["workspace", "noalloc"])
@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("torch_pinned", [False, True])
def test_stage_between_the_insides_of_allocations(dev, torch_pinned, n, entry):
    before = 70_001
    room = before + n + 16
    master = torch.empty(room, pin_memory=True) if torch_pinned else pinned_empty(room, torch.float32)
    g = torch.Generator().manual_seed(n)
    large = n >= 1 << 22
    for k in (3, before) if large else (1, 2, 3, 4, before):
        for j in (1,) if large else (0, 1, 7):
            for again in range(2):   # the second time other values at the same place
                master.copy_(torch.randn(room, generator=g))
                out = torch.full((j + n + 9,), 7.0, dtype=torch.bfloat16, device=dev)
                stage(entry, out[j:j + n], master[k:k + n])
                torch.cuda.synchronize()
                got = out.cpu()
                assert np.array_equal(got[j:j + n].view(torch.int16).numpy().view(np.uint16),
                                      oracle.cast_f32_bf16(master.numpy()[k:k + n])), (k, j, again)
                assert bool((got[:j] == 7.0).all()) and bool((got[j + n:] == 7.0).all()), (k, j, again)


@pytest.mark.parametrize("entry", ["workspace", "noalloc"])
def test_a_large_array_leaves_the_compute_units_to_others(dev, entry):
    """Above 4 Mi elements the transfer is a DMA copy: the casts that follow it
    run for a fraction of its time.  The kernel that reads the link would show
    as one kernel of the whole duration."""
    n = 32 << 20
    src = pinned_empty(n, torch.float32)
    src.zero_()
    dst = torch.empty(n, dtype=torch.bfloat16, device=dev)
    work = torch.empty(8 << 20, dtype=torch.float32, device=dev)

    def call():
        if entry == "noalloc":
            kernels.stage_f32_bf16_noalloc_(dst, src)
        else:
            kernels.stage_f32_bf16_(dst, src, work)

    call()
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    kernels_us = sum(e.device_time_total for e in prof.key_averages() if "cast" in e.key or "seg_kernel" in e.key)
    assert 0 < kernels_us < 500, kernels_us   # 2,251 us is the link's time for the array
