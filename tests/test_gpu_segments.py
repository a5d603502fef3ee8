"""The segment kernels at the edges of their tiles and at every alignment of
source and destination, bit-exact."""

import numpy as np
import pytest
import torch

import oracle
from test1_amd import kernels
from test1_amd.pinned import pinned_empty

pytestmark = pytest.mark.gpu

# one tile is 2048 elements, of a capped grid 16384
SIZES = [1, 7, 8, 9, 15, 2040, 2047, 2048, 2049, 2056, 4096 + 3, 16383, 16384, 16385, 2 * 16384 + 11]
GAP = 24   # elements between two segments that nothing may write


def layout(src_skew, dst_skew):
    """(source offset, destination offset, size) per segment, and the ends."""
    rows, s, d = [], 0, 0
    for n in SIZES:
        s, d = (s + 7) // 8 * 8 + src_skew, (d + 7) // 8 * 8 + dst_skew
        rows.append((s, d, n))
        s, d = s + n + GAP, d + n + GAP
    return rows, s, d


@pytest.mark.parametrize("dst_skew", range(8))
@pytest.mark.parametrize("src_skew", [0, 1, 3, 4, 6])
def test_cast_and_copy_at_every_alignment(dev, src_skew, dst_skew):
    rows, ns, nd = layout(src_skew, dst_skew)
    x = torch.randn(ns, generator=torch.Generator().manual_seed(8 * src_skew + dst_skew))
    bits = oracle.cast_f32_bf16(x.numpy()).view(np.int16)
    exp = np.full(nd, -1, np.int16)
    for s, d, n in rows:
        exp[d:d + n] = bits[s:s + n]
    xs, hs = x.to(dev), torch.from_numpy(bits.copy()).to(dev)
    out = torch.full((nd,), -1, dtype=torch.int16, device=dev)
    kernels.cast_scatter_f32_bf16([(xs[s:s + n], out[d:d + n].view(torch.bfloat16)) for s, d, n in rows])
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), exp)
    host = pinned_empty(nd, torch.int16)
    for dst, wg in ((out, 0), (out, 3), (host, 3)):
        dst.fill_(-1)
        kernels.copy_segs_b16([(hs[s:s + n], dst[d:d + n]) for s, d, n in rows], max_workgroups=wg)
        torch.cuda.synchronize()
        assert np.array_equal(dst.cpu().numpy(), exp), (dst.device, wg)


@pytest.mark.parametrize("wg", [0, 5])
def test_pack_and_unpack_of_neighbours(dev, wg):
    """Segments end to end: two of them share the 16 bytes where they meet."""
    sizes = SIZES * 5   # more than one launch's table
    flat = torch.arange(sum(sizes), device=dev, dtype=torch.int32).to(torch.int16)
    parts = [p.clone() for p in flat.split(sizes)]
    out = torch.zeros_like(flat)
    kernels.pack_b16(parts, out, max_workgroups=wg)
    back = [torch.zeros_like(p) for p in parts]
    kernels.unpack_b16(flat, back, max_workgroups=wg)
    torch.cuda.synchronize()
    assert torch.equal(out, flat)
    assert all(torch.equal(a, b) for a, b in zip(back, parts))


@pytest.mark.parametrize("wg", [0, 1, 5])
def test_unpack_of_host_memory(dev, wg):
    """Tiles of 8192 elements of a capped grid, of 2048 otherwise."""
    sizes = [*SIZES, 8191, 8192, 8193, 3 * 8192 + 5]
    flat = pinned_empty(sum(sizes) + 3, torch.int16)
    flat.copy_(torch.arange(flat.numel(), dtype=torch.int32).to(torch.int16))
    for skew in (0, 3):
        back = [torch.full((n + 2,), -1, dtype=torch.int16, device=dev) for n in sizes]
        kernels.unpack_b16(flat[skew:], [b[1:-1] for b in back], max_workgroups=wg)
        torch.cuda.synchronize()
        for b, want in zip(back, flat[skew:skew + sum(sizes)].split(sizes)):
            assert torch.equal(b[1:-1].cpu(), want) and int(b[0]) == int(b[-1]) == -1
