"""Row gathers against plain indexing, bit for bit: rows that fill a tile,
straddle two or start anywhere, tables and destinations in HBM and in pinned
host memory, ids outside the table, and ids that repeat within and across the
windows in which a row crosses the host link once."""

import numpy as np
import pytest
import torch

import oracle
from test1_amd import kernels
from test1_amd.pinned import pinned_empty

pytestmark = pytest.mark.gpu


def check(dev, nrows, row_len, ids, f32, src_host, dst_host, wg=0, skew=0):
    g = torch.Generator().manual_seed(nrows + row_len)
    values = torch.randn(nrows * row_len, generator=g)
    values[:1] = float("nan")
    bits = torch.from_numpy(oracle.cast_f32_bf16(values.numpy()).view(np.int16))
    data, dtype = (values, torch.float32) if f32 else (bits, torch.int16)
    flat = (pinned_empty(data.numel() + skew, dtype) if src_host
            else torch.empty(data.numel() + skew, dtype=dtype, device=dev))
    flat[skew:].copy_(data)
    n = ids.numel() * row_len
    out = pinned_empty(n + skew + 9, torch.int16) if dst_host else torch.empty(n + skew + 9, dtype=torch.int16,
                                                                               device=dev)
    out.fill_(7)
    bad = torch.zeros(1, dtype=torch.int32, device=dev)
    kernels.gather_rows(flat[skew:].view(nrows, row_len), ids.to(dev), out[skew:skew + n].view(-1, row_len), bad=bad,
                        max_workgroups=wg)
    torch.cuda.synchronize()
    valid = (ids >= 0) & (ids < nrows)
    exp = torch.full((ids.numel(), row_len), -1, dtype=torch.int16)
    exp[valid] = bits.view(nrows, row_len)[ids[valid]]
    got = out.cpu()
    assert torch.equal(got[skew:skew + n].view(-1, row_len), exp)
    assert bool((got[:skew] == 7).all()) and bool((got[skew + n:] == 7).all()), "wrote outside the rows"
    assert int(bad.item()) == int(not bool(valid.all()))


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("src_host,dst_host,wg", [(False, False, 0), (False, False, 3), (True, False, 0),
                                                  (True, False, 2), (False, True, 5), (True, True, 4)])
@pytest.mark.parametrize("row_len,skew", [(8, 0), (64, 0), (72, 1), (1, 0), (7, 3), (507, 0), (2040, 0), (4096, 0),
                                          (8192, 0), (16392, 0), (16384, 5)])
def test_rows_of_any_length(dev, f32, src_host, dst_host, wg, row_len, skew):
    nrows = 37
    g = torch.Generator().manual_seed(row_len)
    ids = torch.randint(0, nrows, (max(3, 40_000 // row_len),), generator=g)
    check(dev, nrows, row_len, ids, f32, src_host, dst_host, wg, skew)
    ids[::3] = torch.tensor([-1, nrows, 1 << 40])[torch.arange(len(ids[::3])) % 3]
    check(dev, nrows, row_len, ids, f32, src_host, dst_host, wg, skew)


@pytest.mark.parametrize("ids", [torch.empty(0, dtype=torch.int64), torch.tensor([0, 5, -1])])
def test_no_rows_asked_for_and_no_rows_to_have(dev, ids):
    check(dev, 1, 16, ids, True, False, False)


@pytest.mark.parametrize("f32,row_len,nrows,ntok", [
    (True, 4096, 100, 300),      # one window, most rows repeated
    (False, 8192, 300, 700),
    (True, 515, 4000, 8192),     # a whole window of rows that start anywhere
    (True, 512, 4001, 8193),     # and one token more
    (False, 1024, 2003, 20_000),
    (True, 1 << 19, 1, 40),      # one row alone
])
def test_repeated_rows_cross_the_link_once(dev, f32, row_len, nrows, ntok):
    """Sizes at which the two-kernel path runs (2 MiB of repeated rows a window,
    where a table of few rows counts as read 8 times)."""
    ids = torch.randint(0, nrows, (ntok,), generator=torch.Generator().manual_seed(ntok))
    check(dev, nrows, row_len, ids, f32, True, False)
    ids[5::7] = -1
    ids[6::11] = nrows
    check(dev, nrows, row_len, ids, f32, True, False)
    ids[:] = nrows - 1   # all the same
    check(dev, nrows, row_len, ids, f32, True, False)


@pytest.mark.parametrize("src_host,dst_host,row_len,ntok,wg", [
    (True, False, 8, 8192, 0), (True, False, 8, 8191, 0),             # short rows, many or few of them
    (True, False, 64, 20_000, 4095), (True, False, 64, 20_000, 4096), (True, False, 72, 20_000, 0),
    (False, True, 72, 3000, 32), (False, True, 72, 3000, 33),         # few or more workgroups into host memory
])
def test_both_sides_of_the_lines_between_the_kernels(dev, src_host, dst_host, row_len, ntok, wg):
    ids = torch.randint(0, 500, (ntok,), generator=torch.Generator().manual_seed(ntok + wg))
    ids[::17] = 500
    for f32 in (True, False):
        check(dev, 500, row_len, ids, f32, src_host, dst_host, wg)


@pytest.mark.parametrize("cap", [256, 257, (1 << 31) - 1])
def test_few_and_many_workgroups_for_a_table_in_hbm(dev, cap):
    """Up to 256 workgroups walk over windows of tokens, more over tiles; and
    2^24 of them would be more lanes than a launch takes."""
    n = (1 << 24) + 1000
    table = torch.arange(80, dtype=torch.int16, device=dev).view(10, 8)
    ids = torch.arange(n, device=dev) % 10
    out = torch.full((n, 8), -1, dtype=torch.int16, device=dev)
    kernels.gather_rows(table, ids, out, max_workgroups=cap)
    torch.cuda.synchronize()
    assert torch.equal(out, table[ids])


@pytest.mark.parametrize("src_host,nrows,row_len,ntok", [(False, 500, 72, 900), (True, 500, 72, 900), (True, 100, 4096, 300)])
def test_gathers_and_staging_in_a_captured_graph(dev, src_host, nrows, row_len, ntok):
    """The routes look at the memory's type on the host: allowed under capture.
    Replays with other ids and values, and eager work between them."""
    flat = pinned_empty(nrows * row_len, torch.float32) if src_host else torch.empty(nrows * row_len, device=dev)
    table = flat.view(nrows, row_len)
    host = pinned_empty(50_000, torch.float32)
    ids = torch.zeros(ntok, dtype=torch.int64, device=dev)
    rows = torch.zeros(ntok, row_len, dtype=torch.int16, device=dev)
    staged = torch.zeros(50_000, dtype=torch.bfloat16, device=dev)
    work = torch.empty(8, dtype=torch.float32, device=dev)

    def step():
        kernels.gather_rows(table, ids, rows)
        kernels.stage_f32_bf16_(staged, host, work)

    flat.zero_()
    host.zero_()
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for rep in range(3):
        g = torch.Generator().manual_seed(rep)
        flat.copy_(torch.randn(flat.numel(), generator=g))
        host.copy_(torch.randn(host.numel(), generator=g))
        ids.copy_(torch.randint(0, nrows, (ntok,), generator=g))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got = rows.cpu(), staged.cpu()
        rows.fill_(-1)
        step()   # eager
        torch.cuda.synchronize()
        assert torch.equal(got[0], rows.cpu()) and torch.equal(got[1], staged.cpu())
        bits = torch.from_numpy(oracle.cast_f32_bf16(flat.cpu().numpy()).view(np.int16)).view(nrows, row_len)
        assert torch.equal(got[0], bits[ids.cpu()]) and torch.equal(got[1], host.bfloat16())
