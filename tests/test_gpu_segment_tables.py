"""Segment tables read from tensors natively: the same as the ones made in
Python, and nothing taken that Python's checks would refuse or treat apart."""

import pytest
import torch

from test1_amd import _native, kernels
from test1_amd.pinned import pinned_empty

pytestmark = pytest.mark.gpu


class Sub(torch.Tensor):
    pass


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.int16, torch.uint16])
def test_tables_equal_the_python_ones(dev, dtype):
    base = torch.zeros(4096, dtype=dtype, device=dev)
    ts = [base[3:70], base[100:612].view(16, 32), base[0:0], base.view(2, 1, 2048)[1], base[1::4096]]
    if dtype.is_floating_point:
        ts.append(torch.nn.Parameter(base[7:9]))
    for as_dst in (False, True):
        table, count, total = _native.segs().list_table(ts, as_dst)
        rows = [(0, t.data_ptr(), t.numel()) if as_dst else (t.data_ptr(), 0, t.numel()) for t in ts]
        assert (count, total) == (len(ts), sum(t.numel() for t in ts))
        assert table == bytes(kernels._seg_array(rows))
    out = [torch.zeros_like(t) for t in ts]
    table, count = _native.segs().pair_table(list(zip(ts, out)), False)
    assert table == bytes(kernels._seg_array([(a.data_ptr(), b.data_ptr(), a.numel()) for a, b in zip(ts, out)]))
    assert _native.segs().list_table((), False) == (b"", 0, 0)


def test_the_rest_is_left_to_the_python_checks(dev):
    ok = torch.zeros(64, dtype=torch.bfloat16, device=dev)
    f32 = torch.zeros(64, device=dev)
    left = [ok[::2], f32, ok.cpu(), pinned_empty(64, torch.bfloat16), ok.as_subclass(Sub), ok.to("meta"), None, 3,
            ok.view(8, 8).t(), ok.to_sparse()]
    for t in left:
        assert _native.segs().list_table([ok, t], False) is None, t
        assert _native.segs().pair_table([(ok, ok), (ok, t)], False) is None, t
    assert _native.segs().list_table(iter([ok]), False) is None
    assert _native.segs().pair_table([(ok, ok[:32])], False) is None     # sizes differ
    assert _native.segs().pair_table([(ok, ok, ok)], False) is None
    assert _native.segs().pair_table([(f32, ok)], True)[1] == 1
    assert _native.segs().pair_table([(ok, ok)], True) is None
    with pytest.raises(ValueError, match=r"srcs\[1\] must be contiguous"):
        kernels.pack_b16([ok, ok[::2]], torch.zeros(256, dtype=torch.bfloat16, device=dev))
    with pytest.raises(TypeError, match="pair 0: need float32 -> bfloat16"):
        kernels.cast_scatter_f32_bf16([(ok, ok)])
    # a subclass and a host destination still run
    dst, host = torch.ones(64, dtype=torch.bfloat16, device=dev), pinned_empty(64, torch.bfloat16)
    kernels.copy_segs_b16([(ok.as_subclass(Sub), dst), (ok, host)])
    torch.cuda.synchronize()
    assert not dst.any() and not host.any()
    inside = []
    torch.func.vmap(lambda x: inside.append(_native.segs().list_table([x], False)) or x)(ok.view(2, 32))
    assert inside == [None]


def test_the_same_results_without_the_module(dev, monkeypatch):
    sizes = [3, 64, 1000, 1]
    parts = [torch.randn(n, device=dev).bfloat16() for n in sizes]
    wide = [p.float() for p in parts]

    def results():
        packed = torch.empty(sum(sizes), dtype=torch.bfloat16, device=dev)
        back, copies, cast = ([torch.zeros_like(p) for p in parts] for _ in range(3))
        kernels.pack_b16(parts, packed)
        kernels.unpack_b16(packed, back)
        kernels.copy_segs_b16(list(zip(parts, copies)))
        kernels.cast_scatter_f32_bf16(list(zip(wide, cast)))
        return [packed, *back, *copies, *cast]

    want = results()
    monkeypatch.setattr(_native, "segs", lambda: None)
    assert all(torch.equal(a, b) for a, b in zip(results(), want))
    assert torch.equal(want[0], torch.cat(parts))
