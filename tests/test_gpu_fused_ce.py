"""The cross-entropy kernels of the fused output unit, against float64."""

import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx

from test1_amd import fused_ce, kernels
from test1_amd.fused_ce import chunked_linear_cross_entropy

pytestmark = pytest.mark.gpu

# Rounding of one result to the type, relative and absolute: half a unit in the
# last of 8, 11 or 24 significant bits is at most 2^-8, 2^-11 or 2^-24 of the
# value; below the normal range it is half the smallest subnormal.
EPS = {torch.bfloat16: (2.0 ** -8, 2.0 ** -134), torch.float16: (2.0 ** -11, 2.0 ** -25),
       torch.float32: (2.0 ** -24, 2.0 ** -126)}
# vocabularies at the edges of every workgroup shape (64 x 16, 256 x 16, 256 x 32,
# 512 x 32, 1024 x 32, x 64, x 96, x 128, x 152 elements, then the streaming kernel)
EDGES = [1, 7, 8, 9, 1024, 1025, 4096, 4097, 8192, 8195, 16384, 16391, 32768, 32769, 65536, 65537, 98304, 98312,
         131072, 131079, 155648, 155649, 160001]


def rows_reference(x, y, ignore_index=-100):
    """(row_loss, gradient) in float64."""
    x = x.double()
    lse = torch.logsumexp(x, dim=1)
    ys = y.clamp(0, x.shape[1] - 1).unsqueeze(1)
    loss = lse - x.gather(1, ys).squeeze(1)
    g = torch.exp(x - lse.unsqueeze(1))
    p = g.clone()
    g.scatter_add_(1, ys, -torch.ones_like(ys, dtype=g.dtype))
    ignored = y == ignore_index
    loss[ignored] = 0.0
    g[ignored] = 0.0
    return loss, g, p


def strided(rows, vocab, dtype, dev):
    return torch.empty(rows, -(-vocab // 64) * 64, dtype=dtype, device=dev)[:, :vocab]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("vocab", EDGES)
def test_rows_match_float64(dev, vocab, dtype):
    rows = 5
    gen = torch.Generator(device=dev).manual_seed(vocab)
    x = (torch.randn(rows, vocab, generator=gen, device=dev) * 3).to(dtype)
    y = torch.randint(0, vocab, (rows,), generator=gen, device=dev)
    y[0], y[1], y[2] = 0, vocab - 1, -100
    ref_loss, ref_g, p = rows_reference(x, y)
    got = strided(rows, vocab, dtype, dev)
    got.copy_(x)
    loss = torch.full((rows,), 7.0, device=dev)
    kernels.ce_rows_(got, y, -100, loss)
    torch.cuda.synchronize()
    # fp32 terms: exp's argument is rounded at |x - lse| <= 40, twice
    assert ((loss.double() - ref_loss).abs() <= 1e-6 * (4 + ref_loss.abs())).all()
    half_ulp, tiny = EPS[dtype]
    bound = half_ulp * ref_g.abs() + 6e-6 * p + tiny
    assert ((got.double() - ref_g).abs() <= bound).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
# 16, 64, 256 or 1024 lanes a row: 16-bit to 128, 1024, fp32 to 64, 512, 8192
@pytest.mark.parametrize("vocab", [1, 8, 15, 64, 65, 128, 129, 512, 513])
@pytest.mark.parametrize("rows", [1, 17, 333])
def test_short_rows_share_a_workgroup(dev, rows, vocab, dtype):
    """Rows of one wave, valid, ignored and bad ones side by side, the last
    workgroup ragged; nothing behind the last row is touched."""
    gen = torch.Generator(device=dev).manual_seed(rows * vocab)
    x = (torch.randn(rows, vocab, generator=gen, device=dev) * 3).to(dtype)
    y = torch.randint(0, vocab, (rows,), generator=gen, device=dev)
    y[1::3], y[2::5] = -100, vocab
    ref_loss, ref_g, p = rows_reference(x, y)
    ref_loss[y == vocab] = float("nan")
    ref_g[y == vocab] = float("nan")
    ld = -(-vocab // 8) * 8
    buf = torch.full((rows + 2, ld), 7.0, dtype=dtype, device=dev)
    buf[:rows, :vocab] = x
    loss = torch.full((rows + 1,), 7.0, device=dev)
    kernels.ce_rows_(buf[:rows, :vocab], y, -100, loss[:rows])
    half_ulp, tiny = EPS[dtype]
    good = y != vocab
    # as in test_rows_match_float64
    assert ((loss[:rows].double() - ref_loss)[good].abs() <= 1e-6 * (4 + ref_loss[good].abs())).all()
    bound = half_ulp * ref_g.abs() + 6e-6 * p + tiny
    assert ((buf[:rows, :vocab].double() - ref_g).abs() <= bound)[good].all()
    assert loss[:rows][~good].isnan().all() and buf[:rows, :vocab][~good].isnan().all()
    assert (buf[rows:] == 7.0).all() and loss[rows] == 7.0


@pytest.mark.parametrize("vocab", [40, 70_003])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_special_values(dev, vocab, dtype):
    """Infinities and NaN give what logsumexp and softmax give; a label outside
    the vocabulary gives NaN; an ignored row gives zeros whatever it holds."""
    inf, nan = float("inf"), float("nan")
    x = torch.randn(8, vocab, device=dev).to(dtype)
    x[0, 3] = inf
    x[1, 5] = nan
    x[2] = -inf
    x[3, 10:] = -inf          # most lanes see only -inf
    x[4, 7] = nan
    y = torch.tensor([1, 2, 3, 4, -100, vocab, -1, 6], device=dev)
    ref_loss, ref_g, _ = rows_reference(x, y)
    ref_loss[5:7] = nan
    ref_g[5:7] = nan
    got = strided(8, vocab, dtype, dev)
    got.copy_(x)
    loss = torch.empty(8, device=dev)
    kernels.ce_rows_(got, y, -100, loss)
    torch.testing.assert_close(loss.double(), ref_loss, rtol=1e-5, atol=1e-5, equal_nan=True)
    torch.testing.assert_close(got.double(), ref_g, rtol=1e-2, atol=1e-5, equal_nan=True)


@pytest.mark.parametrize("vocab", [40, 4096, 160_001])
def test_rows_keep_probabilities_down_to_the_smallest(dev, vocab):
    """logsumexp is 0 exactly, so a probability is exp of its logit: the nearest
    bf16 value, or its neighbour where two ulps of fp32 decide it, down to bf16's
    subnormals (the smallest is 2^-133, exp(-92.2))."""
    x = torch.full((1, vocab), -200.0, device=dev)
    x[0, 0] = 0.0
    x[0, 1:25] = torch.tensor([-30, -40.25, -55.5, -60.75, -70.5, -80, -85, -86, -87, -87.5, -88, -88.5, -89, -89.5, -90,
                               -90.5, -91, -91.5, -92, -92.5, -93, -94, -110, float("-inf")], device=dev)
    x = x.bfloat16()
    want = torch.exp(x[0, 1:25].double())
    got = strided(1, vocab, torch.bfloat16, dev)
    got.copy_(x)
    loss = torch.empty(1, device=dev)
    kernels.ce_rows_(got, torch.zeros(1, dtype=torch.int64, device=dev), -100, loss)
    assert loss.item() == 0.0
    half_ulp = torch.clamp(2.0 ** (torch.floor(torch.log2(want)) - 8), min=2.0 ** -134)
    err = (got[0, 1:25].double() - want).abs()
    assert (err <= half_ulp + 2.0 ** -22 * want).all(), (got[0, 1:25], want)


# one workgroup up to 50,000 rows, then 256 of 256 lanes
@pytest.mark.parametrize("n", [1, 63, 1025, 50_000, 50_001, 65_537, 1_000_003])
def test_mean_of_the_rows(dev, n):
    gen = torch.Generator(device=dev).manual_seed(n)
    row_loss = torch.rand(n, generator=gen, device=dev) * 20
    labels = torch.randint(0, 9, (n,), generator=gen, device=dev)
    row_loss[labels == 3] = 0.0
    loss, count = torch.full((3,), 7.0, device=dev), torch.full((3,), 7.0, device=dev)
    kernels.ce_loss(row_loss, labels, 3, loss[1], count[1])
    valid = int((labels != 3).sum())
    assert count.tolist() == [7.0, float(valid), 7.0] and loss[0] == loss[2] == 7.0
    want = row_loss.double().sum() / valid   # sums in 64 bits, rounded once
    assert (loss[1].isnan() and valid == 0) or abs(loss[1].double() - want) <= 2.0 ** -23 * want


def test_more_rows_than_one_launch_takes(dev):
    """fp32 rows take a workgroup of 1024 lanes each, and a launch fewer than
    2^32 lanes: 2^22 rows and more are launched in parts."""
    n, v = (1 << 22) + 5, 4
    gen = torch.Generator(device=dev).manual_seed(6)
    x = torch.randn(n, v, generator=gen, device=dev)
    y = torch.randint(0, v, (n,), generator=gen, device=dev)
    y[::1000] = -100
    ref_loss, ref_g, p = rows_reference(x, y)
    loss = torch.full((n + 1,), 7.0, device=dev)
    kernels.ce_rows_(x, y, -100, loss[:n])
    torch.cuda.synchronize()
    # as in test_rows_match_float64
    assert ((loss[:n].double() - ref_loss).abs() <= 1e-6 * (4 + ref_loss.abs())).all() and loss[n] == 7.0
    half_ulp, tiny = EPS[torch.float32]
    assert ((x.double() - ref_g).abs() <= half_ulp * ref_g.abs() + 6e-6 * p + tiny).all()


# a lane takes 8 elements, a workgroup 1024
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n_h,n_w", [(1, 1), (7, 9), (8, 1023), (1024, 1025), (3001, 70_003)])
def test_both_gradients_scaled(dev, n_h, n_w, dtype):
    gen = torch.Generator(device=dev).manual_seed(n_h)
    grad_h = torch.randn(n_h, generator=gen, device=dev).to(dtype)
    grad_w = torch.randn(n_w, generator=gen, device=dev)
    up, count = torch.tensor(3.0, device=dev), torch.tensor(7.0, device=dev)
    gh, gw = kernels.ce_scale(up, count, grad_h, grad_w)
    scale = up / count
    assert torch.equal(gh, (grad_h.float() * scale).to(dtype)) and torch.equal(gw, (grad_w * scale).to(dtype))


def test_more_gradients_than_one_launch_scales(dev):
    """A launch scales 2^34 elements; here the hidden gradient alone has more,
    and a little weight gradient stands before it."""
    n = (1 << 34) + 3 * 1024 + 5
    if torch.cuda.mem_get_info(dev)[0] < 5 * n:
        pytest.skip("needs 80 GiB of free GPU memory")
    grad_h = torch.ones(n, dtype=torch.bfloat16, device=dev)
    grad_h[-4000:] = torch.arange(4000, device=dev).bfloat16()
    grad_w = torch.arange(1000, device=dev, dtype=torch.float32)
    gh, gw = kernels.ce_scale(torch.tensor(3.0, device=dev), torch.tensor(2.0, device=dev), grad_h, grad_w)
    assert torch.equal(gw, (grad_w * 1.5).bfloat16())
    assert torch.equal(gh[-4000:], (grad_h[-4000:].float() * 1.5).bfloat16())
    assert all(bool((part == 1.5).all()) for part in gh[:-4000].split(1 << 31))


def exact(h, w, y, scale):
    h, w = h.detach().double().requires_grad_(True), w.detach().double().requires_grad_(True)
    loss = torch.nn.functional.cross_entropy(h @ w.t(), y)
    (scale * loss).backward()
    return loss.detach(), h.grad, w.grad


def rel(a, b):
    return ((a.double() - b).norm() / b.norm()).item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,h,v,chunk", [(1, 64, 16, 0), (300, 72, 1003, 128), (300, 72, 1003, 0), (65, 256, 32_001, 7),
                                         (129, 512, 50_257, 0)])
def test_loss_and_gradients_no_further_off_than_torch_operations(dev, monkeypatch, n, h, v, chunk, dtype):
    """The kernels' loss and gradients against float64, beside those of the
    same steps as torch operations: within the type's rounding, and no further
    off (a tenth allowed: both round the same values in another order)."""
    gen = torch.Generator(device=dev).manual_seed(n + v)
    hid = torch.randn(n, h, generator=gen, device=dev).to(dtype)
    wgt = (torch.randn(v, h, generator=gen, device=dev) * 0.05).to(dtype)
    y = torch.randint(0, v, (n,), generator=gen, device=dev)
    y[n - n // 8:] = -100

    def run():
        a, b = hid.clone().requires_grad_(True), wgt.clone().requires_grad_(True)
        loss = chunked_linear_cross_entropy(a, b, y, chunk_rows=chunk)
        (3.0 * loss).backward()
        return loss.detach(), a.grad, b.grad

    got = run()
    monkeypatch.setattr(fused_ce, "_kernels_take", lambda *a: False)
    plain = run()
    ref = exact(hid, wgt, y, 3.0)
    tol = {torch.bfloat16: 1e-2, torch.float16: 2e-3, torch.float32: 1e-5}[dtype]
    for k, (a, p, r) in enumerate(zip(got, plain, ref)):
        assert a.dtype == p.dtype and a.shape == p.shape
        assert rel(a, r) <= tol, k
        assert rel(a, r) <= 1.1 * rel(p, r) + 1e-6, k


def test_strided_inputs_side_stream_and_repeated_backward(dev):
    """Transposed hidden states and a strided weight on a side stream; the
    saved gradients survive a second backward through the same loss."""
    gen = torch.Generator(device=dev).manual_seed(2)
    hid = torch.randn(96, 40, generator=gen, device=dev).bfloat16().t()           # [40, 96]
    wgt = (torch.randn(501, 192, generator=gen, device=dev) * 0.05).bfloat16()[:, ::2]
    y = torch.randint(0, 501, (80,), generator=gen, device=dev)[::2]
    a, b = hid.detach().requires_grad_(True), wgt.detach().requires_grad_(True)
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        loss = chunked_linear_cross_entropy(a, b, y)
        g1 = torch.autograd.grad(loss, (a, b), retain_graph=True)
        g2 = torch.autograd.grad(loss, (a, b))
    st.synchronize()
    ref = exact(hid, wgt, y, 1.0)
    assert rel(loss, ref[0]) < 1e-3
    for x1, x2, r in zip(g1, g2, ref[1:]):
        assert torch.equal(x1, x2) and rel(x1, r) < 1e-2


@pytest.mark.parametrize("n,chunk", [(40, 0), (300, 128)])   # weight gradient in the backward, in the forward
@pytest.mark.parametrize("pre_dispatch", [False, True])
def test_a_traced_graph_computes_on_its_own_inputs(dev, n, chunk, pre_dispatch):
    """Forward and backward recorded by ``make_fx`` on real tensors and run on
    other inputs: what these give eagerly, to the type's rounding."""
    def inputs(seed):
        gen = torch.Generator(device=dev).manual_seed(seed)
        return (torch.randn(n, 64, generator=gen, device=dev).bfloat16().requires_grad_(True),
                (torch.randn(500, 64, generator=gen, device=dev) * 0.05).bfloat16().requires_grad_(True),
                torch.randint(0, 500, (n,), generator=gen, device=dev))

    def step(h, w, y):
        loss = chunked_linear_cross_entropy(h, w, y, chunk_rows=chunk)
        return (loss, *torch.autograd.grad(loss, (h, w)))

    graph = make_fx(step, pre_dispatch=pre_dispatch)(*inputs(1))
    h, w, y = inputs(2)
    for got, want in zip(graph(h.detach(), w.detach(), y), exact(h, w, y, 1.0)):
        assert rel(got, want) < 1e-2


@pytest.mark.parametrize("n,chunk", [(40, 0), (300, 128)])   # weight gradient in the backward, in the forward
def test_compiled_in_one_graph(dev, n, chunk):
    """A compiler follows the call whole, to torch operations; inputs of other
    values give their own results."""
    def step(h, w, y):
        return chunked_linear_cross_entropy(h, w, y, chunk_rows=chunk)

    compiled = torch.compile(step, backend="aot_eager", fullgraph=True)
    for seed in (1, 2):
        gen = torch.Generator(device=dev).manual_seed(seed)
        h = torch.randn(n, 64, generator=gen, device=dev).bfloat16().requires_grad_(True)
        w = (torch.randn(500, 64, generator=gen, device=dev) * 0.05).bfloat16().requires_grad_(True)
        y = torch.randint(0, 500, (n,), generator=gen, device=dev)
        loss = compiled(h, w, y)
        got = (loss.detach(), *torch.autograd.grad(loss, (h, w)))
        for x, r in zip(got, exact(h, w, y, 1.0)):
            assert rel(x, r) < 1e-2


@pytest.mark.parametrize("n,chunk", [(40, 0), (300, 128)])   # weight gradient in the backward, in the forward
def test_backward_of_a_batch_of_gradients_forward_mode_and_a_negated_one(dev, n, chunk):
    """What the backward is called with can be more than its memory: a batch
    (``is_grads_batched``, ``torch.func.vmap``), a dual tensor, a negated view."""
    gen = torch.Generator(device=dev).manual_seed(4)
    h = torch.randn(n, 64, generator=gen, device=dev).bfloat16().requires_grad_(True)
    w = (torch.randn(500, 64, generator=gen, device=dev) * 0.05).bfloat16().requires_grad_(True)
    y = torch.randint(0, 500, (n,), generator=gen, device=dev)
    loss = chunked_linear_cross_entropy(h, w, y, chunk_rows=chunk)

    def back(up, **kw):
        return torch.autograd.grad(loss, (h, w), grad_outputs=up, retain_graph=True, **kw)

    one = back(torch.ones((), device=dev))
    ups = torch.tensor([1.0, 2.0, -4.0], device=dev)
    for batch in (back(ups, is_grads_batched=True), torch.func.vmap(back)(ups)):
        for got, want in zip(batch, one):
            for k, up in enumerate(ups.tolist()):   # powers of two: the same sums, perhaps in another order
                assert rel(got[k], up * want.double()) <= 2.0 ** -7
    with torch.autograd.forward_ad.dual_level():
        dual = back(torch.autograd.forward_ad.make_dual(ups[0], ups[1]))
        for got, want in zip(dual, one):
            primal, tangent = torch.autograd.forward_ad.unpack_dual(got)
            assert rel(primal, want.double()) <= 2.0 ** -7 and rel(tangent, 2.0 * want.double()) <= 2.0 ** -7
    negated = torch.tensor(0 + 1j, device=dev).conj().imag
    assert negated.is_neg() and negated.item() == -1.0
    for got, want in zip(back(negated), one):
        assert rel(got, -want.double()) <= 2.0 ** -7


def test_all_rows_ignored_is_nan(dev):
    w = torch.randn(32, 16, device=dev).bfloat16()
    loss = chunked_linear_cross_entropy(torch.randn(4, 16, device=dev).bfloat16(), w,
                                        torch.full((4,), -100, device=dev))
    assert torch.isnan(loss)


def test_loss_in_a_captured_graph(dev):
    """Forward and backward captured; four replays with eager work between."""
    gen = torch.Generator(device=dev).manual_seed(3)
    hid = torch.randn(70, 64, generator=gen, device=dev).bfloat16().requires_grad_(True)
    wgt = (torch.randn(900, 64, generator=gen, device=dev) * 0.05).bfloat16().requires_grad_(True)
    y = torch.randint(0, 900, (70,), generator=gen, device=dev)

    def step():
        loss = chunked_linear_cross_entropy(hid, wgt, y, chunk_rows=32)
        return (loss, *torch.autograd.grad(loss, (hid, wgt)))

    want = [t.detach().clone() for t in step()]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for rep in range(4):
        for t in out:
            t.detach().fill_(float(rep + 7))
        step()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for t, w in zip(out, want):
            assert torch.equal(t.detach(), w), rep
