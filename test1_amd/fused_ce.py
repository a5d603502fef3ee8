"""Chunked linear + cross entropy for the output unit: the loss of
``cross_entropy(hidden @ weight.T, labels)`` without materialising the
[N, V] logits.

The reference's output unit uses a fused linear-cross-entropy kernel when one
is installed (slide_fsdp.py:57-63, 85-97: ``LigerFusedLinearCrossEntropyLoss``,
mean reduction, no logits returned) and full logits + ``nn.CrossEntropyLoss``
otherwise.  This is the fused variant built from hipBLASLt GEMMs: rows are
processed in chunks of ``chunk_rows``; for each chunk the logits are formed,
one kernel (``csrc/sf_ce.hip``) turns them into the chunk's loss terms and, in
place, into ``softmax - onehot``, and since the step's backward follows at
once, the gradients with respect to the hidden rows and the weight are formed
right away (as the fused kernel does) and only scaled in the backward; the
weight's of few tokens is formed there, where its scaling costs nothing.  Peak
extra memory is one chunk of logits with its hidden rows transposed and up to
128 MiB of partial sums, plus an fp32 weight gradient, instead of the [N, V]
logits in bf16 and fp32 and their gradient.

Numerics: logsumexp, softmax and the loss are fp32; the logits are the bf16
GEMM's output widened, as ``nn.CrossEntropyLoss`` on bf16 logits sees them;
the gradient of the logits is rounded to bf16 for the two gradient GEMMs and
the weight gradient stays in fp32 until the backward has scaled it.  Rows whose
label is ``ignore_index`` contribute nothing; the mean is over the other rows
(NaN if there are none, as ``nn.CrossEntropyLoss``).

On a host, and for inputs the kernels do not take (``_kernels_take``), the
same steps run as torch operations.
"""

from __future__ import annotations

import torch

from . import kernels


_DTYPES = (torch.bfloat16, torch.float16, torch.float32)
_PLAIN = (torch.Tensor, torch.nn.Parameter)


def _traced() -> bool:
    """Whether something records the operations of this call: a compiler, a
    JIT trace, or a dispatch mode, ``make_fx``'s among them, to which the
    tensors themselves are plain ones.  What is called through pointers is not
    in such a record: a graph made of it would return memory that nothing
    fills.  Asked first: a compiler does not follow the other questions."""
    return (torch.compiler.is_compiling() or torch._C._is_tracing() or torch._C._len_torch_dispatch_stack() > 0
            or torch._ops._len_torch_dispatch_stack_pre_dispatch() > 0)


_PLAIN_KEYS = 0
for _key in ("CPU", "CUDA", "ADInplaceOrView", "AutogradCPU", "AutogradCUDA", "AutocastCPU", "AutocastCUDA"):
    _PLAIN_KEYS |= torch._C.DispatchKeySet(getattr(torch._C.DispatchKey, _key)).raw_repr()


def _memory_is_value(t: torch.Tensor) -> bool:
    """Whether a kernel that reads ``t``'s memory gets all of it: no batch of a
    vmap, no wrapper of a function transform, no pending negation (such tensors
    are of the plain type and differ in their dispatch keys), and no
    forward-mode derivative beside it."""
    return torch._C._dispatch_keys(t).raw_repr() & ~_PLAIN_KEYS == 0 and torch.autograd.forward_ad._current_level < 0


def _kernels_take(hidden: torch.Tensor, weight: torch.Tensor, labels: torch.Tensor) -> bool:
    """Inputs the HIP kernels run on: one GPU, one float type, int64 labels, at
    least one row.  Left to torch: what its operations refuse by themselves
    (mixed types or devices, other label types), the empty cases, autocast to
    another type (it would round the products), a traced call, and tensor
    subclasses."""
    return (not _traced()
            and hidden.device.type == "cuda" and weight.device == hidden.device and labels.device == hidden.device
            and hidden.dtype in _DTYPES and weight.dtype == hidden.dtype and labels.dtype == torch.int64
            and hidden.numel() > 0 and weight.numel() > 0 and weight.shape[0] < 1 << 31
            and hidden.shape[0] < 1 << 31
            and not (torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") != hidden.dtype)
            and type(hidden) in _PLAIN and type(weight) in _PLAIN and type(labels) in _PLAIN)


_PARTS_VOCAB = 16384   # the shortest vocabulary that ``_vocabulary_parts`` divides
_PARTS_TILES = 64      # and the most tiles of a product


def _tiles(rows: int, hidden_size: int) -> int:
    return -(-rows // 256) * -(-hidden_size // 256)


def _row_elements(vocab: int, element_size: int) -> int:
    """Elements from a row of logits to the next: rows 128 bytes apart or a
    multiple of it keep the kernel's 128-bit accesses and the products' operand
    loads aligned for any vocabulary.  Vocabularies under 64 are not padded
    beyond what the kernel needs, 16 bytes (fp32: nothing)."""
    unit = 64 if vocab >= 64 else 8 if element_size == 2 else 1
    return -(-vocab // unit) * unit


def auto_chunk_rows(tokens: int, vocab: int, hidden_size: int, element_size: int) -> int:
    """Rows per chunk when the caller names none.  One chunk where possible:
    the products run at 0.80-1.47 PFLOP/s on 523 rows against 4092 (hidden
    4096, vocabulary 128256), and every chunk after the first reads and writes
    the whole fp32 weight gradient again.  What a chunk may take beside that
    gradient is what the torch operations take at their peak with chunks of 256
    MiB of fp32 logits.  16-bit: the next chunk's logits, a temporary of
    ``logsumexp`` and the 16-bit gradient of the chunk before, 640 MiB, or that
    gradient and a 16-bit product of the weight gradient's size; here a chunk
    has its logits, its hidden rows transposed, and partial sums of at most 128
    MiB (``_vocabulary_parts``), which the first chunk finds in the weight
    gradient's memory and a short last one behind its logits.  fp32: logits, and
    a product that is not made here."""
    if element_size == 4:
        return max(1, hidden_size, (256 << 20) // (4 * vocab))
    ld = _row_elements(vocab, 2)
    if 2 * (ld + hidden_size) * (tokens + 63) <= 512 << 20:   # with any partial sums
        return max(1, tokens)
    peak = max(640 << 20, (128 << 20) + 2 * vocab * hidden_size)
    rows = peak // (2 * (ld + hidden_size))
    # the fewest rows of a chunk whose partial sums have to be allocated
    least = tokens if tokens <= rows else rows - (64 << 20) // ld
    if (vocab >= _PARTS_VOCAB and _tiles(max(1, least), hidden_size) <= _PARTS_TILES
            and not (tokens <= rows and 16 * tokens <= vocab)):
        rows = (peak - (128 << 20)) // (2 * (ld + hidden_size))
    # equal chunks, whole tiles of 256 rows if that fits, else whole 64s, to
    # which the transposed rows are padded (8192 x 4096 x 128256 in 4096 + 4096
    # 20.8 ms, in 4416 + 3776 26.1)
    if rows < 64:
        return max(1, rows)
    rows = rows // 64 * 64
    if tokens > rows:
        equal = -(-tokens // -(-tokens // rows))
        rows = next(r for r in (-(-equal // 256) * 256, -(-equal // 64) * 64) if r <= rows)
    return rows


def _transposed_hidden_pays(rows: int, hidden: torch.Tensor, vocab: int) -> bool:
    """Whether the weight gradient's product of a chunk of ``rows`` takes the
    hidden rows transposed and padded (``kernels.ce_hidden``): a library's
    kernel with one operand laid out along the sum is a tenth to a third
    faster, measured from 34 GFLOP (25 us) up, where the transposing launch
    (4 us and up to a half percent of the product) is small beside that.  us,
    tokens x hidden x vocabulary, as they are | transposed and padded: 777 x
    1024 x 32000 80 | 69, 127 x 4096 x 128256 708 | 474, 4092 x 4096 x 128256
    4198 | 3490; below, 510 x 512 x 4096 21.8 | 22.2.  Only rows that lie one
    behind the other: what is laid out along the sum already needs nothing.
    And only where the transposed rows take no more than the torch operations'
    fp32 logits with their temporary, or 16-bit product, beside the logits."""
    h = hidden.shape[1]
    return (hidden.element_size() == 2 and hidden.stride(1) == 1 and hidden.stride(0) >= h
            and 2 * rows * h * vocab >= 1 << 35 and rows * h <= max(3 * rows * vocab, vocab * h))


def _vocabulary_parts(rows: int, weight: torch.Tensor, own: bool = False) -> int:
    """Parts in which the hidden gradient's product of a chunk of ``rows`` sums
    over the vocabulary (1: the product as it is).  The library sums each of
    its 256 x 256 tiles in one workgroup; with as many parts as give every
    compute unit one, at most 16 (powers of two: three, five or six parts ran
    slower than two, four or eight), us, one product | parts before they are
    added up, tokens x hidden x vocabulary: 1023 x 4096 x 128256 1461 | 807,
    510 x 4096 x 32000 299 | 134, 777 x 1024 x 32000 174 | 69, 4000 x 768 x
    30522 287 | 203.  Above 64 tiles a shape gains or loses (whole calls: 2046
    x 2560 x 151936, 80 tiles, 5776 | 5362, of a 60000 vocabulary 1863 | 1989,
    3500 x 1536 x 152064, 84 tiles, 6617 | 7454), as it does with short sums
    (the product alone, 510 x 512 x 4096 19.2 | 17.9).  The parts are at most
    512 tiles of fp32.  Adding them up is a launch more, which makes a call that
    the host's 240 us bound 20 to 35 us slower (300 x 1024 x 17000, 64 x 1024 x
    30000, 250 x 1024 x 32000); so only where the call moves 800 MiB or its
    products take 34 GFLOP each (whole calls: 4000 x 64 x 30522, 1.2 GB, 386 |
    312; 777 x 1024 x 32000, 51 GFLOP, 380 | 286; 4092 x 1024 x 50257 in chunks
    of 256 6073 | 3654).  ``own``: the weight gradient is formed from its factors
    in the backward (``_own_weight_grad``) and moves less, which leaves the sum
    itself as the larger part: one element of it takes the time of 6 kB, and the
    line is at 700 MB (whole calls on a host that needs 180 us for one, and on
    one that needs 265; below, 64 x 5120 x 16384 196 | 192, 272 | 300, 250 x 4096
    x 16384 217 | 196, 260 | 295; above, 100 x 2560 x 32000 258 | 191, 271 | 297,
    200 x 1024 x 60000 351 | 225, 356 | 294, 100 x 512 x 100000 369 | 273, 371 |
    292, 200 x 256 x 152064 460 | 217, 463 | 299).  Operands that start on
    16-byte boundaries only."""
    v, h = weight.shape
    tiles = _tiles(rows, h)
    if (weight.element_size() != 2 or tiles > _PARTS_TILES or v < _PARTS_VOCAB or h % 8 != 0 or not weight.is_contiguous()
            or weight.data_ptr() % 16 != 0):
        return 1
    # the weight read twice, its gradient written (in fp32 and rounded, or once);
    # the logits written, turned into their gradient in place and read twice
    moved = ((6 * h if own else 14 * h) + 10 * rows) * v
    if moved + 6000 * v < 700_000_000 if own else moved < 800 << 20 and 2 * rows * h * v < 1 << 35:
        return 1
    parts = 2
    while parts < 16 and parts * tiles < 256:
        parts *= 2
    return parts


def _grad_hidden(g: torch.Tensor, ld: int, weight: torch.Tensor, own: bool, out: torch.Tensor, scratch) -> None:
    """out = g @ weight for the gradient of a chunk's logits, ``ld`` elements
    from row to row.  ``own``: see ``_vocabulary_parts``.  ``scratch(elements)``:
    fp32 memory for the parts."""
    n, v = g.shape
    h = weight.shape[1]
    nparts = _vocabulary_parts(n, weight, own)
    if nparts == 1:
        torch.mm(g, weight, out=out)
        return
    part = v // nparts // 8 * 8
    parts = scratch(nparts * n * h).view(nparts, n, h)
    torch.bmm(g.as_strided((nparts, n, part), (part, ld, 1)), weight[:nparts * part].view(nparts, part, h),
              out_dtype=torch.float32, out=parts)
    kernels.ce_grad_hidden(g, weight, parts, out)


def _own_weight_grad(n: int, hidden: torch.Tensor) -> bool:
    """Whether the weight gradient of ``n`` tokens in one chunk is formed in the
    backward, from the gradient of the logits and the transposed hidden rows,
    scaled as it is formed (``kernels.ce_weight_grad``): up to 256 tokens, whose
    factors fit the registers (us a call, as a product into fp32 and a scaling
    | so, tokens x hidden x vocabulary: 256 x 4096 x 128256 1757 | 1555, 4 x 4096
    x 128256 1461 | 847; with half the columns a wave 300 x 2560 x 50257 591 |
    658), and where they are no larger than the fp32 gradient that would be
    kept instead."""
    h = hidden.shape[1]
    return (hidden.element_size() == 2 and n <= 256 and -(-n // 64) * 64 <= 2 * h and h % 8 == 0
            and hidden.stride(1) == 1 and hidden.stride(0) >= h)


def _forward_kernels(ctx, hidden: torch.Tensor, weight: torch.Tensor, labels: torch.Tensor, ignore_index: int,
                     chunk_rows: int) -> torch.Tensor:
    n, h = hidden.shape
    v = weight.shape[0]
    dev = hidden.device
    labels = labels.contiguous()
    grad_hidden = torch.empty((n, h), dtype=hidden.dtype, device=dev)
    row_loss = torch.empty(n, dtype=torch.float32, device=dev)
    loss = torch.empty((), dtype=torch.float32, device=dev)
    n_valid = torch.empty((), dtype=torch.float32, device=dev)
    step = max(1, min(n, int(chunk_rows)))
    ld = _row_elements(v, hidden.element_size())
    own = step == n and _own_weight_grad(n, hidden)
    transposed = own or _transposed_hidden_pays(step, hidden, v)
    # a chunk's rows, as many as the weight gradient's product sums over
    height = (lambda m: -(-m // 64) * 64) if transposed else (lambda m: m)
    buf = torch.empty((height(step), ld), dtype=hidden.dtype, device=dev)
    hidden_t = torch.empty(h * height(step), dtype=hidden.dtype, device=dev) if transposed else None
    grad_weight = None if own else torch.empty((v, h), dtype=torch.float32, device=dev)
    wt = weight.t()
    f32_out = {} if hidden.dtype == torch.float32 else dict(out_dtype=torch.float32)
    for s in range(0, n, step):
        e = min(n, s + step)
        hc = hidden[s:e]
        g = buf[:e - s, :v]
        torch.mm(hc, wt, out=g)
        kernels.ce_rows_(g, labels[s:e], ignore_index, row_loss[s:e])

        def scratch(k: int) -> torch.Tensor:
            # the weight gradient's memory is free until its first product, the
            # logits' behind a chunk shorter than the others
            if s == 0 and not own and k <= grad_weight.numel():
                return grad_weight.view(-1)[:k]
            behind = buf[height(e - s):].view(-1)
            if 2 * k <= behind.numel():
                return behind[:2 * k].view(torch.float32)
            return torch.empty(k, dtype=torch.float32, device=dev)

        _grad_hidden(g, ld, weight, own, grad_hidden[s:e], scratch)
        if transposed:
            pad = height(e - s)
            ht = hidden_t[:h * pad].view(h, pad)
            kernels.ce_hidden(hc, ht, buf[:pad])
            g, hc = buf[:pad, :v], ht.t()
        if own:
            break
        if s == 0:
            torch.mm(g.t(), hc, **f32_out, out=grad_weight)
        else:
            torch.addmm(grad_weight, g.t(), hc, **f32_out, out=grad_weight)
    kernels.ce_loss(row_loss, labels, ignore_index, loss, n_valid)
    if own:
        ctx.vocab = v
        ctx.save_for_backward(grad_hidden, buf, hidden_t.view(h, -1), n_valid)
    else:
        ctx.save_for_backward(grad_hidden, grad_weight, n_valid)
    return loss


def _torch_chunk_rows(vocab: int) -> int:
    return max(1, (256 << 20) // (4 * vocab))


def _forward_torch(ctx, hidden: torch.Tensor, weight: torch.Tensor, labels: torch.Tensor, ignore_index: int,
                   chunk_rows: int) -> torch.Tensor:
    n, h = hidden.shape
    v = weight.shape[0]
    dev = hidden.device
    grad_hidden = torch.empty_like(hidden)
    grad_weight = torch.zeros((v, h), dtype=torch.float32, device=dev)
    loss_sum = torch.zeros((), dtype=torch.float32, device=dev)
    valid_all = labels != ignore_index
    n_valid = valid_all.sum().to(torch.float32)
    wt = weight.t()
    for s in range(0, n, max(1, int(chunk_rows))):
        e = min(n, s + int(chunk_rows))
        hc = hidden[s:e]
        yc = labels[s:e]
        valid = valid_all[s:e]
        ysafe = torch.where(valid, yc, torch.zeros_like(yc))
        logits = torch.mm(hc, wt).float()                       # [C, V], widened bf16 GEMM output
        lse = torch.logsumexp(logits, dim=1)
        target = logits.gather(1, ysafe.unsqueeze(1)).squeeze(1)
        loss_sum += torch.where(valid, lse - target, torch.zeros_like(lse)).sum()
        logits.sub_(lse.unsqueeze(1)).exp_()                    # softmax, in place
        rows = torch.arange(e - s, device=dev)
        logits[rows, ysafe] -= 1.0                              # - onehot
        logits.mul_(valid.unsqueeze(1).to(logits.dtype))        # ignored rows: no gradient
        g = logits.to(hidden.dtype)
        del logits
        grad_hidden[s:e] = torch.mm(g, weight)
        grad_weight.add_(torch.mm(g.t(), hc))
    ctx.save_for_backward(grad_hidden, grad_weight, n_valid)
    return loss_sum / n_valid


def _saved_plain(t: torch.Tensor, dtype: torch.dtype, device: torch.device) -> bool:
    return (type(t) is torch.Tensor and t.dtype == dtype and t.device == device and t.numel() > 0 and t.is_contiguous()
            and t.data_ptr() % 16 == 0)


class ChunkedLinearCrossEntropy(torch.autograd.Function):
    @staticmethod
    def forward(ctx, hidden: torch.Tensor, weight: torch.Tensor, labels: torch.Tensor, ignore_index: int,
                chunk_rows: int) -> torch.Tensor:
        if hidden.dim() != 2 or weight.dim() != 2 or hidden.shape[1] != weight.shape[1]:
            raise ValueError("chunked linear cross entropy: hidden [N, H] and weight [V, H] expected")
        if labels.shape != hidden.shape[:1]:
            raise ValueError("chunked linear cross entropy: one label per hidden row expected")
        ctx.weight_dtype = weight.dtype
        take = _kernels_take(hidden, weight, labels)
        if chunk_rows <= 0:
            chunk_rows = (auto_chunk_rows(hidden.shape[0], weight.shape[0], weight.shape[1], hidden.element_size()) if take
                          else _torch_chunk_rows(weight.shape[0]))
        if not take:
            return _forward_torch(ctx, hidden, weight, labels, ignore_index, chunk_rows)
        with torch.cuda.device(hidden.device):
            return _forward_kernels(ctx, hidden, weight, labels, ignore_index, chunk_rows)

    @staticmethod
    def backward(ctx, grad_loss: torch.Tensor):
        grad_hidden, *weight_parts, n_valid = ctx.saved_tensors
        # The kernels take what the forward saved, unless hooks brought it back
        # otherwise or the backward itself is differentiated, batched or traced.
        dtype, dev = ctx.weight_dtype, grad_hidden.device
        part = dtype if len(weight_parts) == 2 else torch.float32
        if (not _traced() and dev.type == "cuda" and dtype in _DTYPES and _saved_plain(grad_hidden, dtype, dev)
                and _saved_plain(n_valid, torch.float32, dev) and all(_saved_plain(t, part, dev) for t in weight_parts)
                and type(grad_loss) is torch.Tensor and grad_loss.device == dev and grad_loss.dtype == torch.float32
                and not (torch.is_grad_enabled() and grad_loss.requires_grad) and _memory_is_value(grad_loss)):
            with torch.cuda.device(grad_hidden.device):
                if len(weight_parts) == 2:
                    g, hidden_t = weight_parts
                    return (*kernels.ce_weight_grad(grad_loss, n_valid, grad_hidden, g, ctx.vocab, hidden_t),
                            None, None, None)
                return (*kernels.ce_scale(grad_loss, n_valid, grad_hidden, weight_parts[0]), None, None, None)
        if len(weight_parts) == 2:
            g, hidden_t = weight_parts
            grad_weight = g[:, :ctx.vocab].t().float() @ hidden_t.t().float()
        else:
            grad_weight = weight_parts[0]
        scale = (grad_loss.to(torch.float32) / n_valid)
        gh = (grad_hidden.to(torch.float32) * scale).to(grad_hidden.dtype)
        gw = (grad_weight * scale).to(ctx.weight_dtype)
        return gh, gw, None, None, None


def chunked_linear_cross_entropy(hidden: torch.Tensor, weight: torch.Tensor, labels: torch.Tensor,
                                 ignore_index: int = -100, chunk_rows: int = 0) -> torch.Tensor:
    """Mean cross entropy of ``hidden @ weight.T`` against ``labels``.
    ``chunk_rows`` <= 0 picks the chunks (``auto_chunk_rows`` on a GPU, else
    ~256 MiB of fp32 logits)."""
    if chunk_rows <= 0:
        chunk_rows = 0 if hidden.is_cuda else _torch_chunk_rows(weight.shape[0])
    return ChunkedLinearCrossEntropy.apply(hidden, weight, labels, int(ignore_index), int(chunk_rows))
