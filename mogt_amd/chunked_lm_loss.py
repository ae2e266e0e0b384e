"""Tied-head cross-entropy without materialised logits (chunked_lm_loss.py:5-84).

``chunked_linear_cross_entropy(hidden_states, weight, labels, chunk_size=...)``
keeps the reference's contract: the mean over all B*L tokens of the
cross-entropy of ``hidden @ weight.T`` against ``labels``, computed over
``chunk_size`` token rows at a time, storing only the hidden states, labels and
weight (plus 4 bytes per token here) for a backward that recomputes the
logits.  The argument checks and their ``ValueError`` messages are the
reference's interface.

How it runs here:

* Each block of token rows is one GEMM (``rows.float() @ weight.float().T``,
  so autocast applies as in the reference's forward) followed by the HIP row
  kernels of ``csrc/lm_loss.hip``: the forward kernel reads the block once and
  writes per-row loss and log-sum-exp; the backward kernel reads the block
  once and writes ``scale * (softmax - onehot)`` as an fp32 block.
* The backward recomputes each block's logits under the autocast state the
  forward ran under (recorded at forward time), so they match the forward's
  logits, whose log-sum-exp it reuses.  The two gradient GEMMs run in fp32
  with autocast off, as the reference's backward does.
* fp32 GEMMs of blocks large enough (``_split_ok``) run on the bf16 matrix
  cores from exact three-piece splits of their fp32 operands
  (``csrc/split_gemm.hip``), the cross-entropy rows in the logits product's
  epilogue where one slice of it fills the GPU: the logits are then not
  written, and the gradient block only as its pieces.  The rest go to the BLAS
  library.
* Labels equal to -100 (F.cross_entropy's default ``ignore_index``) add zero
  loss, as in the reference's forward, and a zero gradient row; the
  reference's backward subtracts 1 at column ``vocab - 100`` for them.

``logits_cross_entropy(logits, labels)`` is the same loss for logits that are
kept anyway (MOGTForCausalLM's ``return_logits`` path, model_mogt.py:326-348):
the summed cross-entropy over the token count, on the same row kernels.
"""
from __future__ import annotations

import torch

from . import ops

IGNORE_INDEX = -100


def _token_blocks(total: int, size: int):
    """Consecutive row slices of at most ``size`` rows covering ``total``."""
    for lo in range(0, total, size):
        yield slice(lo, min(lo + size, total))


class _AutocastState:
    """The CUDA autocast setting of the forward, replayed in the backward."""

    def __init__(self):
        self.enabled = torch.is_autocast_enabled("cuda")
        self.dtype = torch.get_autocast_dtype("cuda")

    def __call__(self):
        return torch.autocast("cuda", dtype=self.dtype, enabled=self.enabled)


def _block_logits(rows: torch.Tensor, w32: torch.Tensor) -> torch.Tensor:
    """One block's logits exactly as the reference forms them (fp32 copies,
    matmul under the caller's autocast state)."""
    return rows.float().matmul(w32.t())


# Where a block's fp32 GEMMs take the split form, in multiply-adds of one of
# them (rows x vocab x D).  Small heads take the host time of their launches in
# both forms, of which the split form has fewer with its cross-entropy
# epilogues (1024 x 4000 x 256, 2^30: 305 us a forward and backward against the
# library's 344 - 374; below 2^30 the two cross) and more under autocast, whose
# logits stay with the library (2048 x 4000 x 512, 2^32: 428 against 424).
# Above, the matrix units decide (256 x 32000 x 768, 2^32.6: 355 against 682 us,
# autocast 434 against 603; 1024 rows: 788 against 2023, autocast 803 against
# 1555).
SPLIT_MIN_MACS = 1 << 30
SPLIT_MIN_MACS_AUTOCAST = 6_000_000_000

# Few rows against a weight that is split (not bf16) and past the caches: both
# forms are bound by reading it, and the split form moves it as three pieces that
# it first writes, forward and backward.  bf16 / fp32 hidden states, library over
# split form: 128256 x 2048: 96 rows 0.82 / 0.69, 160 rows 1.32 / 1.07; 128256 x
# 4096: 128 rows 0.92 / 0.74, 160 rows 1.07 / 0.83, 400 rows 1.96 / 1.41; 128000 x
# 512: 48 rows 0.94 / 0.79, 96 rows 1.39 / 1.13.  At 32000 x 768 (2^24.6) 48 rows
# gain already (1.73 / 1.34).
SPLIT_CACHED_WEIGHT = 1 << 25   # elements


def _split_min_rows(V: int, D: int, hidden: torch.dtype, weight: torch.dtype) -> int:
    if weight == torch.bfloat16 or V * D <= SPLIT_CACHED_WEIGHT:
        return 1
    return max(64, D // 16) if hidden == torch.bfloat16 else max(96, D // 12)


def _span_ok(rows: int, ld: int) -> bool:
    """Whether an operand of ``rows`` rows of stride ``ld`` stays within the
    kernels' 32-bit byte offsets, a block of 256 rows across the contraction and
    all of it along (``mogt_split_gemm``'s limits)."""
    return max(256, ops.split_pad(rows) + ops.SPLIT_K) * ld * 2 < 1 << 31


def _split_ok(rows: torch.Tensor, weight: torch.Tensor, chunk: int, autocast: bool) -> bool:
    """Whether this head's fp32 GEMMs run from bf16 pieces: tensors on the GPU,
    a contraction of whole stages, a first block large enough to gain, and the
    gradient block, weight and hidden rows within the kernels' offsets."""
    n, D = min(rows.shape[0], chunk), rows.shape[1]
    V = weight.shape[0]
    return (rows.is_cuda and weight.is_cuda and rows.device == weight.device and D % ops.SPLIT_K == 0
            and n * V * D >= (SPLIT_MIN_MACS_AUTOCAST if autocast else SPLIT_MIN_MACS)
            and n >= _split_min_rows(V, D, rows.dtype, weight.dtype)
            and _span_ok(n, ops.split_pad(V)) and _span_ok(V, D) and _span_ok(n, D))


def _in_place(x: torch.Tensor) -> bool:
    """Whether the kernels can read bf16 rows where they are."""
    return (x.stride(1) == 1 and x.stride(0) % 8 == 0 and x.stride(0) >= x.shape[1]
            and _span_ok(x.shape[0], x.stride(0)) and ops._plain((x,)) and x.data_ptr() % 16 == 0)


def _pieces(x: torch.Tensor) -> torch.Tensor:
    """``x [rows, D]`` as the bf16 pieces of its fp32 value (one where it is
    bf16 already, in place if the kernels can read it there; a traced call,
    which has no pointer to look at, copies it)."""
    if x.dtype != torch.bfloat16:
        return ops.split_pieces(x.float())
    if not _in_place(x):
        # a clone, not contiguous(): that returns an x which is misaligned, or one
        # row of any stride, as it is
        x = x.clone(memory_format=torch.contiguous_format)
    return x.unsqueeze(0)


class _Head:
    """The tied head's GEMMs for one call: logits of a block of rows, and a
    block's share of the two gradients."""

    def __init__(self, rows: torch.Tensor, weight: torch.Tensor, chunk: int, autocast: _AutocastState):
        self.weight = weight
        self.autocast = autocast
        self.split = _split_ok(rows, weight, chunk, autocast.enabled)
        self._w32 = self._pieces = None

    @property
    def w32(self) -> torch.Tensor:
        if self._w32 is None:
            self._w32 = self.weight.float()
        return self._w32

    @property
    def pieces(self) -> torch.Tensor:
        if self._pieces is None:
            self._pieces = _pieces(self.weight)
        return self._pieces

    def logits(self, block: torch.Tensor) -> torch.Tensor:
        """The block's logits from the library, under the caller's autocast."""
        return _block_logits(block, self.w32)

    def loss_rows(self, block: torch.Tensor, targets: torch.Tensor):
        """The block's per-row loss and log-sum-exp."""
        if self.split and not self.autocast.enabled:
            return ops.split_head_loss(_pieces(block), self.pieces, self.weight.shape[1], targets,
                                       ignore_index=IGNORE_INDEX)
        return ops.lm_ce_forward(self.logits(block), targets, ignore_index=IGNORE_INDEX)

    def new_weight_grad(self) -> torch.Tensor:
        # the split form writes it with the first block
        make = torch.empty if self.split else torch.zeros
        return make(self.weight.shape, dtype=torch.float32, device=self.weight.device)

    def backward(self, targets, lse, scale, block, d_rows, d_w32, first: bool) -> None:
        """d_rows = g @ weight and d_w32 += g^T @ block in fp32, for the gradient
        g of the block's logits, recomputed under the forward's autocast state.
        Only library calls stand inside the autocast regions: a graph cannot be
        traced with this library's functions there."""
        logits = None
        if not self.split or self.autocast.enabled:
            with self.autocast():
                logits = self.logits(block)
        if not self.split:
            # fp32 gradient block, whatever the logits' dtype
            g = ops.lm_ce_grad(logits, targets, lse, scale, ignore_index=IGNORE_INDEX)
            with torch.autocast("cuda", enabled=False):
                d_rows.copy_(g.matmul(self.w32))
                d_w32.addmm_(g.t(), block.float())
            return
        V, D = self.weight.shape
        rows = _pieces(block)
        if logits is None:
            g = ops.split_head_grad_pieces(rows, self.pieces, D, targets, lse, scale, ignore_index=IGNORE_INDEX)
        else:
            g = ops.lm_ce_grad_pieces(logits, targets, lse, scale, ignore_index=IGNORE_INDEX)
        direct = d_rows.dtype in (torch.float32, torch.bfloat16) and d_rows.is_contiguous()
        dh = d_rows if direct else torch.empty(d_rows.shape, dtype=torch.float32, device=d_rows.device)
        ops.split_gemm_(dh, g, self.pieces, V, k_slow_b=True)
        if not direct:
            d_rows.copy_(dh)
        ops.split_gemm_(d_w32, g, rows, block.shape[0], k_slow_a=True, k_slow_b=True, accumulate=not first)


class _NotTwiceDifferentiable(torch.autograd.Function):
    """Gradients that a second differentiation refuses (through ``grads`` as well
    as through ``inputs``) instead of taking them as constants."""

    @staticmethod
    def forward(ctx, n_inputs: int, *tensors):
        return tuple(g.view_as(g) for g in tensors[n_inputs:])

    @staticmethod
    def backward(ctx, *grad_outputs):
        raise RuntimeError("chunked_linear_cross_entropy has no second derivative")


class _ChunkedLinearCrossEntropy(torch.autograd.Function):
    """chunked_lm_loss.py:5-72 on the HIP cross-entropy rows."""

    @staticmethod
    def forward(ctx, hidden_states, weight, labels, chunk_size: int):
        if hidden_states.ndim != 3:
            raise ValueError("hidden_states must be [B, L, D]")
        if labels.shape != hidden_states.shape[:2]:
            raise ValueError("labels must be [B, L]")
        if weight.ndim != 2 or weight.shape[1] != hidden_states.shape[-1]:
            raise ValueError("weight must be [V, D]")
        chunk_size = int(chunk_size)
        if chunk_size <= 0:
            raise ValueError("chunk_size must be positive")

        n_tok = labels.numel()
        rows = hidden_states.reshape(n_tok, hidden_states.shape[-1])
        targets = labels.reshape(n_tok).to(torch.int64).contiguous()
        ctx.autocast = _AutocastState()
        head = _Head(rows, weight, chunk_size, ctx.autocast)
        per_row = torch.empty(n_tok, dtype=torch.float32, device=hidden_states.device)
        lse = torch.empty(n_tok, dtype=torch.float32, device=hidden_states.device)
        with torch.no_grad():
            for sl in _token_blocks(n_tok, chunk_size):
                loss_rows, lse_rows = head.loss_rows(rows[sl], targets[sl])
                per_row[sl] = loss_rows
                lse[sl] = lse_rows
        ctx.save_for_backward(hidden_states, weight, targets, lse)
        ctx.chunk_size = chunk_size
        return per_row.sum() / n_tok

    @staticmethod
    def backward(ctx, grad_output):
        hidden_states, weight, targets, lse = ctx.saved_tensors
        n_tok = targets.numel()
        rows = hidden_states.reshape(n_tok, hidden_states.shape[-1])
        scale = (grad_output.float() / n_tok).reshape(1)
        head = _Head(rows, weight, ctx.chunk_size, ctx.autocast)
        d_rows = torch.empty_like(rows)
        d_w32 = head.new_weight_grad()
        with torch.no_grad():
            for i, sl in enumerate(_token_blocks(n_tok, ctx.chunk_size)):
                head.backward(targets[sl], lse[sl], scale, rows[sl], d_rows[sl], d_w32, first=i == 0)
        d_hidden, d_weight = d_rows.view_as(hidden_states), d_w32.to(weight.dtype)
        if torch.is_grad_enabled() and not torch.compiler.is_compiling():   # create_graph
            d_hidden, d_weight = _NotTwiceDifferentiable.apply(3, hidden_states, weight, grad_output, d_hidden, d_weight)
        return d_hidden, d_weight, None, None


def chunked_linear_cross_entropy(hidden_states, weight, labels, *, chunk_size: int):
    """Memory-efficient CE for tied LM heads (chunked_lm_loss.py:75-84): only the
    hidden states, labels and LM weight are kept; logits are recomputed chunk by
    chunk in backward."""
    return _ChunkedLinearCrossEntropy.apply(hidden_states, weight, labels, int(chunk_size))


class _LogitsCrossEntropy(torch.autograd.Function):
    """sum of per-row cross-entropy / row count, for logits the caller keeps."""

    @staticmethod
    def forward(ctx, logits, labels):
        targets = labels.to(torch.int64).contiguous()
        block = logits if logits.stride(-1) == 1 else logits.contiguous()
        loss_rows, lse = ops.lm_ce_forward(block, targets, ignore_index=IGNORE_INDEX)
        ctx.save_for_backward(block, targets, lse)
        return loss_rows.sum() / max(targets.numel(), 1)

    @staticmethod
    def backward(ctx, grad_output):
        block, targets, lse = ctx.saved_tensors
        scale = (grad_output.float() / max(targets.numel(), 1)).reshape(1)
        grad = block.clone()
        ops.lm_ce_backward_(grad, targets, lse, scale, ignore_index=IGNORE_INDEX)
        return grad, None


def logits_cross_entropy(logits: torch.Tensor, labels: torch.Tensor) -> torch.Tensor:
    """Summed cross-entropy of ``logits [N, V]`` against ``labels [N]`` divided by
    N (the chunked loss of model_mogt.py:326-348 with the logits kept); labels
    of -100 add zero."""
    if logits.ndim != 2 or labels.shape != logits.shape[:1]:
        raise ValueError("logits must be [N, V] and labels [N]")
    return _LogitsCrossEntropy.apply(logits, labels)
