"""Chunked fused linear + cross-entropy on gfx950.

Same function, arguments and semantics as torchure/loss/fused_linear_ce.py:130-136:
``fused_linear_cross_entropy(hidden, weight, labels, ignore_index=-100, chunk_size=...)``
returns the mean loss over non-ignored tokens (F.cross_entropy(reduction="mean")
semantics, :22-24), computes grad_hidden and grad_weight during the forward pass
(:42-58) and scales them in place by grad_out / n_valid in backward (:94-127).

Per chunk of rows:
  logits = h @ W^T                  bf16 GEMM: tm_ce_logits_ld_bf16, this package's MFMA GEMM, for dim a
                                    multiple of 64 (torch.matmul on other shapes)
  tm_ce_rows_padded_bf16            one fused kernel: logsumexp, per-row loss and
                                    grad_logits = bf16(softmax - onehot), in place
  grad_h = grad_logits @ W          bf16 GEMM: tm_ce_grad_h_ld_bf16, a split-K MFMA GEMM with a
                                    fixed-order reduction, where grad_h_gemm_fits; hipBLASLt on
                                    other shapes
  grad_W += grad_logits^T @ h       bf16 GEMM: tm_ce_grad_w_ld_bf16, this package's MFMA GEMM, for dim
                                    a multiple of 64 (and rows too where the logits are unpadded;
                                    torch.matmul otherwise), then tm_ce_grad_w_fold into fp32
The chunk's logits are padded to whole MFMA steps: rows a multiple of 64 elements (padded_vocab)
apart and their number a multiple of 64 or 128 (padded_rows), the padding zero once they are gradients. An odd
vocabulary then keeps its rows 16-byte aligned, and any number of tokens is a whole number of
K slices for grad_W. The logits and the row kernel run over several chunks at a time
(group_chunks), the gradients chunk by chunk;
then tm_ce_mean_loss sums the per-row losses in a fixed order (deterministic).

The last chunk's bf16 grad_W is not added in forward: it waits for backward, where
tm_ce_finish adds it and applies grad_out / n_valid in the same pass. With a single
chunk (the usual case at 4 GiB of logits) the fp32 grad_W is then written once,
straight from the bf16 GEMM output (6 B per element), instead of a zero fill, an
accumulate and a scaling pass (22 B per element). With several chunks, the chunks'
bf16 grad_W wait and are added up to 8 at a time (tm_ce_grad_w_fold: one read and one
write of the fp32 grad_W per fold; a fold also starts once 4 GiB of chunks wait), and the
chunks still waiting are added together with the last in backward. The fp32 additions and
the scaling are the reference's, in the reference's order, so the bits are unchanged.

Only the gradients autograd needs are computed. With grad mode off, or no input that
requires a gradient (evaluation), the call returns the loss from the logits GEMM and
tm_ce_rows_loss_bf16, which runs the same per-row arithmetic without the gradient
write, so the loss bits are those of the training path. When only one input requires a
gradient, the other's GEMM is skipped. The reference computes both gradients whenever
the weight requires one (fused_linear_ce.py:63-93) and lets autograd drop them.

Hidden states are bf16 or fp32. fp32 inside bf16 CUDA autocast is the trainer's call
(objectives/autoregressive.py:38-44): it passes the final norm's fp32 output, for which the
reference's buffers take fp32 (:65,68) and autocast runs the products on bf16 casts. Here
hidden is cast to bf16 once (RNE, as autocast does), grad_hidden stays a bf16 GEMM output
until backward, and tm_ce_finish writes the fp32 gradient float(gh) * grad_out / n_valid
(the reference's fp32 copy and mul_, :80,120). fp32 hidden states outside autocast take the
reference's fp32 path: fp32 GEMMs on weight.to(fp32), tm_ce_rows_f32 on fp32 logits, grad_W
summed in fp32 by the product, and tm_ce_finish for the scaling of both.

Chunking: 1024 rows by default, the reference's default (:131). ``chunk_size=None`` or
``"auto"`` opts into MI355X sizing: chunks whose bf16 logits take up to 4 GiB, so that
with 288 GB of HBM the whole Qwen3 vocabulary for 8K-16K tokens fits in one chunk, the
fp32 grad_W is written once, by the backward hand-over, instead of being read and written
for every fold of 1024-row chunks, and the GEMMs get large M.
"""

from __future__ import annotations

import contextlib
import ctypes
import threading

import torch

from torchure_amd import _native
from torchure_amd.core import tables
from torchure_amd.optimizer.working import current_copy

DEFAULT_LOGITS_BYTES = 4 << 30


class CallOrder:
    """Puts the GPU work of this op's calls on one device in host call order.

    hipBLASLt's gfx950 solutions for this op's products are stream-K kernels (``SK3`` in
    their names): a persistent grid of one workgroup per CU in which workgroups spin on
    flags until other workgroups of the same launch have written their partial tiles, so
    every workgroup of the launch must be resident at once. Two such launches running at
    the same time on two streams can each hold CUs with spinning workgroups while the
    workgroups they wait for cannot be placed, and neither finishes. So each call's stream
    first waits for an event recorded at the end of the previous call's GPU work on that
    device (skipped when both run on one stream), and the host side of a call runs under a
    lock, so that calls from two host threads cannot interleave either. The event is
    always recorded before the next call waits on it, so a wait never sits in front of the
    work that signals it. GEMMs that a caller runs on other streams are not ordered by
    this; they must not overlap a call.

    ``current_stream`` and ``make_event`` are injectable so the ordering can be checked on
    the CPU with stand-in streams and events."""

    def __init__(self, current_stream=None, make_event=None):
        self._current_stream = current_stream or torch.cuda.current_stream
        self._make_event = make_event or torch.cuda.Event
        self._lock = threading.RLock()
        self._last: dict = {}  # device index -> (stream, event) of the last call there

    @contextlib.contextmanager
    def call(self, device: torch.device):
        if device.type != "cuda":  # the call raises on its argument checks; nothing to order
            yield None
            return
        key = device.index if device.index is not None else -1
        with self._lock:
            stream = self._current_stream(device)
            prev = self._last.get(key)
            if prev is not None and prev[0] != stream:
                stream.wait_event(prev[1])
            try:
                yield stream
            finally:
                done = self._make_event()
                done.record(stream)
                self._last[key] = (stream, done)


CALL_ORDER = CallOrder()


def auto_chunk_rows(n_rows: int, vocab: int, logits_bytes: int = DEFAULT_LOGITS_BYTES) -> int:
    rows = max(256, logits_bytes // (2 * vocab) // 256 * 256)
    return max(1, min(n_rows, rows))


def _fp32_hidden_under_autocast(hidden) -> bool:
    """fp32 hidden states inside bf16 CUDA autocast: the reference trainer's call (its final
    RMSNorm leaves the fp32 residual stream in fp32), where autocast runs the op's products as
    bf16 GEMMs and the hidden-state gradient stays fp32."""
    return (hidden.dtype == torch.float32 and torch.is_autocast_enabled("cuda")
            and torch.get_autocast_dtype("cuda") == torch.bfloat16)


def _checked(hidden, weight, labels, chunk_size):
    """Argument checks shared by all paths; returns (n, v, chunk rows, mode): "bf16" (bf16
    hidden), "autocast" (fp32 hidden inside bf16 autocast: bf16 products) or "fp32" (fp32 hidden
    outside autocast: fp32 products, as the reference's with w = weight.to(fp32))."""
    who = "fused_linear_cross_entropy"
    for t, what in ((hidden, "hidden"), (labels, "labels")):  # made contiguous by the caller
        tables.require_device_tensor(t, who, what)
    if weight.device.type != "cuda":  # any strides: the op works on its contiguous bf16 cast
        raise RuntimeError(f"{who}: weight must be on a ROCm GPU device, got {weight.device} "
                           "(torchure_amd has no CPU path)")
    if torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") != torch.bfloat16:
        # autocast would run the products in its dtype (the reference's GEMMs too), and the
        # row kernel reads bf16 logits
        raise NotImplementedError(
            f"{who}: CUDA autocast with {torch.get_autocast_dtype('cuda')} is not supported; the "
            "products run as bf16 GEMMs (bf16 autocast, or none)")
    if _fp32_hidden_under_autocast(hidden):
        mode = "autocast"
    elif hidden.dtype == torch.float32 and not torch.is_autocast_enabled("cuda"):
        mode = "fp32"
    elif hidden.dtype == torch.bfloat16:
        mode = "bf16"
    else:
        raise NotImplementedError(
            f"{who}: hidden must be bfloat16, or float32 (inside bf16 CUDA autocast or outside autocast), "
            f"got {hidden.dtype} with autocast " + ("on" if torch.is_autocast_enabled("cuda") else "off"))
    if labels.dtype != torch.int64:
        raise RuntimeError(f"{who}: labels must be int64")
    n, d = hidden.shape
    v = weight.shape[0]
    if weight.shape[1] != d or labels.shape[0] != n:
        raise RuntimeError(f"{who}: shapes hidden {tuple(hidden.shape)}, weight {tuple(weight.shape)}, "
                           f"labels {tuple(labels.shape)} do not match")
    if weight.device != hidden.device or labels.device != hidden.device:
        raise RuntimeError(f"{who}: hidden, weight and labels must be on one device")
    auto = chunk_size is None or (isinstance(chunk_size, str) and chunk_size == "auto")
    if isinstance(chunk_size, str) and not auto:
        raise ValueError(f"{who}: chunk_size must be a positive int, None or 'auto', got {chunk_size!r}")
    chunk = auto_chunk_rows(n, v) if auto else int(chunk_size)
    if chunk < 1:
        raise ValueError(f"{who}: chunk_size must be positive, got {chunk_size}")
    return n, v, chunk, mode


def _bf16(logits: torch.Tensor) -> torch.Tensor:
    """The row kernel reads bf16 bits: refuse anything else loudly."""
    if logits.dtype != torch.bfloat16 or not logits.is_contiguous():
        raise RuntimeError(f"fused_linear_cross_entropy: the logits GEMM returned {logits.dtype} "
                           f"(contiguous: {logits.is_contiguous()}), the row kernels need contiguous bfloat16")
    return logits


def _mean_loss(row_loss, labels, n, ignore_index, lib, stream):
    """(mean loss as a 0-d tensor, the loss sum and n_valid as one tensor) from the per-row losses."""
    out2 = torch.empty(2, dtype=torch.float32, device=row_loss.device)
    loss = torch.empty((), dtype=torch.float32, device=row_loss.device)
    _native.check(lib.tm_ce_mean_loss(row_loss.data_ptr(), labels.data_ptr(), n, int(ignore_index),
                                      out2.data_ptr(), loss.data_ptr(), stream), "tm_ce_mean_loss")
    return loss, out2


def logits_gemm_fits(h: torch.Tensor, w: torch.Tensor) -> bool:
    """Chunks whose logits run on this package's GEMM (tm_ce_logits_bf16): bf16 operands, both
    contiguous and 16-byte aligned, dim a multiple of 64. Other shapes take torch.matmul."""
    return (h.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and h.dim() == 2 and w.dim() == 2
            and h.shape[1] == w.shape[1] and h.shape[1] % 64 == 0 and h.shape[0] > 0 and w.shape[0] > 0
            and h.is_contiguous() and w.is_contiguous() and h.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0)


def _logits(h: torch.Tensor, w: torch.Tensor, lib, stream) -> torch.Tensor:
    """logits = h @ w.T (fused_linear_ce.py:38): a bf16 GEMM, fp32 accumulation, bf16 result."""
    if not logits_gemm_fits(h, w):
        return _bf16(torch.matmul(h, w.t()))
    rows, dim = h.shape
    out = torch.empty((rows, w.shape[0]), dtype=torch.bfloat16, device=h.device)
    _native.check(lib.tm_ce_logits_bf16(out.data_ptr(), h.data_ptr(), w.data_ptr(), rows, w.shape[0], dim, stream),
                  "tm_ce_logits_bf16")
    return out


def padded_rows(rows: int) -> int:
    """Rows of a chunk's padded logits: whole 64-row K slices of the grad_W GEMM, and from 129
    rows an even number of them, at least 4 (its persistent kernel's form)."""
    return -(-rows // 64) * 64 if rows <= 128 else max(256, -(-rows // 128) * 128)


def padded_vocab(vocab: int) -> int:
    """Elements from one padded logits row to the next: whole 64-column K slices of the grad_h
    GEMM; every row then starts on a 16-byte boundary (on a cache line), for any vocabulary."""
    return -(-vocab // 64) * 64


def grad_w_gemm_fits(g: torch.Tensor, h: torch.Tensor) -> bool:
    """Unpadded chunks whose grad_W runs on this package's GEMM: bf16 operands, both contiguous and
    16-byte aligned, vocab and dim multiples of 8. Other shapes take torch.matmul."""
    return (g.dtype == torch.bfloat16 and h.dtype == torch.bfloat16 and g.dim() == 2 and h.dim() == 2
            and g.shape[0] == h.shape[0] and g.shape[0] > 0 and g.shape[1] % 8 == 0
            and h.shape[1] % 8 == 0 and g.shape[1] > 0 and h.shape[1] > 0 and g.is_contiguous() and h.is_contiguous()
            and g.data_ptr() % 16 == 0 and h.data_ptr() % 16 == 0)


def _grad_w(g: torch.Tensor, h: torch.Tensor, lib, stream) -> torch.Tensor:
    """A chunk's gw = grad_logits.t() @ h (fused_linear_ce.py:57) from unpadded grad_logits: bf16
    GEMM, bf16 result (V x D). Rows off a multiple of 64 are copied into a zero-padded buffer. The
    product does without the copy and the workspace for its split sums where memory for them is
    short."""
    rows, vocab = g.shape
    if not grad_w_gemm_fits(g, h) or (rows % 64 and h.shape[1] % 64):
        return torch.matmul(g.t(), h)
    out = torch.empty((vocab, h.shape[1]), dtype=torch.bfloat16, device=g.device)
    pad = rows if rows % 64 == 0 else padded_rows(rows)
    nbytes = lib.tm_ce_grad_w_ld_workspace_bytes(pad, vocab, h.shape[1])
    padded, ws = g, None
    try:
        if pad != rows:
            padded = torch.zeros((pad, vocab), dtype=torch.bfloat16, device=g.device)
            padded[:rows].copy_(g)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=g.device) if nbytes else None
    except torch.OutOfMemoryError:
        if pad != rows:
            return torch.matmul(g.t(), h, out=out)
    _native.check(lib.tm_ce_grad_w_ld_bf16(out.data_ptr(), padded.data_ptr(), vocab, pad, h.data_ptr(), rows, vocab,
                                           h.shape[1], None if ws is None else ws.data_ptr(), 0 if ws is None else nbytes,
                                           stream), "tm_ce_grad_w_ld_bf16")
    return out


SPLITK_GRAD_H_MAX_TILES = 64


def _grad_h_takes(rows: int, dim: int, vocab: int) -> bool:
    """Sizes that tm_ce_grad_h_ld_bf16 accepts."""
    return 0 < rows <= 1 << 20 and 0 < dim <= 1 << 16 and dim % 8 == 0 and 0 < vocab <= 0x7FFFFF00


def splitk_grad_h_fits(rows: int, dim: int, vocab: int) -> bool:
    """Chunks whose grad_h runs on the split-K MFMA GEMM (tm_ce_grad_h_bf16): the shapes it
    tiles (rows and dim multiples of 256, vocab of 64), except where the library GEMM measured
    faster on MI355X: more than SPLITK_GRAD_H_MAX_TILES output tiles of 256 x 256 with dim a
    power of two. With few tiles and K = vocab a library GEMM leaves most of the 256 CUs idle and
    the split-K kernel spreads K over them; with many, the library's kernels fill the chip
    themselves, and beat this kernel by 3-11% when dim is a power of two, but run 12-51% behind
    it at the other Qwen3 head widths (ms per call at V = 151,936, split-K / hipBLASLt):

        dim   rows 1024      2048           4096           8192
        1024  0.28 / 0.72    0.62 / 1.03    1.07 / 1.44    2.06 / 1.99
        2048  0.51 / 0.89    1.00 / 1.61    2.00 / 1.93    4.13 / 3.69
        2560  0.66 / 1.00    1.33 / 1.84    2.75 / 3.38    5.24 / 7.44
        4096  1.03 / 1.82    2.05 / 1.91    4.11 / 3.66    8.13 / 7.40
        5120  1.38 / 1.87    2.98 / 3.34    5.58 / 6.85    10.85 / 13.16
    """
    if not _grad_h_takes(rows, dim, vocab) or rows % 256 or dim % 256 or vocab % 64:
        return False
    return (rows // 256) * (dim // 256) <= SPLITK_GRAD_H_MAX_TILES or (dim & (dim - 1)) != 0


RAGGED_GRAD_H_MIN_VOCAB = 4097
RAGGED_GRAD_H_MAX_TILES = 96
RAGGED_GRAD_H_LONG_VOCAB = 16384


def grad_h_gemm_fits(rows: int, dim: int, vocab: int) -> bool:
    """Padded chunks whose grad_h runs on this package's GEMM: those ``splitk_grad_h_fits`` accepts,
    and of the ragged ones (rows or dim off a multiple of 256, a vocabulary off a multiple of 64)
    those of a vocabulary above 4096, of at most 64 tiles at a power-of-two width and 96 at others,
    and at those other widths of any more tiles from a vocabulary of RAGGED_GRAD_H_LONG_VOCAB up.
    us per call on MI355X, this package / hipBLASLt on the same padded logits:

        rows x dim (tiles)    vocab 1984     4097-5001      7296         12001         20032         32001
        1184 x  384  (10)       15 /  20      18 /  25     22 /  33
        2046 x 1216  (40)       24 /  28      39 /  53     56 /  59
        4000 x 1024  (64)       26 /  26      56 /  55     75 /  67    103 / 113     159 / 211     248 / 335
        4001 x 1216  (80)       33 /  36      65 /  77     82 /  97    120 / 160     193 / 251     299 / 406
        6001 x  832  (96)       34 /  37      74 /  77     95 /  96    151 / 161     240 / 294     383 / 466
        3000 x 2560 (120)       38 /  37      88 /  82    113 / 103    170 / 169     279 / 384     442 / 616
        7129 x 1216 (140)       51 /  47     119 /  98    152 / 126    232 / 209     388 / 526     593 / 806
        8000 x 2560 (320)      104 / 100     221 / 227    358 / 253    536 / 423     804 / 697    1219 / 1686

    With few tiles the library leaves CUs idle. With many it fills the chip and this kernel's splits
    only cost their partials, until K is long: past some 16,000 (20,000 at 320 tiles) the library's
    kernels for these widths fall behind by a quarter to a half. The lower line is not one of speed: a ragged chunk of
    a vocabulary up to 4096 keeps the library's product and its bits, though this kernel would be
    the faster there too (from level to 2x at up to 96 tiles)."""
    if splitk_grad_h_fits(rows, dim, vocab):
        return True
    if not (_grad_h_takes(rows, dim, vocab) and vocab >= RAGGED_GRAD_H_MIN_VOCAB
            and (rows % 256 or dim % 256 or vocab % 64)):
        return False
    tiles = -(-rows // 256) * -(-dim // 256)
    if dim & (dim - 1) == 0:
        return tiles <= SPLITK_GRAD_H_MAX_TILES
    return tiles <= RAGGED_GRAD_H_MAX_TILES or vocab >= RAGGED_GRAD_H_LONG_VOCAB


GROUP_BYTES = 1 << 30  # logits of the chunks whose logits and row pass run together, at most
GROUP_ROWS = 16384  # and their rows


def group_chunks(rows: int, chunk: int, vocab: int, grad: bool) -> int:
    """Chunks whose logits GEMM and row pass run as one launch each. Both work row by row, so the
    chunking fixes none of their bits (as it does grad_W's, which stay per chunk), and more rows
    fill the last round of tiles better: a 1024-row chunk of the Qwen3-0.6B head has 9.3 rounds of
    256 x 256 tiles and takes 10, three together 27.8 (8192 rows: 8709 -> 8374 us a call; 2500 x
    768 x 32,001: 610 -> 578). Chunks with padding rows of their own (not a
    multiple of 128) are not contiguous in K and run one by one. Bounded by GROUP_BYTES (0.4% of
    the GPU's memory; a caller's larger chunk is taken as it is), and by rows, so that the hidden
    states keep 32-bit offsets."""
    most = min(GROUP_BYTES // (2 * chunk * padded_vocab(vocab)), GROUP_ROWS // chunk)
    if rows <= chunk or most <= 1 or (grad and padded_rows(chunk) != chunk):
        return 1
    chunks = -(-rows // chunk)
    return -(-chunks // -(-chunks // most))  # groups of about the same size


FOLD_CHUNKS = 8  # chunks per grad_W fold (tm_ce_grad_w_fold takes at most 8)
FOLD_BYTES = 4 << 30  # bf16 chunk grad_W held before a fold, at most


def _fold(lib, grad_weight, chunks, accumulated, stream) -> None:
    """grad_weight = ((grad_weight or +0) + float(c0) + float(c1) + ...), the reference's
    `grad_weight += gw` per chunk in order (fused_linear_ce.py:80-81), in one pass over the fp32
    buffer."""
    ptrs = (ctypes.c_void_p * len(chunks))(*[c.data_ptr() for c in chunks])
    _native.check(lib.tm_ce_grad_w_fold(grad_weight.data_ptr(), ptrs, len(chunks), chunks[0].numel(),
                                        int(accumulated), None, None, stream), "tm_ce_grad_w_fold")


class GradHidden:
    """grad_h = grad_logits @ W (fused_linear_ce.py:52, stored at :79) for the chunks of one
    call on unpadded logits: the split-K MFMA GEMM on the chunks ``splitk_grad_h_fits`` accepts,
    reading W as it is stored, with one fp32 partials workspace shared by the chunks
    (stream-ordered), and torch.matmul (hipBLASLt) on the others. ``w`` is the contiguous bf16
    weight (V x D)."""

    def __init__(self, w: torch.Tensor, chunk_rows, lib, stream):
        self.w, self.lib, self.stream = w, lib, stream
        self.vocab, self.dim = w.shape
        fits = [r for r in set(chunk_rows) if splitk_grad_h_fits(r, self.dim, self.vocab)]
        self.ws = None
        if fits:
            nbytes = max(lib.tm_ce_grad_h_workspace_bytes(r, self.vocab, self.dim) for r in fits)
            self.ws = torch.empty(nbytes, dtype=torch.uint8, device=w.device)

    def __call__(self, grad_logits: torch.Tensor, out: torch.Tensor) -> None:
        rows = grad_logits.shape[0]
        if self.ws is None or not splitk_grad_h_fits(rows, self.dim, self.vocab):
            torch.matmul(grad_logits, self.w, out=out)
            return
        if not (grad_logits.is_contiguous() and out.is_contiguous() and out.dtype == torch.bfloat16):
            raise RuntimeError("fused_linear_cross_entropy: grad_h GEMM operands must be contiguous bf16")
        _native.check(self.lib.tm_ce_grad_h_bf16(out.data_ptr(), grad_logits.data_ptr(), self.w.data_ptr(), rows,
                                                 self.vocab, self.dim, self.ws.data_ptr(), self.ws.numel(),
                                                 self.stream), "tm_ce_grad_h_bf16")


def _copy_at_hand(weight: torch.Tensor):
    """The current bf16 working copy of an fp32 master (attached with
    torchure_amd.attach_bf16_working_params and rewritten by each AdamW step), which holds the
    bits of ``weight.to(bf16)``, or None. A copy that does not start on a 16-byte boundary (the
    optimizer accepts copies at any offset) is not taken: this op's kernels read the weight in
    16-byte vectors, and the cast gives a fresh, aligned buffer with the same bits."""
    if weight.dtype == torch.float32:
        w = current_copy(weight)
        if w is not None and w.data_ptr() % 16 == 0:
            return w.detach()
    return None


def _bf16_weight(weight: torch.Tensor) -> torch.Tensor:
    """The contiguous bf16 weight the products run on: ``weight.to(bf16)`` (RNE, as autocast
    casts), or its current working copy, which skips the cast's read of 4 and write of 2 bytes
    per element."""
    w = _copy_at_hand(weight)
    return weight.to(torch.bfloat16).contiguous() if w is None else w


def _castable(t: torch.Tensor) -> bool:
    """fp32 values that tm_ce_cast2 may read from memory as they are; anything else (other
    strides, a tensor subclass with a cast of its own, a lazy negation) takes ``Tensor.to``."""
    return (t.dtype == torch.float32 and type(t) in (torch.Tensor, torch.nn.Parameter) and t.is_contiguous()
            and not t.is_neg())


def _run_chunks(hidden, weight, labels, ignore_index, chunk, mode, grad, want_h, want_w):
    """The chunk loop on padded logits (``_tm_host.ce_forward``), for operands that the MFMA
    kernels take (dim a multiple of 64, bf16 ones 16-byte aligned), or None on others. Returns
    (loss, (loss sum, n_valid), grad_hidden, grad_weight, grad_W chunks still to be added,
    accumulated). autocast's casts, or the weight's, are made there in one launch.

    Where memory is short, whichever allocation of the call it fails: once more with one chunk's
    logits at a time (the same bits), then None, for the unpadded loop, which holds neither padding
    nor a workspace for grad_W."""
    (n, d), v = hidden.shape, weight.shape[0]
    if n == 0 or d == 0 or v == 0 or d % 64:
        return None
    h, cast_h = hidden, mode == "autocast"
    if cast_h and not _castable(h):
        h, cast_h = h.to(torch.bfloat16), False
    w, cast_w = _copy_at_hand(weight), False
    if w is None:
        cast_w = _castable(weight)
        w = weight if cast_w else weight.to(torch.bfloat16).contiguous()
    if not (cast_h or h.data_ptr() % 16 == 0) or not (cast_w or w.data_ptr() % 16 == 0):
        return None
    chunk = min(chunk, n)
    last = n - (n - 1) // chunk * chunk
    group = group_chunks(n, chunk, v, grad)
    for held in (group, 1) if group > 1 else (1,):
        try:
            return _native.ce_host().ce_forward(
                h, w, cast_h, cast_w, labels, int(ignore_index), chunk, held,
                (padded_rows(chunk), padded_rows(last)), padded_vocab(v),
                (grad_h_gemm_fits(chunk, d, v), grad_h_gemm_fits(last, d, v)), grad, want_h, want_w,
                FOLD_CHUNKS, FOLD_BYTES, _native.stream_handle(hidden.device))
        except torch.OutOfMemoryError:
            pass
    return None


def _bf16_operands(hidden, weight, mode):
    """(hidden, weight) in bf16 as the products read them (autocast's casts, RNE)."""
    return hidden.to(torch.bfloat16) if mode == "autocast" else hidden, _bf16_weight(weight)


def _loss_only(hidden, weight, labels, ignore_index, chunk_size):
    """The loss when no input needs a gradient (e.g. evaluation under torch.no_grad): the
    same logits GEMM and the same per-row arithmetic as the training path, so the same
    bits, without the two gradient GEMMs or the gradient write. The reference's forward
    computes and drops the gradients in this case (fused_linear_ce.py:63-93)."""
    n, v, chunk, mode = _checked(hidden, weight, labels, chunk_size)
    if mode == "fp32":
        return _fp32_chunks(hidden, weight, labels, ignore_index, n, v, chunk, False, False, False)[0]
    done = _run_chunks(hidden, weight, labels, ignore_index, chunk, mode, False, False, False)
    if done is not None:
        return done[0]
    lib = _native.lib()
    stream = _native.stream_handle(hidden.device)
    hb, w = _bf16_operands(hidden, weight, mode)
    row_loss = torch.empty(n, dtype=torch.float32, device=hidden.device)
    for s in range(0, n, chunk):
        e = min(s + chunk, n)
        logits = _logits(hb[s:e], w, lib, stream)
        _native.check(lib.tm_ce_rows_loss_bf16(logits.data_ptr(), v, labels[s:e].data_ptr(), e - s, v,
                                               int(ignore_index), row_loss[s:].data_ptr(), stream),
                      "tm_ce_rows_loss_bf16")
        del logits
    return _mean_loss(row_loss, labels, n, ignore_index, lib, stream)[0]


def _fp32_chunks(hidden, weight, labels, ignore_index, n, v, chunk, grad, want_h, want_w):
    """fp32 hidden states outside autocast. The reference then casts the weight to fp32 once
    (fused_linear_ce.py:65), its three products are fp32 GEMMs and its buffers are fp32
    (:66-72). This loop does the same: per chunk, fp32 logits from the library product, their
    rows a multiple of 32 elements apart, tm_ce_rows_f32 in place (the chunk math of :39-51 on
    fp32 logits), grad_h = grad_logits @ w into the fp32 grad_hidden (:52,79), and
    grad_logits^T @ h into the fp32 grad_weight (:57,80-81): the first chunk's product is
    written there, the later ones are added by the product (a zero fill and an fp32 `+=` would
    pass over it three times more a chunk). Backward scales both in place. Returns what
    ``_run_chunks`` does."""
    lib = _native.lib()
    stream = _native.stream_handle(hidden.device)
    w = weight.to(torch.float32).contiguous()
    ld = -(-v // 32) * 32
    grad_hidden = torch.empty(hidden.shape, dtype=torch.float32, device=hidden.device) if want_h else None
    grad_weight = None
    if want_w:
        grad_weight = (torch.empty if n else torch.zeros)(weight.shape, dtype=torch.float32, device=weight.device)
    row_loss = torch.empty(n, dtype=torch.float32, device=hidden.device)
    rows_of = lib.tm_ce_rows_f32 if grad else lib.tm_ce_rows_loss_f32
    for s in range(0, n, chunk):
        e = min(s + chunk, n)
        h = hidden[s:e]
        logits = torch.empty((e - s, ld), dtype=torch.float32, device=hidden.device)[:, :v]
        torch.mm(h, w.t(), out=logits)
        _native.check(rows_of(logits.data_ptr(), ld, labels[s:e].data_ptr(), e - s, v, int(ignore_index),
                              row_loss[s:].data_ptr(), stream), "tm_ce_rows_f32")
        if want_h:
            torch.mm(logits, w, out=grad_hidden[s:e])
        if want_w and s == 0:
            torch.mm(logits.t(), h, out=grad_weight)
        elif want_w:
            grad_weight.addmm_(logits.t(), h)
        del logits
    loss, out2 = _mean_loss(row_loss, labels, n, ignore_index, lib, stream)
    return loss, out2, grad_hidden, grad_weight, [], True


def _chunks_unpadded(hidden, weight, labels, ignore_index, n, v, chunk, mode, want_h, want_w):
    """The chunk loop for what ``_run_chunks`` does not take (a dim off 64, unaligned or strided
    operands, no rows) or finds no memory for: logits rows vocab elements apart, library products
    where this package's GEMMs do not fit. Returns what ``_run_chunks`` does."""
    lib = _native.lib()
    stream = _native.stream_handle(hidden.device)
    hb, w = _bf16_operands(hidden, weight, mode)  # cast once, not per chunk
    # bf16 GEMM output either way; for fp32 hidden it is widened and scaled in backward
    grad_hidden = torch.empty(hidden.shape, dtype=torch.bfloat16, device=hidden.device) if want_h else None
    # Chunks' bf16 grad_W wait in `pending` and are folded into the fp32 grad_W several at a
    # time (one pass per fold); the last chunk, and those still pending, wait for backward.
    grad_weight, pending, accumulated = None, [], False
    row_loss = torch.empty(n, dtype=torch.float32, device=hidden.device)
    grad_h_of = GradHidden(w, [min(chunk, n - s) for s in range(0, n, chunk)], lib, stream) if want_h else None
    for s in range(0, n, chunk):
        e = min(s + chunk, n)
        h = hb[s:e]
        logits = _logits(h, w, lib, stream)  # (C, V) bf16
        _native.check(lib.tm_ce_rows_bf16(logits.data_ptr(), v, labels[s:e].data_ptr(), e - s, v,
                                          int(ignore_index), row_loss[s:].data_ptr(), stream),
                      "tm_ce_rows_bf16")
        if want_h:
            grad_h_of(logits, grad_hidden[s:e])
        if want_w:
            pending.append(_grad_w(logits, h, lib, stream))  # (V, D) bf16
            if e < n and (len(pending) == FOLD_CHUNKS or len(pending) * pending[0].numel() * 2 >= FOLD_BYTES):
                if grad_weight is None:
                    grad_weight = torch.empty(weight.shape, dtype=torch.float32, device=weight.device)
                _fold(lib, grad_weight, pending, accumulated, stream)
                accumulated = True
                pending = []
        del logits
    loss, out2 = _mean_loss(row_loss, labels, n, ignore_index, lib, stream)
    return loss, out2, grad_hidden, grad_weight, pending, accumulated


class _FusedLinearCE(torch.autograd.Function):
    @staticmethod
    def forward(ctx, hidden, weight, labels, ignore_index, chunk_size):
        n, v, chunk, mode = _checked(hidden, weight, labels, chunk_size)
        want_h, want_w = ctx.needs_input_grad[0], ctx.needs_input_grad[1]
        # grad_hidden as held for backward: bf16, bf16 that becomes fp32, or fp32
        ctx.kind = {"bf16": 0, "autocast": 1, "fp32": 2}[mode]
        ctx.want_w = want_w
        ctx.weight_meta = (weight.shape, weight.device)
        if mode == "fp32":
            done = _fp32_chunks(hidden, weight, labels, ignore_index, n, v, chunk, True, want_h, want_w)
        else:
            done = _run_chunks(hidden, weight, labels, ignore_index, chunk, mode, True, want_h, want_w)
            if done is None:
                done = _chunks_unpadded(hidden, weight, labels, ignore_index, n, v, chunk, mode, want_h, want_w)
        # what backward needs, consumed by it
        ctx.stash = done[1:]
        return done[0]

    @staticmethod
    def backward(ctx, grad_out):
        if ctx.stash is None:
            raise RuntimeError(
                "fused_linear_cross_entropy: backward called twice. the stashed grads are "
                "consumed in place on the first call, so retain_graph does not work through this op")
        out2, grad_hidden, grad_weight, chunks, accumulated = ctx.stash
        ctx.stash = None
        if ctx.want_w and not chunks and grad_weight is None:
            # no rows at all: the reference scales its zero-filled buffer
            shape, device = ctx.weight_meta
            grad_weight, accumulated = torch.zeros(shape, dtype=torch.float32, device=device), True
        # fused_linear_ce.py:107-126: the chunks still waiting (at most FOLD_CHUNKS) added into grad_W
        # with the scaling, and grad_h scaled (under autocast float(bf16 GEMM result) * scale), in one
        # launch; where there is no memory for both results beside the chunks, one after the other
        finish, stream = _native.ce_host().ce_backward, _native.stream_handle(out2.device)
        try:
            grad_hidden, grad_weight = finish(grad_out, out2, grad_hidden, ctx.kind, grad_weight, chunks, accumulated,
                                              stream)
            return grad_hidden, grad_weight, None, None, None
        except torch.OutOfMemoryError:
            pass
        grad_weight = finish(grad_out, out2, None, ctx.kind, grad_weight, chunks, accumulated, stream)[1]
        del chunks
        grad_hidden = finish(grad_out, out2, grad_hidden, ctx.kind, None, [], True, stream)[0]
        return grad_hidden, grad_weight, None, None, None


def fused_linear_cross_entropy(
    hidden: torch.Tensor,  # (B, S, D) or (N, D), bf16 or fp32
    weight: torch.Tensor,  # (V, D) lm_head weight
    labels: torch.Tensor,  # (B, S) or (N,), already shifted, int64
    ignore_index: int = -100,
    chunk_size: int | str | None = 1024,
) -> torch.Tensor:
    """Mean cross-entropy of ``hidden @ weight.T`` against ``labels`` over the rows whose
    label is not ``ignore_index``, in chunks of ``chunk_size`` rows, as
    torchure/loss/fused_linear_ce.py:130-136 (default 1024 rows, as there: each chunk's bf16
    grad_W is rounded before it is added, so the chunking fixes grad_W's bits).
    ``chunk_size=None`` or ``"auto"`` sizes chunks by a 4 GiB logits budget instead
    (``auto_chunk_rows``): the whole Qwen3 vocabulary for 8K-16K tokens in one chunk, one
    fp32 grad_W pass and large GEMMs, at the cost of other grad_W bits and up to 4 GiB of
    logits plus one bf16 grad_W (V x D) held from forward to backward."""
    if hidden.dim() == 3:
        hidden = hidden.reshape(-1, hidden.shape[-1])
        labels = labels.reshape(-1)
    hidden, labels = hidden.contiguous(), labels.contiguous()
    with CALL_ORDER.call(hidden.device):  # one call's GEMMs at a time per device
        if not (torch.is_grad_enabled() and (hidden.requires_grad or weight.requires_grad)):
            return _loss_only(hidden, weight, labels, ignore_index, chunk_size)
        return _FusedLinearCE.apply(hidden, weight, labels, ignore_index, chunk_size)
