"""GPU parity of the chunked fused linear + cross-entropy (torchure/loss/fused_linear_ce.py).

Checks:
- the fused CE-row kernel vs an fp64 restatement on the same bf16 logits: per-row
  loss within 1e-6 relative, grad_logits = bf16(softmax - onehot) within 1 bf16 ulp;
  the in-register path (V <= 163,840), the two-read path (larger V) and the
  element-wise path (rows not 16-byte aligned) are all exercised;
- the whole op (forward + backward through autograd) vs the reference's own
  composition (torchure/loss/fused_linear_ce.py, same torch calls) on the same
  device: same GEMMs, so the loss agrees within 1e-5 relative and the grads
  within bf16 resolution;
- the reference's own test cases (tests/fused_linear_ce.py), against an unfused
  lm_head + F.cross_entropy at that test's bars, plus the trainer's own call (fp32 hidden
  under bf16 autocast, 4096-row chunks);
- the grad_W hand-over (one chunk, or two in one pass) bit for bit against torch's `+=` and
  `mul_`, and the whole chunk loop bit for bit for 1, 2, 3, 4 and 7 chunks;
- fp32 hidden under autocast, ignore_index values inside the vocabulary, non-contiguous
  inputs, the loss-only path and gradients for only one input.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle
from oracle.torch_composition import fused_linear_ce_reference
from tests import _helpers as H

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")
    import torchure_amd

    torchure_amd._native.lib()
    yield


def _ce_rows(logits_bits: np.ndarray, labels: np.ndarray, ignore: int):
    from torchure_amd import _native

    rows, v = logits_bits.shape
    d_logits = torch.from_numpy(logits_bits.view(np.int16).copy()).to(DEV)
    d_labels = torch.from_numpy(labels.astype(np.int64)).to(DEV)
    d_loss = torch.empty(rows, dtype=torch.float32, device=DEV)
    rc = _native.lib().tm_ce_rows_bf16(d_logits.data_ptr(), v, d_labels.data_ptr(), rows, v, ignore,
                                       d_loss.data_ptr(), _native.stream_handle(DEV))
    _native.check(rc, "tm_ce_rows_bf16")
    torch.cuda.synchronize()
    return d_logits.cpu().numpy().view(np.uint16), d_loss.cpu().numpy()


@pytest.mark.parametrize("vocab", [4096, 1001, 151936, 200000])
def test_ce_rows_kernel_vs_fp64(vocab):
    r = H.rng(vocab)
    rows = 37
    x = (r.standard_normal((rows, vocab)) * 3.0).astype(np.float32)
    bits = oracle.bf16_rne(x).reshape(rows, vocab)
    labels = r.integers(0, vocab, rows)
    labels[[3, 17]] = -100
    grad_bits, loss = _ce_rows(bits, labels, -100)
    xd = oracle.bf16_to_f32(bits).reshape(rows, vocab).astype(np.float64)
    mx = xd.max(axis=1, keepdims=True)
    lse = (mx + np.log(np.exp(xd - mx).sum(axis=1, keepdims=True)))[:, 0]
    valid = labels != -100
    want_loss = np.where(valid, lse - xd[np.arange(rows), np.where(valid, labels, 0)], 0.0)
    np.testing.assert_allclose(loss, want_loss, rtol=1e-6, atol=1e-6)
    probs = np.exp(xd - lse[:, None])
    probs[np.arange(rows)[valid], labels[valid]] -= 1.0
    probs[~valid] = 0.0
    want_bits = oracle.bf16_rne(probs.astype(np.float32)).reshape(rows, vocab)
    diff = np.abs(grad_bits.astype(np.int32) - want_bits.astype(np.int32))
    # ulp distance on same-sign values; sign flips can only occur at |value| ~ 0
    assert diff.max() <= 1, (diff.max(), np.argwhere(diff > 1)[:4])
    assert (diff == 0).mean() > 0.99
    assert np.all(grad_bits[~valid] == 0)


@pytest.mark.parametrize("vocab", [
    3, 8, 2048, 2056, 4104, 6152, 8200, 10240,       # one wave a row, 4 to 20 vectors a thread
    10248, 12296, 16392, 20480, 20488, 24585, 40960,  # two and four waves
    40968, 81920, 81928, 98312, 163840, 163843,       # eight and sixteen waves
    163848, 165000,                                   # too long for registers
])
def test_ce_rows_at_the_edges_of_the_row_shapes(vocab):
    """The row kernel on both sides of every change of its threads and vectors a row: losses and
    gradients against fp64, the loss-only pass bit for bit equal, -inf, NaN and +inf where only
    some threads or batches see them, and nothing written past the rows. Bounds: a sum of
    positive exponentials in fp32 is off by at most one rounding of 2^-24 per addition on the
    longest chain: 20 vectors of 3 levels, 5 rescales and 10 merges on the vector path (38, and 3
    an exponential), vocab / 1024 on an odd row's element path; lse moves by that plus its own
    roundings, and a gradient is one bf16 rounding of a value that close."""
    from torchure_amd import _native

    lib, st = _native.lib(), _native.stream_handle(DEV)
    g = torch.Generator(device=DEV).manual_seed(vocab)
    rows = 13
    buf = torch.zeros(rows * vocab + 16, dtype=torch.bfloat16, device=DEV)
    buf[rows * vocab:] = 7.0
    x = buf[: rows * vocab].view(rows, vocab)
    x.copy_(torch.randn(rows, vocab, device=DEV, generator=g) * 3.0)
    x[1, : vocab // 2] = float("-inf")       # whole threads' vectors
    x[2, : max(1, vocab - 2)] = float("-inf")
    x[3] = 3.390625e38                       # equal to the largest finite values
    x[4] -= 300.0
    x[5, vocab // 3] = float("nan")
    x[6] = float("-inf")
    x[6, vocab - 1] = float("nan")           # a NaN under a maximum of -inf elsewhere
    x[7, vocab // 2] = float("inf")
    labels = torch.randint(0, vocab, (rows,), device=DEV, generator=g)
    labels[1:3] = vocab - 1
    labels[8] = -100
    xd = x.double()
    loss_only, loss = torch.empty(rows, device=DEV), torch.empty(rows, device=DEV)
    for fn, out in ((lib.tm_ce_rows_loss_bf16, loss_only), (lib.tm_ce_rows_bf16, loss)):
        _native.check(fn(x.data_ptr(), vocab, labels.data_ptr(), rows, vocab, -100, out.data_ptr(), st), "rows")
    assert torch.equal(loss_only.view(torch.int32), loss.view(torch.int32))
    assert (buf[rows * vocab:] == 7.0).all()
    fine = [r for r in range(rows) if r not in (5, 6, 7)]
    lse = torch.logsumexp(xd, dim=1)
    want = lse - xd.gather(1, labels.clamp_min(0)[:, None])[:, 0]
    want[8] = 0.0
    chain = 41 + (vocab // 1024 if vocab % 8 else 0)
    tol = 2.0 ** -24 * (chain + 2 * lse.abs())
    assert ((loss.double() - want).abs() <= tol)[fine].all(), (loss, want)
    assert loss[5].isnan() and loss[6].isnan() and not loss[7].isfinite()
    probs = torch.exp(xd - lse[:, None])
    probs[torch.arange(rows), labels.clamp_min(0)] -= 1.0
    probs[8] = 0.0
    got = x.double()
    # one rounding (2^-9 relative), the exponent's error at |lse|, and the p - 1 of a sure label
    off = (got - probs).abs() - (2.0 ** -8 * probs.abs() + (4e-6 + 2.0 ** -22 * lse.abs()[:, None].clamp_max(512)))
    assert (off <= 0)[fine].all(), off[fine].max()
    assert got[5].isnan().all() and got[6].isnan().all()


@pytest.mark.parametrize("grad", [False, True])
def test_ce_rows_beyond_one_launch_of_single_waves(grad):
    """More rows than one launch of 64-thread workgroups holds (2^32 work-items). Rows 8 elements
    apart are 16-byte aligned, which a vocabulary this short runs with one wave a row (packed rows
    of 2 would take 1024 threads each). Every row on both sides of the line is checked: the losses,
    the gradients (p - 1 and p of two logits, RNE) and, with them, the cleared padding."""
    from torchure_amd import _native

    line = 0xFFFFFFFF // 64
    rows, v, ld = line + 77, 2, 8
    x = torch.zeros(rows, ld, dtype=torch.bfloat16, device=DEV)
    x[:, 1] = (torch.arange(rows, device=DEV) % 5).to(torch.bfloat16)
    x[:, v:] = 7.0  # past the vocabulary: not part of the row
    labels = torch.zeros(rows, dtype=torch.int64, device=DEV)
    labels[line - 1::3] = -100
    loss = torch.full((rows,), -1.0, device=DEV)
    lib, stream = _native.lib(), _native.stream_handle(DEV)
    if grad:
        _native.check(lib.tm_ce_rows_padded_bf16(x.data_ptr(), ld, labels.data_ptr(), rows, rows, v, -100,
                                                 loss.data_ptr(), stream), "rows")
    else:
        _native.check(lib.tm_ce_rows_loss_bf16(x.data_ptr(), ld, labels.data_ptr(), rows, v, -100, loss.data_ptr(),
                                               stream), "rows")
    a = torch.arange(5, device=DEV).double()
    kind, valid = torch.arange(rows, device=DEV) % 5, labels != -100
    assert bool(valid[line - 2]) and not bool(valid[line - 1]) and bool(valid[line]) and not bool(valid[line + 2])
    want = torch.where(valid, torch.log1p(torch.exp(a)).float()[kind], 0.0)
    torch.testing.assert_close(loss, want, rtol=1e-6, atol=1e-6)
    p = torch.sigmoid(a)
    g = torch.zeros(5, ld, dtype=torch.float64, device=DEV)
    g[:, 0], g[:, 1] = -p, p
    g = g.to(torch.bfloat16).view(torch.int16)
    for r in range(0, rows, 1 << 24):  # torch's own gather does not fill results of over 2^29 elements
        got, ok = x[r:r + (1 << 24)], valid[r:r + (1 << 24)]
        if not grad:
            assert bool((got[:, v:] == 7.0).all())
            continue
        # one ulp of bf16: the kernel's p is fp32, and p - 1 cancels
        off = (got.view(torch.int16) - g[kind[r:r + (1 << 24)]]).abs()[ok]
        assert int(off.max()) <= 1 and int(off[:, v:].max()) == 0
        assert not bool(got.view(torch.int16)[~ok].any())


def test_ce_rows_beyond_one_launch():
    """More rows than one launch of 1024-thread blocks holds (2^32 work-items): the
    entry point splits them, and every row still matches an fp64 restatement (here in
    torch float64 on the device, over all 4.2M rows)."""
    from torchure_amd import _native

    rows, v = 0xFFFFFFFF // 1024 + 2001, 16
    g = torch.Generator(device=DEV).manual_seed(11)
    # unit-scale logits: no row has a softmax entry within 1e-4 of 1, where fp32's
    # p - 1 cancels (the reference's fp32 softmax loses the same bits there)
    logits = torch.randn(rows, v, device=DEV, generator=g).to(torch.bfloat16)
    labels = torch.randint(0, v, (rows,), device=DEV, generator=g)
    labels[::1009] = -100
    xd = logits.double()
    work = logits.clone()
    loss = torch.empty(rows, dtype=torch.float32, device=DEV)
    rc = _native.lib().tm_ce_rows_bf16(work.data_ptr(), v, labels.data_ptr(), rows, v, -100,
                                       loss.data_ptr(), _native.stream_handle(DEV))
    _native.check(rc, "tm_ce_rows_bf16")
    valid = labels != -100
    lse = torch.logsumexp(xd, dim=1)
    picked = xd.gather(1, labels.clamp(min=0)[:, None])[:, 0]
    want = torch.where(valid, lse - picked, torch.zeros_like(lse))
    torch.testing.assert_close(loss.double(), want, rtol=1e-6, atol=1e-6)
    probs = torch.exp(xd - lse[:, None])
    probs[valid.nonzero()[:, 0], labels[valid]] -= 1.0
    probs[~valid] = 0.0
    want_bits = probs.float().to(torch.bfloat16).view(torch.int16).int()
    diff = (work.view(torch.int16).int() - want_bits).abs()
    assert int(diff.max()) <= 1
    assert float((diff == 0).double().mean()) > 0.99
    del xd, probs


@pytest.mark.parametrize("chunk", [None, 300])
def test_fused_linear_ce_matches_reference_composition(chunk):
    from torchure_amd.loss import fused_linear_cross_entropy

    g = torch.Generator(device=DEV).manual_seed(7)
    n, d, v = 1000, 256, 4096
    hidden = (torch.randn(n, d, device=DEV, generator=g) * 1.0).to(torch.bfloat16)
    weight = torch.randn(v, d, device=DEV, generator=g) * 0.05
    labels = torch.randint(0, v, (n,), device=DEV, generator=g)
    labels[::37] = -100
    h1 = hidden.clone().requires_grad_(True)
    w1 = weight.clone().requires_grad_(True)
    loss = fused_linear_cross_entropy(h1, w1, labels, -100, chunk)
    loss.backward()
    ref_loss, ref_gh, ref_gw = fused_linear_ce_reference(hidden, weight, labels, -100,
                                                         chunk_size=chunk or 1024)
    torch.cuda.synchronize()
    assert abs(loss.item() - ref_loss.item()) <= 1e-5 * abs(ref_loss.item())
    gh_err = (h1.grad.float() - ref_gh.float()).abs().max().item()
    gw_err = (w1.grad - ref_gw).abs().max().item()
    print(f"chunk {chunk}: loss {loss.item():.6f} ref {ref_loss.item():.6f}, "
          f"max |d grad_h| {gh_err:.3e} (scale {ref_gh.float().abs().max().item():.3e}), "
          f"max |d grad_w| {gw_err:.3e} (scale {ref_gw.abs().max().item():.3e})")
    assert gh_err <= 1e-2 * ref_gh.float().abs().max().item()
    assert gw_err <= 1e-2 * ref_gw.abs().max().item()
    assert w1.grad.dtype == torch.float32 and h1.grad.dtype == torch.bfloat16


def test_fused_linear_ce_all_ignored_and_double_backward():
    from torchure_amd.loss import fused_linear_cross_entropy

    n, d, v = 64, 32, 512
    hidden = torch.randn(n, d, device=DEV).to(torch.bfloat16).requires_grad_(True)
    weight = (torch.randn(v, d, device=DEV) * 0.1).requires_grad_(True)
    labels = torch.full((n,), -100, dtype=torch.int64, device=DEV)
    loss = fused_linear_cross_entropy(hidden, weight, labels)
    loss.backward(retain_graph=True)
    assert loss.item() == 0.0
    assert torch.count_nonzero(hidden.grad).item() == 0 and torch.count_nonzero(weight.grad).item() == 0
    with pytest.raises(RuntimeError, match="backward called twice"):
        loss.backward()


@pytest.mark.parametrize("nw,k,accumulate,nh,wide,off_w,off_h", [
    (0, 0, 0, 1, 0, 0, 0), (1, 1, 0, 0, 0, 0, 0),
    (255, 1, 0, 511, 1, 0, 0), (257, 8, 1, 513, 0, 0, 0),      # around a slice of each part
    (1000, 2, 1, 1027, 1, 1, 1), (1000, 3, 0, 1030, 0, 1, 3),  # nothing aligned
    (515, 0, 1, 4096, 0, 0, 2),                                # no chunks: a plain scale; 4-byte grad_h
    (70000, 5, 1, 33000, 1, 0, 0),
])
def test_ce_finish_bit_exact(nw, k, accumulate, nh, wide, off_w, off_h):
    """tm_ce_finish: grad_W's chunks added in order and scaled, grad_h scaled (bf16 by the bf16
    scale, or widened and scaled in fp32), each the same bits as the separate operations in torch,
    and nothing else written."""
    from torchure_amd import _native

    lib, st = _native.lib(), _native.stream_handle(DEV)
    g = torch.Generator(device=DEV).manual_seed(nw + nh)

    def fenced(n, off, dtype):
        buf = torch.randn(n + 64, device=DEV, generator=g).to(dtype)
        return buf, buf.clone(), buf[off: off + n]

    wbuf, wkeep, w = fenced(nw, off_w, torch.float32)
    chunks = [fenced(nw, off_w, torch.bfloat16)[2] for _ in range(k)]
    _, _, src = fenced(nh, off_h, torch.bfloat16)
    if nh:
        src[0] = -0.0
    hbuf, hkeep, dst = fenced(nh, off_h, torch.float32 if wide else torch.bfloat16)
    out, n_valid = torch.tensor(0.37, device=DEV), torch.tensor(123.0, device=DEV)
    scale = out / n_valid
    want = w.clone() if accumulate else torch.zeros_like(w)
    for c in chunks:
        want += c.float()
    want = want * scale
    want_h = src.float() * scale if wide else src * scale.to(torch.bfloat16)
    import ctypes
    ptrs = (ctypes.c_void_p * k)(*[c.data_ptr() for c in chunks])
    _native.check(lib.tm_ce_finish(w.data_ptr(), ptrs, k, nw, accumulate, src.data_ptr(), dst.data_ptr(), nh, wide,
                                   out.data_ptr(), n_valid.data_ptr(), st), "tm_ce_finish")
    bits = torch.int32 if wide else torch.int16
    assert torch.equal(w.view(torch.int32), want.view(torch.int32))
    assert torch.equal(dst.view(bits), want_h.view(bits))
    wkeep[off_w: off_w + nw] = w
    hkeep[off_h: off_h + nh] = dst
    assert torch.equal(wbuf, wkeep) and torch.equal(hbuf, hkeep)


@pytest.mark.parametrize("n0,n1,off", [(0, 1, 0), (511, 0, 0), (513, 1025, 0), (4099, 300, 1), (1 << 20, 777, 0)])
def test_ce_cast2_equals_the_device_cast(n0, n1, off):
    """Two arrays cast in one launch: torch's device cast bit for bit, special values included, at
    slice edges and unaligned starts, and nothing past either array written."""
    from torchure_amd import _native

    g = torch.Generator(device=DEV).manual_seed(n0 + n1)
    parts = []
    for n in (n0, n1):
        src = torch.randn(n + 8, device=DEV, generator=g)
        special = torch.tensor([float("nan"), float("inf"), -float("inf"), -0.0, 1e-40, 3.4e38, 1.00390625, 1.01171875], device=DEV)
        src[: min(8, n + 8)] = special
        dst = torch.full((n + 8,), 5.0, dtype=torch.bfloat16, device=DEV)
        parts.append((src[off: off + n], dst[off: off + n], dst))
    (s0, d0, b0), (s1, d1, b1) = parts
    _native.check(_native.lib().tm_ce_cast2(d0.data_ptr(), s0.data_ptr(), n0, d1.data_ptr(), s1.data_ptr(), n1,
                                            _native.stream_handle(DEV)), "tm_ce_cast2")
    for src, dst, buf in parts:
        want = torch.full_like(buf, 5.0)
        want[off: off + src.numel()] = src.to(torch.bfloat16)
        assert torch.equal(buf.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("accumulate,scaled,n,offset", [
    (0, 0, 4096, 0), (1, 0, 4096, 0), (0, 1, 4096, 0), (1, 1, 4096, 0),
    (1, 1, 1003, 0), (1, 1, 2050, 1), (0, 1, 777, 3)])
def test_ce_grad_w_handover_bit_exact(accumulate, scaled, n, offset):
    """tm_ce_grad_w vs the reference's torch ops on the same data
    (fused_linear_ce.py:80-81 `grad_weight += gw` on a zero-filled fp32 buffer, :126
    `grad_weight.mul_(grad_out / n_valid)`), bit for bit, including -0, +-inf, NaN and
    subnormal bf16 inputs, odd sizes and buffers that are not 16-byte aligned."""
    from torchure_amd import _native

    r = H.rng(n + 7 * offset + accumulate)
    chunk_bits = oracle.bf16_rne((r.standard_normal(n + offset) * 0.3).astype(np.float32))
    chunk_bits[offset:offset + 6] = [0x8000, 0x0000, 0x7F80, 0xFF80, 0x7FC0, 0x0001]
    chunk = torch.from_numpy(chunk_bits.view(np.int16).copy()).to(DEV)[offset:]
    acc0 = torch.from_numpy((r.standard_normal(n + offset) * 0.1).astype(np.float32)).to(DEV)[offset:]
    acc0[0] = acc0[6] = -0.0  # -0 + -0 keeps the sign only when accumulating
    grad_out = torch.tensor([0.37], dtype=torch.float32, device=DEV)
    n_valid = torch.tensor([977.0], dtype=torch.float32, device=DEV)

    if accumulate:
        want = acc0.clone()
    else:
        want = torch.zeros(n, dtype=torch.float32, device=DEV)
    want += chunk.view(torch.bfloat16).float()
    if scaled:
        want.mul_(grad_out[0] / n_valid[0])

    got = acc0.clone() if accumulate else torch.full((n,), 123.0, device=DEV)
    got_base = torch.empty(n + offset, dtype=torch.float32, device=DEV)
    got_view = got_base[offset:]
    got_view.copy_(got)
    rc = _native.lib().tm_ce_grad_w(got_view.data_ptr(), chunk.data_ptr(), n, accumulate,
                                    grad_out.data_ptr() if scaled else None,
                                    n_valid.data_ptr() if scaled else None, _native.stream_handle(DEV))
    _native.check(rc, "tm_ce_grad_w")
    torch.cuda.synchronize()
    a = got_view.cpu().numpy().view(np.uint32)
    b = want.cpu().numpy().view(np.uint32)
    assert np.array_equal(a, b), np.argwhere(a != b)[:5]


@pytest.mark.parametrize("accumulate,scaled,n,offset", [
    (0, 0, 4096, 0), (1, 0, 4096, 0), (0, 1, 4096, 0), (1, 1, 4096, 0), (1, 1, 1003, 0), (0, 1, 777, 3)])
def test_ce_grad_w2_handover_bit_exact(accumulate, scaled, n, offset):
    """tm_ce_grad_w2 (two chunks in one pass) vs the reference's torch ops on the same data:
    `grad_weight += gw` for one chunk and then the next, on a zero-filled (or given) fp32
    buffer, then `mul_(grad_out / n_valid)` (fused_linear_ce.py:80-81,126), bit for bit,
    with -0, +-inf, NaN and subnormal bf16 inputs, odd sizes and unaligned buffers."""
    from torchure_amd import _native

    r = H.rng(3 * n + 11 * offset + accumulate + 5)
    bits = []
    for k in range(2):
        b = oracle.bf16_rne((r.standard_normal(n + offset) * 0.3).astype(np.float32))
        b[offset + 3 * k:offset + 3 * k + 6] = [0x8000, 0x0000, 0x7F80, 0xFF80, 0x7FC0, 0x0001]
        bits.append(torch.from_numpy(b.view(np.int16).copy()).to(DEV)[offset:])
    acc0 = torch.from_numpy((r.standard_normal(n + offset) * 0.1).astype(np.float32)).to(DEV)[offset:]
    acc0[0] = acc0[9] = -0.0
    grad_out = torch.tensor([0.37], dtype=torch.float32, device=DEV)
    n_valid = torch.tensor([977.0], dtype=torch.float32, device=DEV)

    want = acc0.clone() if accumulate else torch.zeros(n, dtype=torch.float32, device=DEV)
    want += bits[0].view(torch.bfloat16).float()
    want += bits[1].view(torch.bfloat16).float()
    if scaled:
        want.mul_(grad_out[0] / n_valid[0])

    got_base = torch.full((n + offset,), 123.0, dtype=torch.float32, device=DEV)
    got = got_base[offset:]
    if accumulate:
        got.copy_(acc0)
    rc = _native.lib().tm_ce_grad_w2(got.data_ptr(), bits[0].data_ptr(), bits[1].data_ptr(), n, accumulate,
                                     grad_out.data_ptr() if scaled else None,
                                     n_valid.data_ptr() if scaled else None, _native.stream_handle(DEV))
    _native.check(rc, "tm_ce_grad_w2")
    torch.cuda.synchronize()
    a = got.cpu().numpy().view(np.uint32)
    b = want.cpu().numpy().view(np.uint32)
    assert np.array_equal(a, b), np.argwhere(a != b)[:5]


@pytest.mark.parametrize("k,accumulate,scaled,n,offset", [
    (1, 0, 1, 4096, 0), (3, 1, 0, 4096, 0), (5, 0, 0, 1003, 0), (8, 1, 1, 4096, 0),
    (8, 0, 1, 2050, 1), (7, 1, 1, 777, 3)])
def test_ce_grad_w_fold_bit_exact(k, accumulate, scaled, n, offset):
    """tm_ce_grad_w_fold (k chunks in one pass) vs the reference's torch ops on the same data:
    `grad_weight += gw` once per chunk in order, on a zero-filled (or given) fp32 buffer, then
    `mul_(grad_out / n_valid)` (fused_linear_ce.py:80-81,126), bit for bit, with -0, +-inf, NaN
    and subnormal bf16 inputs, odd sizes and buffers that are not 16-byte aligned."""
    import ctypes

    from torchure_amd import _native

    r = H.rng(5 * n + 13 * offset + 17 * k + accumulate)
    bits = []
    for j in range(k):
        b = oracle.bf16_rne((r.standard_normal(n + offset) * 0.3).astype(np.float32))
        b[offset + 2 * j:offset + 2 * j + 6] = [0x8000, 0x0000, 0x7F80, 0xFF80, 0x7FC0, 0x0001]
        bits.append(torch.from_numpy(b.view(np.int16).copy()).to(DEV)[offset:])
    acc0 = torch.from_numpy((r.standard_normal(n + offset) * 0.1).astype(np.float32)).to(DEV)[offset:]
    acc0[0] = acc0[20] = -0.0
    grad_out = torch.tensor([0.37], dtype=torch.float32, device=DEV)
    n_valid = torch.tensor([977.0], dtype=torch.float32, device=DEV)

    want = acc0.clone() if accumulate else torch.zeros(n, dtype=torch.float32, device=DEV)
    for b in bits:
        want += b.view(torch.bfloat16).float()
    if scaled:
        want.mul_(grad_out[0] / n_valid[0])

    got_base = torch.full((n + offset,), 123.0, dtype=torch.float32, device=DEV)
    got = got_base[offset:]
    if accumulate:
        got.copy_(acc0)
    ptrs = (ctypes.c_void_p * k)(*[b.data_ptr() for b in bits])
    rc = _native.lib().tm_ce_grad_w_fold(got.data_ptr(), ptrs, k, n, accumulate,
                                         grad_out.data_ptr() if scaled else None,
                                         n_valid.data_ptr() if scaled else None, _native.stream_handle(DEV))
    _native.check(rc, "tm_ce_grad_w_fold")
    torch.cuda.synchronize()
    a = got.cpu().numpy().view(np.uint32)
    w = want.cpu().numpy().view(np.uint32)
    assert np.array_equal(a, w), np.argwhere(a != w)[:5]


@pytest.mark.parametrize("chunk", [700, 350, 256, 175, 128, 100, 80, 64, 40])
def test_fused_linear_ce_grad_w_equals_chunkwise_reference_ops(chunk):
    """Folding the chunks' hand-overs and deferring the last chunk change nothing: grad_W of
    the op with 1, 2, 3, 4, 7, 9 and 18 chunks (folds of 8 in forward, the rest with the last
    in backward) equals, bit for bit, the reference's chunk loop run
    on the same kernels -- zero buffer, `+=` of each chunk's bf16 grad_W, then
    `mul_(grad_out / n_valid)` (fused_linear_ce.py:67-91,117-126) -- and grad_h likewise
    (`grad_hidden[s:e] = gh`, then `mul_(scale.to(bf16))`)."""
    from torchure_amd import _native
    from torchure_amd.loss import fused_linear_cross_entropy

    g = torch.Generator(device=DEV).manual_seed(11)
    n, d, v = 700, 128, 2048
    hidden = torch.randn(n, d, device=DEV, generator=g).to(torch.bfloat16)
    weight = torch.randn(v, d, device=DEV, generator=g) * 0.05
    labels = torch.randint(0, v, (n,), device=DEV, generator=g)
    labels[::13] = -100
    h1 = hidden.clone().requires_grad_(True)
    w1 = weight.clone().requires_grad_(True)
    loss = fused_linear_cross_entropy(h1, w1, labels, -100, chunk)
    (loss * 3.0).backward()
    gh_ref, gw_ref = _chunk_loop_on_the_same_kernels(hidden, weight, labels, chunk, 3.0)
    torch.cuda.synchronize()
    assert torch.equal(w1.grad.view(torch.int32), gw_ref.view(torch.int32))
    assert torch.equal(h1.grad.view(torch.int16), gh_ref.view(torch.int16))


def _chunk_loop_on_the_same_kernels(hidden, weight, labels, chunk, grad_out):
    """The reference's chunk loop (fused_linear_ce.py:67-91,117-126) run on this build's GEMMs
    and row kernel: a zero fp32 grad_W, `+=` of each chunk's bf16 grad_W, `grad_hidden[s:e] =
    gh`, then both scaled by grad_out / n_valid (grad_h by its bf16 rounding)."""
    from torchure_amd import _native
    from torchure_amd.loss.fused_linear_ce import GradHidden, _grad_w, _logits

    n, v = hidden.shape[0], weight.shape[0]
    lib = _native.lib()
    stream = _native.stream_handle(DEV)
    w = weight.to(torch.bfloat16).contiguous()
    gw_ref = torch.zeros(weight.shape, dtype=torch.float32, device=DEV)
    gh_ref = torch.empty_like(hidden)
    row_loss = torch.empty(n, dtype=torch.float32, device=DEV)
    grad_h = GradHidden(w, [min(chunk, n - s) for s in range(0, n, chunk)], lib, stream)
    for s in range(0, n, chunk):
        e = min(s + chunk, n)
        logits = _logits(hidden[s:e], w, lib, stream)
        _native.check(lib.tm_ce_rows_bf16(logits.data_ptr(), v, labels[s:e].data_ptr(), e - s, v, -100,
                                          row_loss[s:].data_ptr(), stream), "tm_ce_rows_bf16")
        gh = torch.empty((e - s, w.shape[1]), dtype=torch.bfloat16, device=DEV)
        grad_h(logits, gh)
        gh_ref[s:e] = gh
        gw_ref += _grad_w(logits, hidden[s:e], lib, stream)
    n_valid = (labels != -100).sum().clamp_min(1)
    scale = torch.tensor(grad_out, device=DEV) / n_valid
    gw_ref.mul_(scale)
    gh_ref.mul_(scale.to(torch.bfloat16))
    return gh_ref, gw_ref


def test_default_chunking_is_the_reference_1024_rows():
    """Called without chunk_size, the op chunks by 1024 rows, the reference's default
    (fused_linear_ce.py:131): grad_W and grad_h equal the reference's chunk loop at 1024 rows
    bit for bit (2600 rows: chunks of 1024, 1024 and 552). chunk_size=None and "auto" take the
    4 GiB logits budget instead, here one chunk: the bits of chunk_size=2600."""
    from torchure_amd.loss import fused_linear_cross_entropy

    g = torch.Generator(device=DEV).manual_seed(12)
    n, d, v = 2600, 128, 2048
    hidden = torch.randn(n, d, device=DEV, generator=g).to(torch.bfloat16)
    weight = torch.randn(v, d, device=DEV, generator=g) * 0.05
    labels = torch.randint(0, v, (n,), device=DEV, generator=g)
    labels[::17] = -100

    def run(*chunk_arg):
        h = hidden.clone().requires_grad_(True)
        w = weight.clone().requires_grad_(True)
        fused_linear_cross_entropy(h, w, labels, -100, *chunk_arg).backward()
        return h.grad, w.grad

    gh, gw = run()
    gh_ref, gw_ref = _chunk_loop_on_the_same_kernels(hidden, weight, labels, 1024, 1.0)
    torch.cuda.synchronize()
    assert torch.equal(gw.view(torch.int32), gw_ref.view(torch.int32))
    assert torch.equal(gh.view(torch.int16), gh_ref.view(torch.int16))
    gh_one, gw_one = run(n)
    for auto in (None, "auto"):
        gh_a, gw_a = run(auto)
        assert torch.equal(gw_a.view(torch.int32), gw_one.view(torch.int32))
        assert torch.equal(gh_a.view(torch.int16), gh_one.view(torch.int16))
    with pytest.raises(ValueError, match="chunk_size"):
        run("large")


def test_out_of_range_label_gives_nan_loss():
    """A label outside [0, vocab) other than ignore_index is an error in the reference (its
    gather asserts on the device); here the row loss, and so the mean loss, is NaN."""
    labels = np.array([3, -1, 100000, -100, 7], dtype=np.int64)
    r = H.rng(11)
    bits = oracle.bf16_rne((r.standard_normal((5, 4096)) * 2.0).astype(np.float32)).reshape(5, 4096)
    _, loss = _ce_rows(bits, labels, -100)
    assert np.isfinite(loss[[0, 4]]).all() and loss[3] == 0.0
    assert np.isnan(loss[1]) and np.isnan(loss[2])


@pytest.mark.parametrize("v", [4096, 1001, 200000])
def test_ce_rows_edge_rows_vs_fp64(v):
    """Rows the random tests do not reach: masked vocabulary entries (-inf), a range wide
    enough that most results are denormal or zero (the full-range exp fallback), constant
    rows, large magnitudes, and a label on a -inf logit (infinite loss). On the in-register
    path (4096), the element-wise path (1001: rows not 16-byte aligned) and the two-read
    path (200000)."""
    r = H.rng(21)
    rows = []
    x = (r.standard_normal(v) * 2.0).astype(np.float32); x[::3] = -np.inf; rows.append(x)      # masked
    x = np.linspace(-200.0, 20.0, v).astype(np.float32); rows.append(x)                       # denormal tail
    rows.append(np.full(v, 1.5, dtype=np.float32))                                            # constant
    x = (r.standard_normal(v) * 1e4).astype(np.float32); rows.append(x)                       # large spread
    x = (r.standard_normal(v) + 1e30).astype(np.float32); rows.append(x)                      # huge offset
    x = (r.standard_normal(v)).astype(np.float32); x[5] = -np.inf; rows.append(x)             # label on -inf
    bits = oracle.bf16_rne(np.stack(rows)).reshape(len(rows), v)
    labels = np.array([1, v - 96, 7, 123, 99, 5], dtype=np.int64)
    grad_bits, loss = _ce_rows(bits, labels, -100)
    xd = oracle.bf16_to_f32(bits).reshape(len(rows), v).astype(np.float64)
    mx = xd.max(axis=1, keepdims=True)
    lse = (mx + np.log(np.exp(xd - mx).sum(axis=1, keepdims=True)))[:, 0]
    want_loss = lse - xd[np.arange(len(rows)), labels]
    assert np.isinf(loss[5]) and loss[5] > 0
    np.testing.assert_allclose(loss[:5], want_loss[:5], rtol=1e-6, atol=1e-6)
    probs = np.exp(xd - lse[:, None])
    probs[np.arange(len(rows)), labels] -= 1.0
    want_bits = oracle.bf16_rne(probs.astype(np.float32)).reshape(len(rows), v)
    diff = np.abs(grad_bits.astype(np.int32) - want_bits.astype(np.int32))
    assert diff.max() <= 1, (diff.max(), np.argwhere(diff > 1)[:4])
    assert np.all(grad_bits[0, ::3] == 0)  # exp(-inf) = 0 exactly


@pytest.mark.parametrize("b,s,d,v,chunk,ignore_frac,hidden_dtype", [
    (2, 128, 64, 1000, 64, 0.1, torch.bfloat16),          # uneven chunks
    (2, 256, 128, 5000, 512, 0.0, torch.bfloat16),        # one chunk
    (2, 4096, 1024, 151936, 1024, 0.05, torch.bfloat16),  # the Qwen3 head at the reference's chunk size
    (2, 4096, 1024, 151936, None, 0.05, torch.bfloat16),  # the same with this build's default (one chunk)
    (2, 4096, 1024, 151936, 4096, 0.05, torch.float32),   # the trainer's call: fp32 hidden, autocast
])
def test_reference_cases_vs_plain_cross_entropy(b, s, d, v, chunk, ignore_frac, hidden_dtype):
    """The cases and bars of the reference's own test (tests/fused_linear_ce.py:23-56): the
    op against an unfused lm_head + F.cross_entropy on fp32 logits, through autograd, with
    bf16 hidden states and an fp32 head weight: |loss difference| < 2e-3 * max(1, loss) and
    relative L2 error of both grads < 3e-2. The unfused side uses 2-D products only. The
    last case is the trainer's own call (objectives/autoregressive.py:38-44, ce_chunk_size 4096 from :21):
    fp32 hidden states with both sides run under bf16 autocast."""
    import contextlib

    import torch.nn.functional as F

    from torchure_amd.loss import fused_linear_cross_entropy

    fp32 = hidden_dtype == torch.float32
    amp = (lambda: torch.autocast("cuda", dtype=torch.bfloat16)) if fp32 else contextlib.nullcontext
    torch.manual_seed(0)
    hidden = (torch.randn(b, s, d, device=DEV, dtype=torch.bfloat16) * 0.5).to(hidden_dtype)
    weight = torch.randn(v, d, device=DEV, dtype=torch.float32) * 0.02
    labels = torch.randint(0, v, (b, s), device=DEV)
    labels[torch.rand(b, s, device=DEV) < ignore_frac] = -100

    h1 = hidden.clone().requires_grad_(True)
    w1 = weight.clone().requires_grad_(True)
    with amp():
        logits = h1.reshape(-1, d) @ w1.to(torch.bfloat16).t()
        loss_ref = F.cross_entropy(logits.float(), labels.reshape(-1), ignore_index=-100)
    loss_ref.backward()
    del logits

    h2 = hidden.clone().requires_grad_(True)
    w2 = weight.clone().requires_grad_(True)
    with amp():
        loss = fused_linear_cross_entropy(h2, w2, labels, -100, chunk)
    loss.backward()

    def rel(a, b_):
        return float((a.float() - b_.float()).norm() / b_.float().norm().clamp_min(1e-12))

    dh, dw = rel(h2.grad, h1.grad), rel(w2.grad, w1.grad)
    print(f"V={v} chunk={chunk}: loss {loss.item():.6f} vs {loss_ref.item():.6f}, rel dh {dh:.2e}, dw {dw:.2e}")
    assert abs(loss_ref.item() - loss.item()) < 2e-3 * max(1.0, loss_ref.item())
    assert dh < 3e-2
    assert dw < 3e-2
    assert h2.grad.dtype == hidden_dtype and h1.grad.dtype == hidden_dtype and w2.grad.dtype == torch.float32


@pytest.mark.parametrize("vocab", [4096, 1001, 200000])
def test_loss_only_rows_equal_gradient_rows(vocab):
    """tm_ce_rows_loss_bf16 gives the row losses of tm_ce_rows_bf16 bit for bit (register,
    element-wise and streaming paths) and leaves the logits untouched."""
    from torchure_amd import _native

    g = torch.Generator(device=DEV).manual_seed(vocab)
    rows = 29
    logits = (torch.randn(rows, vocab, device=DEV, generator=g) * 3.0).to(torch.bfloat16)
    labels = torch.randint(0, vocab, (rows,), device=DEV, generator=g)
    labels[[2, 11]] = -100
    keep = logits.clone()
    a = torch.empty(rows, device=DEV)
    b = torch.empty(rows, device=DEV)
    lib, s = _native.lib(), _native.stream_handle(DEV)
    _native.check(lib.tm_ce_rows_loss_bf16(logits.data_ptr(), vocab, labels.data_ptr(), rows, vocab, -100,
                                           a.data_ptr(), s), "tm_ce_rows_loss_bf16")
    assert torch.equal(logits.view(torch.int16), keep.view(torch.int16))
    _native.check(lib.tm_ce_rows_bf16(logits.data_ptr(), vocab, labels.data_ptr(), rows, vocab, -100,
                                      b.data_ptr(), s), "tm_ce_rows_bf16")
    assert torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("chunk", [None, 300])
def test_loss_without_grad_and_partial_grads(chunk):
    """Under torch.no_grad the op takes the loss-only path and returns the training path's
    loss bit for bit. With only the weight (or only the hidden states) requiring a
    gradient, that gradient equals the one computed with both, bit for bit, and the other
    input gets none."""
    from torchure_amd.loss import fused_linear_cross_entropy

    g = torch.Generator(device=DEV).manual_seed(3)
    n, d, v = 1000, 256, 4096
    hidden = torch.randn(n, d, device=DEV, generator=g).to(torch.bfloat16)
    weight = torch.randn(v, d, device=DEV, generator=g) * 0.05
    labels = torch.randint(0, v, (n,), device=DEV, generator=g)
    labels[::23] = -100

    h = hidden.clone().requires_grad_(True)
    w = weight.clone().requires_grad_(True)
    loss = fused_linear_cross_entropy(h, w, labels, -100, chunk)
    loss.backward()
    with torch.no_grad():
        eval_loss = fused_linear_cross_entropy(h, w, labels, -100, chunk)
    assert not eval_loss.requires_grad
    assert eval_loss.view(torch.int32).item() == loss.detach().view(torch.int32).item()
    # inputs that require no gradient: the loss-only path too
    plain = fused_linear_cross_entropy(hidden, weight, labels, -100, chunk)
    assert plain.view(torch.int32).item() == loss.detach().view(torch.int32).item()

    w_only = weight.clone().requires_grad_(True)
    l1 = fused_linear_cross_entropy(hidden, w_only, labels, -100, chunk)
    l1.backward()
    assert torch.equal(w_only.grad, w.grad)
    assert l1.detach().view(torch.int32).item() == loss.detach().view(torch.int32).item()

    h_only = hidden.clone().requires_grad_(True)
    l2 = fused_linear_cross_entropy(h_only, weight, labels, -100, chunk)
    l2.backward()
    assert torch.equal(h_only.grad.view(torch.int16), h.grad.view(torch.int16))


@pytest.mark.parametrize("chunk", [None, 300])
def test_fp32_hidden_under_autocast(chunk):
    """fp32 hidden states inside bf16 autocast, the reference trainer's call: the products
    run on autocast's bf16 casts and grad_hidden is fp32 = float(bf16 GEMM result) * scale
    (fused_linear_ce.py:68,80,120). With 512 valid rows the scale is a power of two, so both
    scalings are exact and the fp32 path's results follow bit for bit from the bf16 path's on
    hidden.to(bf16): the same loss, the same grad_W, and grad_h widened exactly. Against the
    reference composition run under autocast the bars of the composition test hold, and fp16
    autocast is refused."""
    from torchure_amd.loss import fused_linear_cross_entropy

    g = torch.Generator(device=DEV).manual_seed(11)
    n, d, v = 1000, 256, 4096
    hidden = torch.randn(n, d, device=DEV, generator=g)
    weight = torch.randn(v, d, device=DEV, generator=g) * 0.05
    labels = torch.randint(0, v, (n,), device=DEV, generator=g)
    labels[torch.randperm(n, device=DEV, generator=g)[:n - 512]] = -100

    hb = hidden.to(torch.bfloat16).requires_grad_(True)
    wb = weight.clone().requires_grad_(True)
    loss_b = fused_linear_cross_entropy(hb, wb, labels, -100, chunk)
    loss_b.backward()

    hf = hidden.clone().requires_grad_(True)
    wf = weight.clone().requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        loss_f = fused_linear_cross_entropy(hf, wf, labels, -100, chunk)
    loss_f.backward()
    assert hf.grad.dtype == torch.float32 and wf.grad.dtype == torch.float32
    assert loss_f.dtype == torch.float32
    assert loss_f.detach().view(torch.int32).item() == loss_b.detach().view(torch.int32).item()
    assert torch.equal(wf.grad.view(torch.int32), wb.grad.view(torch.int32))
    assert torch.equal(hf.grad.view(torch.int32), hb.grad.float().view(torch.int32))

    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        eval_loss = fused_linear_cross_entropy(hidden, weight, labels, -100, chunk)
    assert eval_loss.view(torch.int32).item() == loss_b.detach().view(torch.int32).item()

    # a scale that is not a power of two, against the reference composition under autocast
    labels2 = labels.clone()
    labels2[::37] = -100
    h2 = hidden.clone().requires_grad_(True)
    w2 = weight.clone().requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        loss2 = fused_linear_cross_entropy(h2, w2, labels2, -100, chunk)
        ref_loss, ref_gh, ref_gw = fused_linear_ce_reference(hidden, weight, labels2, -100,
                                                             chunk_size=chunk or 1024)
    loss2.backward()
    torch.cuda.synchronize()
    assert ref_gh.dtype == torch.float32
    assert abs(loss2.item() - ref_loss.item()) <= 1e-5 * abs(ref_loss.item())
    gh_err = (h2.grad - ref_gh).abs().max().item()
    gw_err = (w2.grad - ref_gw).abs().max().item()
    print(f"fp32 hidden, chunk {chunk}: loss {loss2.item():.6f} ref {ref_loss.item():.6f}, "
          f"max |d grad_h| {gh_err:.3e}, max |d grad_w| {gw_err:.3e}")
    assert gh_err <= 1e-2 * ref_gh.abs().max().item()
    assert gw_err <= 1e-2 * ref_gw.abs().max().item()

    with pytest.raises(NotImplementedError, match="autocast"), torch.autocast("cuda", dtype=torch.float16):
        fused_linear_cross_entropy(hidden, weight, labels)
    # bf16 hidden under fp16 autocast: autocast would make the logits fp16, so it is refused too
    with pytest.raises(NotImplementedError, match="autocast"), torch.autocast("cuda", dtype=torch.float16):
        fused_linear_cross_entropy(hidden.to(torch.bfloat16).requires_grad_(True), weight, labels)
    with pytest.raises(NotImplementedError, match="autocast"), torch.autocast("cuda", dtype=torch.float16):
        with torch.no_grad():
            fused_linear_cross_entropy(hidden.to(torch.bfloat16), weight, labels)


@pytest.mark.parametrize("ignore_index", [7, 0])
def test_ignore_index_inside_the_vocabulary(ignore_index):
    """ignore_index may be a real class id (F.cross_entropy semantics, fused_linear_ce.py:40,86):
    rows labelled with it are left out of the loss, the mean and both gradients, and the class
    is still scored for the other rows. Checked against the reference composition with the same
    ignore_index, in one chunk and in several, at that test's bars."""
    from torchure_amd.loss import fused_linear_cross_entropy

    g = torch.Generator(device=DEV).manual_seed(100 + ignore_index)
    n, d, v = 700, 128, 1000
    hidden = torch.randn(n, d, device=DEV, generator=g).to(torch.bfloat16)
    weight = torch.randn(v, d, device=DEV, generator=g) * 0.05
    labels = torch.randint(0, v, (n,), device=DEV, generator=g)
    labels[labels == ignore_index] = (ignore_index + 2) % v  # only the rows set below are ignored
    labels[1::9] = (ignore_index + 1) % v  # the neighbouring class, scored as usual
    labels[::5] = ignore_index
    for chunk in (None, 128):
        h = hidden.clone().requires_grad_(True)
        w = weight.clone().requires_grad_(True)
        loss = fused_linear_cross_entropy(h, w, labels, ignore_index, chunk)
        loss.backward()
        ref_loss, ref_gh, ref_gw = fused_linear_ce_reference(hidden, weight, labels, ignore_index,
                                                             chunk_size=chunk or 1024)
        torch.cuda.synchronize()
        assert abs(loss.item() - ref_loss.item()) <= 1e-5 * abs(ref_loss.item())
        assert (h.grad[::5] == 0).all()  # ignored rows get no gradient
        assert (h.grad[1::5].abs().sum(dim=1) > 0).all()
        gh_err = (h.grad.float() - ref_gh.float()).abs().max().item()
        gw_err = (w.grad - ref_gw).abs().max().item()
        assert gh_err <= 1e-2 * ref_gh.float().abs().max().item()
        assert gw_err <= 1e-2 * ref_gw.abs().max().item()
        with torch.no_grad():
            ev = fused_linear_cross_entropy(hidden, weight, labels, ignore_index, chunk)
        assert ev.view(torch.int32).item() == loss.detach().view(torch.int32).item()


def test_non_contiguous_inputs_give_the_contiguous_bits():
    """hidden as a transposed view and a strided weight slice: the op works on contiguous
    copies (as torch's products accept any strides), so loss and both gradients equal the
    contiguous call bit for bit, and the gradients reach the views' bases."""
    from torchure_amd.loss import fused_linear_cross_entropy

    g = torch.Generator(device=DEV).manual_seed(21)
    n, d, v = 600, 128, 3000
    hidden = torch.randn(n, d, device=DEV, generator=g).to(torch.bfloat16)
    weight = torch.randn(v, d, device=DEV, generator=g) * 0.05
    labels = torch.randint(0, v, (n,), device=DEV, generator=g)
    labels[::11] = -100

    h1 = hidden.clone().requires_grad_(True)
    w1 = weight.clone().requires_grad_(True)
    l1 = fused_linear_cross_entropy(h1, w1, labels, -100, 256)
    l1.backward()

    hbase = hidden.t().contiguous().requires_grad_(True)  # (d, n); its transpose is (n, d), strided
    wbase = torch.zeros(v, 2 * d, device=DEV)
    wbase[:, ::2] = weight
    wbase.requires_grad_(True)
    h2, w2 = hbase.t(), wbase[:, ::2]
    assert not h2.is_contiguous() and not w2.is_contiguous()
    l2 = fused_linear_cross_entropy(h2, w2, labels, -100, 256)
    l2.backward()
    torch.cuda.synchronize()
    assert l1.detach().view(torch.int32).item() == l2.detach().view(torch.int32).item()
    assert torch.equal(hbase.grad.t().contiguous().view(torch.int16), h1.grad.view(torch.int16))
    assert torch.equal(wbase.grad[:, ::2].contiguous().view(torch.int32), w1.grad.view(torch.int32))
    assert torch.count_nonzero(wbase.grad[:, 1::2]).item() == 0


@pytest.mark.parametrize("vocab", [4096, 1001, 151936])
def test_ce_rows_f32_kernel_vs_fp64(vocab):
    """tm_ce_rows_f32 (fp32 logits, the fp32-hidden path outside autocast) against an fp64
    restatement of fused_linear_ce.py:39-51 on the same fp32 logits: row losses within 1e-6
    relative; gradients within 2e-6 relative of exp(x - lse), plus the fp32 rounding of lse and
    of x - lse (2^-23 of their magnitudes), plus 1e-7 absolute at the label (p - 1 cancels);
    ignored rows exactly zero; tm_ce_rows_loss_f32 gives the same loss bits
    and leaves the logits untouched. V = 1001 takes the element-wise path (rows not 16-byte
    aligned), and rows hold -inf entries and a wide range."""
    from torchure_amd import _native

    g = torch.Generator(device=DEV).manual_seed(vocab)
    rows = 64
    x = torch.randn(rows, vocab, device=DEV, generator=g) * 4.0
    x[3, ::7] = float("-inf")
    x[5] *= 20.0
    labels = torch.randint(0, vocab, (rows,), device=DEV, generator=g)
    labels[::9] = -100
    labels[3] = 1  # a finite entry of the masked row
    lib, stream = _native.lib(), _native.stream_handle(DEV)
    work = x.clone()
    loss = torch.empty(rows, dtype=torch.float32, device=DEV)
    _native.check(lib.tm_ce_rows_f32(work.data_ptr(), vocab, labels.data_ptr(), rows, vocab, -100,
                                     loss.data_ptr(), stream), "tm_ce_rows_f32")
    ro = x.clone()
    loss2 = torch.empty(rows, dtype=torch.float32, device=DEV)
    _native.check(lib.tm_ce_rows_loss_f32(ro.data_ptr(), vocab, labels.data_ptr(), rows, vocab, -100,
                                          loss2.data_ptr(), stream), "tm_ce_rows_loss_f32")
    xd = x.double()
    lse = torch.logsumexp(xd, dim=1)
    valid = labels != -100
    picked = xd.gather(1, labels.clamp(min=0)[:, None])[:, 0]
    want_loss = torch.where(valid, lse - picked, torch.zeros_like(lse))
    p = torch.exp(xd - lse[:, None])
    want = p.clone()
    idx = valid.nonzero()[:, 0]
    want[idx, labels[idx]] -= 1.0
    want[~valid] = 0.0
    torch.cuda.synchronize()
    assert torch.equal(ro, x)
    assert torch.equal(loss.view(torch.int32), loss2.view(torch.int32))
    torch.testing.assert_close(loss.double(), want_loss, rtol=1e-6, atol=1e-6)
    err = (work.double() - want).abs()
    # fp32 rounding of lse (half an ulp of |lse|) and of the difference x - lse move the
    # exponent by up to (|lse| + |x - lse|) * 2^-24 each
    dist = (xd - lse[:, None]).abs()
    dist = torch.where(torch.isfinite(dist), dist, torch.zeros_like(dist))  # -inf entries: p = 0 exactly
    rel = 2e-6 + (lse.abs()[:, None] + dist) * 2.0 ** -23
    bound = p * rel + 1e-7 * (want != p).double() + 1e-30
    bound[~valid] = 0.0
    assert bool((err <= bound).all()), float((err / bound.clamp_min(1e-300)).max())
    assert bool((work[~valid] == 0).all())


@pytest.mark.parametrize("vocab", [
    1, 4, 1024, 1028, 2048, 2052, 4096, 4100, 8192, 8196, 12288, 12292, 20480,  # 1 to 20 vectors, four waves
    20484, 24580, 40960, 40964, 49156, 81920,  # eight and sixteen waves
    81924, 90001,                              # too long for registers
    3001, 10241, 81922,                        # packed rows off 16 bytes
])
def test_ce_rows_f32_at_the_edges_of_the_row_shapes(vocab):
    """tm_ce_rows_f32 on both sides of every change of its threads and vectors a row, rows packed
    (off 16 bytes where the vocabulary is) and 32 elements apart: losses and gradients against
    fp64, the loss-only pass bit for bit equal, -inf, NaN, +inf and the type's lowest value where
    only some threads or batches see them, nothing written past the vocabulary. Bounds: a sum of
    positive terms is off by at most one rounding of 2^-24 per addition on the longest chain: 3 a
    vector, 7 rescales of 5 (with their exponentials) and 10 additions over the lanes, or vocab /
    1024 online steps of 5; lse moves by that plus its own roundings and the difference's."""
    from torchure_amd import _native

    lib, st = _native.lib(), _native.stream_handle(DEV)
    g = torch.Generator(device=DEV).manual_seed(vocab)
    rows, low = 13, torch.finfo(torch.float32).min
    x = torch.randn(rows, vocab, device=DEV, generator=g) * 3.0
    x[1, : vocab // 2] = float("-inf")
    x[2, : max(0, vocab - 2)] = low          # whole threads at the mask value
    x[3] = 3.3e38
    x[4] -= 300.0
    x[5, vocab // 3] = float("nan")
    x[6] = float("-inf")
    x[6, vocab - 1] = float("nan")
    x[7, vocab // 2] = float("inf")
    labels = torch.randint(0, vocab, (rows,), device=DEV, generator=g)
    labels[1:3] = vocab - 1
    labels[7] = 0 if vocab > 1 else -100     # not the +inf entry
    labels[8] = -100
    xd = x.double()
    lse = torch.logsumexp(xd, dim=1)
    want = lse - xd.gather(1, labels.clamp_min(0)[:, None])[:, 0]
    want[labels == -100] = 0.0
    probs = torch.exp(xd - lse[:, None])
    grads = probs.clone()
    grads[torch.arange(rows), labels.clamp_min(0)] -= 1.0
    grads[labels == -100] = 0.0
    fine = [r for r in range(rows) if r not in (5, 6, 7)]
    chain = max(20, vocab // 4096) * 3 + max(7, vocab // 16384) * 5 + 10 + vocab // 1024 * 5 * (vocab % 4 != 0)
    tol = 2.0 ** -24 * (chain + 4 * lse.abs())
    for ld in (vocab, -(-vocab // 32) * 32):
        buf = torch.full((rows, ld), 7.0, device=DEV)
        buf[:, :vocab] = x
        loss_only, loss = torch.empty(rows, device=DEV), torch.empty(rows, device=DEV)
        for fn, out in ((lib.tm_ce_rows_loss_f32, loss_only), (lib.tm_ce_rows_f32, loss)):
            _native.check(fn(buf.data_ptr(), ld, labels.data_ptr(), rows, vocab, -100, out.data_ptr(), st), "rows")
        assert torch.equal(loss_only.view(torch.int32), loss.view(torch.int32))
        assert (buf[:, vocab:] == 7.0).all()
        assert ((loss.double() - want).abs() <= tol)[fine].all(), (loss, want)
        assert loss[5].isnan() and loss[6].isnan()
        got = buf[:, :vocab].double()
        dist = (xd - lse[:, None]).abs().clamp_max(200.0)  # further off the probability is 0 either way
        off = (got - grads).abs() - (probs * (2.0 * tol[:, None] + 2.0 ** -22 * (1 + dist)) + 2.0 ** -23)
        assert (off <= 0)[fine].all(), off[fine].max()
        assert got[5].isnan().all() and got[6].isnan().all()
        if vocab > 1:  # as torch.logsumexp: lse = +inf, no probability anywhere but at the +inf entry
            assert loss[7] == float("inf")
            rest = torch.arange(vocab, device=DEV) != vocab // 2
            rest[0] = False
            assert (got[7, rest] == 0).all() and got[7, vocab // 2].isnan()


@pytest.mark.parametrize("n", [1, 63, 64 * 64, 64 * 64 + 1, 300_001])
def test_finish_scales_fp32_grad_h_in_place(n):
    """tm_ce_finish with an fp32 grad_h: both gradients times grad_out / n_valid, the bits of the
    fp32 product, in one launch, for sizes on both sides of a workgroup's slice."""
    from torchure_amd import _native

    g = torch.Generator(device=DEV).manual_seed(n)
    gh, gw = torch.randn(n + 1, device=DEV, generator=g), torch.randn(n + 5, device=DEV, generator=g)
    gh[0], gw[0] = float("inf"), -0.0
    keep = gh[n].clone()
    go, out2 = torch.tensor(3.0, device=DEV), torch.tensor([5.0, 7.0], device=DEV)
    want_h, want_w = gh[:n] * (go / out2[1]), gw * (go / out2[1])
    _native.ce_host().ce_backward(go, out2, gh[:n], 2, gw, [], True, _native.stream_handle(DEV))
    assert torch.equal(gh[:n].view(torch.int32), want_h.view(torch.int32)) and gh[n] == keep
    assert torch.equal(gw.view(torch.int32), want_w.view(torch.int32))


@pytest.mark.parametrize("chunk", [None, 300])
def test_fp32_hidden_without_autocast(chunk):
    """fp32 hidden states outside autocast: the reference runs fp32 GEMMs on w =
    weight.to(fp32) (fused_linear_ce.py:38,52,57,65) and returns fp32 gradients. Against the
    reference composition (the same torch calls) on the same device: loss within 1e-6
    relative, both gradients within 1e-5 of their scale; against an fp64 unfused cross
    entropy: loss within 1e-5 relative and gradients within 1e-4 relative L2. The loss-only
    call gives the training loss bits; a bf16 weight gets its gradient as autograd hands it
    over (fp32 cast to the weight's dtype), as in the reference."""
    import torch.nn.functional as F

    from torchure_amd.loss import fused_linear_cross_entropy

    g = torch.Generator(device=DEV).manual_seed(23)
    n, d, v = 1000, 256, 4096
    hidden = torch.randn(n, d, device=DEV, generator=g)
    weight = torch.randn(v, d, device=DEV, generator=g) * 0.05
    labels = torch.randint(0, v, (n,), device=DEV, generator=g)
    labels[::37] = -100
    h1 = hidden.clone().requires_grad_(True)
    w1 = weight.clone().requires_grad_(True)
    loss = fused_linear_cross_entropy(h1, w1, labels, -100, chunk)
    (loss * 2.0).backward()
    assert loss.dtype == torch.float32 and h1.grad.dtype == torch.float32 and w1.grad.dtype == torch.float32
    ref_loss, ref_gh, ref_gw = fused_linear_ce_reference(hidden, weight, labels, -100, chunk_size=chunk or n)
    torch.cuda.synchronize()
    assert abs(loss.item() - ref_loss.item()) <= 1e-6 * abs(ref_loss.item())
    assert (h1.grad - 2.0 * ref_gh).abs().max().item() <= 1e-5 * ref_gh.abs().max().item() * 2.0
    assert (w1.grad - 2.0 * ref_gw).abs().max().item() <= 1e-5 * ref_gw.abs().max().item() * 2.0

    hd = hidden.double().requires_grad_(True)
    wd = weight.double().requires_grad_(True)
    ld = F.cross_entropy(hd @ wd.t(), labels, ignore_index=-100)
    (ld * 2.0).backward()

    def rel(a, b):
        return float((a.double() - b).norm() / b.norm())

    assert abs(loss.item() - ld.item()) <= 1e-5 * ld.item()
    assert rel(h1.grad, hd.grad) < 1e-4 and rel(w1.grad, wd.grad) < 1e-4

    with torch.no_grad():
        ev = fused_linear_cross_entropy(hidden, weight, labels, -100, chunk)
    assert ev.view(torch.int32).item() == loss.detach().view(torch.int32).item()

    wb = weight.to(torch.bfloat16).requires_grad_(True)
    h2 = hidden.clone().requires_grad_(True)
    fused_linear_cross_entropy(h2, wb, labels, -100, chunk).backward()
    assert wb.grad.dtype == torch.bfloat16 and h2.grad.dtype == torch.float32
    with pytest.raises(NotImplementedError, match="float16"):
        fused_linear_cross_entropy(hidden.half().requires_grad_(True), weight, labels)


def test_fp32_weight_with_current_working_copy():
    """An fp32 head weight with an attached bf16 working copy: while the copy is current the op
    reads it instead of casting the master, with the cast's bits (loss, grad_h and grad_W equal a
    weight without a copy, bit for bit, training and loss-only); the copy really is what the op
    reads (bytes overwritten behind autograd's back change the loss, and a refresh restores it);
    a master modified in place makes the copy stale and the op casts again; after AdamW.step()
    the copy is current again, and a copy modified in place through torch is not taken."""
    import torchure_amd as ta
    from torchure_amd import _native
    from torchure_amd.loss import fused_linear_cross_entropy
    from torchure_amd.optimizer.working import current_copy

    g = torch.Generator(device=DEV).manual_seed(31)
    n, d, v = 1500, 256, 6000
    hidden = torch.randn(n, d, device=DEV, generator=g).to(torch.bfloat16)
    labels = torch.randint(0, v, (n,), device=DEV, generator=g)
    labels[::9] = -100
    master = torch.nn.Parameter(torch.randn(v, d, device=DEV, generator=g) * 0.05)
    (copy,) = ta.attach_bf16_working_params([master])

    def run(weight):
        h = hidden.clone().requires_grad_(True)
        loss = fused_linear_cross_entropy(h, weight, labels, -100, 512)
        gh, gw = torch.autograd.grad(loss, (h, weight))
        with torch.no_grad():
            eval_loss = fused_linear_cross_entropy(hidden, weight, labels, -100, 512)
        return loss.detach(), gh, gw, eval_loss

    def same(a, b):
        return all(torch.equal(x.view(torch.int32) if x.dtype == torch.float32 else x.view(torch.int16),
                               y.view(torch.int32) if y.dtype == torch.float32 else y.view(torch.int16))
                   for x, y in zip(a, b))

    plain = torch.nn.Parameter(master.detach().clone())
    assert same(run(master), run(plain))
    assert torch.equal(run(master)[0], run(plain)[3])  # loss-only gives the training bits

    # overwrite the copy's bytes without an autograd version bump: the op reads the copy
    junk = (torch.randn(v, d, device=DEV, generator=g) * 0.05).to(torch.bfloat16)
    _native.check(_native.lib().tm_stream_copy(copy.data_ptr(), junk.data_ptr(), junk.numel() * 2,
                                               _native.stream_handle(DEV)), "tm_stream_copy")
    torch.cuda.synchronize()
    assert not torch.equal(run(master)[0], run(plain)[0])
    ta.refresh_bf16_working_params([master])
    assert same(run(master), run(plain))

    # a master changed in place: the copy is stale, the op casts the master again
    with torch.no_grad():
        master.mul_(1.5)
        plain.mul_(1.5)
    _native.check(_native.lib().tm_stream_copy(copy.data_ptr(), junk.data_ptr(), junk.numel() * 2,
                                               _native.stream_handle(DEV)), "tm_stream_copy")
    torch.cuda.synchronize()
    assert same(run(master), run(plain))
    # AdamW.step() writes the copy with the master, so the op reads it again afterwards
    ta.refresh_bf16_working_params([master])
    opt = ta.AdamW([master], lr=1e-3, fused=True)
    master.grad = torch.randn(v, d, device=DEV, generator=g) * 1e-3
    opt.step()
    with torch.no_grad():
        plain.copy_(master)
    assert current_copy(master) is copy
    assert same(run(master), run(plain))
    # a copy changed in place through torch is no longer taken for the cast
    with torch.no_grad():
        copy.add_(1.0)
    assert current_copy(master) is None
    assert same(run(master), run(plain))


def test_offset_working_copy_is_not_taken():
    """A current bf16 working copy that starts 2 bytes past a 16-byte boundary (the optimizer
    accepts copies at any offset) is not read by the op, whose kernels read the weight in
    16-byte vectors: the op casts the master instead and gives the bits of a weight without a
    copy, training and loss-only."""
    from torchure_amd.loss import fused_linear_cross_entropy
    from torchure_amd.loss.fused_linear_ce import _bf16_weight
    from torchure_amd.optimizer.working import current_copy, mark_current

    g = torch.Generator(device=DEV).manual_seed(37)
    n, d, v = 1024, 256, 4096
    hidden = torch.randn(n, d, device=DEV, generator=g).to(torch.bfloat16)
    labels = torch.randint(0, v, (n,), device=DEV, generator=g)
    master = torch.nn.Parameter(torch.randn(v, d, device=DEV, generator=g) * 0.05)
    pool = torch.zeros(v * d + 8, dtype=torch.bfloat16, device=DEV)
    copy = pool[1:1 + v * d].view(v, d)
    assert copy.data_ptr() % 16 == 2
    copy.copy_(master.detach().to(torch.bfloat16))
    master._tm_working = copy
    mark_current(master, copy)
    assert current_copy(master) is copy
    assert _bf16_weight(master).data_ptr() % 16 == 0
    plain = torch.nn.Parameter(master.detach().clone())

    def run(weight):
        h = hidden.clone().requires_grad_(True)
        loss = fused_linear_cross_entropy(h, weight, labels, -100, 512)
        gh, gw = torch.autograd.grad(loss, (h, weight))
        with torch.no_grad():
            eval_loss = fused_linear_cross_entropy(hidden, weight, labels, -100, 512)
        return loss.detach(), gh, gw, eval_loss

    for x, y in zip(run(master), run(plain)):
        assert torch.equal(x, y)


def test_two_calls_on_two_streams_equal_sequential():
    """Two calls issued back to back from the host on two streams, with no synchronisation
    between them, give the bits of the same two calls run one after the other on one stream:
    each call's stream waits for the previous call's work on the device (CallOrder), so the
    two calls' GEMMs never run at the same time. The shapes use the Qwen3 head's width and the
    reference's 1024-row chunks."""
    from torchure_amd.loss import fused_linear_cross_entropy

    g = torch.Generator(device=DEV).manual_seed(41)
    n, d, v = 2048, 1024, 32768
    inputs = []
    for _ in range(2):
        hidden = torch.randn(n, d, device=DEV, generator=g).to(torch.bfloat16)
        weight = (torch.randn(v, d, device=DEV, generator=g) * 0.02).to(torch.bfloat16)
        labels = torch.randint(0, v, (n,), device=DEV, generator=g)
        inputs.append((hidden, weight, labels))

    def one(hidden, weight, labels):
        h = hidden.clone().requires_grad_(True)
        w = weight.clone().requires_grad_(True)
        loss = fused_linear_cross_entropy(h, w, labels, -100, 1024)
        loss.backward()
        return loss.detach(), h.grad, w.grad

    torch.cuda.synchronize()
    seq = [one(*x) for x in inputs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(DEV), torch.cuda.Stream(DEV)]
    for s in streams:
        s.wait_stream(torch.cuda.current_stream(DEV))
    out = []
    for s, x in zip(streams, inputs):
        with torch.cuda.stream(s):
            out.append(one(*x))
    torch.cuda.synchronize()
    for a, b in zip(seq, out):
        for x, y in zip(a, b):
            assert torch.equal(x, y)


@pytest.mark.parametrize("mode", ["bf16", "autocast"])
@pytest.mark.parametrize("n,chunk", [(640, 256), (256, 256), (2304, 256)])
def test_native_chunk_loop_equals_the_unpadded_loop(mode, n, chunk):
    """The native loop on padded logits and the Python loop on unpadded ones, on shapes that need
    no padding (every kernel then runs on the same operands): the same bits of loss, counts,
    gradients and hand-over (1, 3 and 9 chunks: one fold), with and without each gradient."""
    from torchure_amd.loss import fused_linear_ce as fce

    g = torch.Generator(device=DEV).manual_seed(n)
    d, v = 256, 4096
    hidden = torch.randn(n, d, device=DEV, generator=g)
    hidden = hidden if mode == "autocast" else hidden.to(torch.bfloat16)
    weight = torch.randn(v, d, device=DEV, generator=g) * 0.05
    labels = torch.randint(0, v, (n,), device=DEV, generator=g)
    labels[::9] = -100
    bits = {torch.float32: torch.int32, torch.bfloat16: torch.int16}
    for want_h, want_w in ((True, True), (True, False), (False, True)):
        a = fce._run_chunks(hidden, weight, labels, -100, chunk, mode, True, want_h, want_w)
        b = fce._chunks_unpadded(hidden, weight, labels, -100, n, v, chunk, mode, want_h, want_w)
        assert a[5] == b[5] and len(a[4]) == len(b[4])
        for x, y in zip([*a[:4], *a[4]], [*b[:4], *b[4]]):
            assert (x is None) == (y is None)
            assert x is None or torch.equal(x.view(bits[x.dtype]), y.view(bits[y.dtype]))
    loss = fce._run_chunks(hidden, weight, labels, -100, chunk, mode, False, False, False)[0]
    assert torch.equal(loss.view(torch.int32), a[0].view(torch.int32))


def test_operands_the_native_loop_does_not_read_as_they_are():
    """Weights that are strided, of another dtype or off 16 bytes, and hidden states off 16 bytes:
    the op gives the gradients of the plain call on the same values (the same bits where the
    products run on the same kernels), and a failed native call raises NativeError."""
    from torchure_amd import _native
    from torchure_amd.loss import fused_linear_cross_entropy

    g = torch.Generator(device=DEV).manual_seed(5)
    n, d, v = 384, 128, 1024
    hidden = torch.randn(n, d, device=DEV, generator=g).to(torch.bfloat16)
    weight = (torch.randn(v, d, device=DEV, generator=g) * 0.05).to(torch.bfloat16)
    labels = torch.randint(0, v, (n,), device=DEV, generator=g)

    def run(h, w):
        h, w = h.detach().requires_grad_(True), w.detach().requires_grad_(True)
        loss = fused_linear_cross_entropy(h, w, labels, -100, 128)
        loss.backward()
        return loss.detach(), h.grad, w.grad.to(torch.bfloat16)  # a bf16 weight's gradient is rounded

    def off16(t):
        buf = torch.empty(t.numel() + 8, dtype=t.dtype, device=DEV)
        out = buf[1: 1 + t.numel()].view(t.shape)
        out.copy_(t)
        return out

    plain = run(hidden, weight)
    strided = torch.empty(d, v, dtype=torch.bfloat16, device=DEV).t()
    strided.copy_(weight)
    for h, w, same in ((hidden, weight.float(), True), (hidden, strided, True), (hidden, weight.double(), True),
                       (off16(hidden), weight, False), (hidden, off16(weight), False)):
        for x, y in zip(run(h, w), plain):
            if same:
                assert torch.equal(x.view(torch.int32 if x.dtype == torch.float32 else torch.int16),
                                   y.view(torch.int32 if y.dtype == torch.float32 else torch.int16))
            else:  # library products: the last bit of some bf16 results
                torch.testing.assert_close(x.float(), y.float(), rtol=2.0 ** -7, atol=2.0 ** -16)
    with pytest.raises(_native.NativeError, match="tm_ce_logits_ld_bf16"):
        _native.ce_host().ce_forward(hidden, weight, False, False, labels, -100, 128, 1, (128, 128), 64, (False, False),
                                     True, True, True, 8, 1 << 30, _native.stream_handle(DEV))


def _same_bits(a, b):
    for x, y in zip([*a[:4], *a[4]], [*b[:4], *b[4]]):
        assert (x is None) == (y is None)
        kind = None if x is None else torch.int32 if x.dtype == torch.float32 else torch.int16
        assert x is None or torch.equal(x.view(kind), y.view(kind))


@pytest.mark.parametrize("n,d,v,chunk", [
    (2500, 192, 4001, 1024),  # one group, a ragged last chunk and vocabulary
    (1300, 128, 1000, 128),   # 11 chunks (a fold among them), the last of 20 rows
    (17000, 64, 300, 1024),   # more rows than a group takes: two groups
    (900, 128, 1000, 200),    # chunks with padding of their own run one by one
])
def test_logits_of_several_chunks_together_keep_the_bits(monkeypatch, n, d, v, chunk):
    """The logits and the row pass of several chunks as one launch each, against chunk by chunk."""
    from torchure_amd.loss import fused_linear_ce as fce

    g = torch.Generator(device=DEV).manual_seed(n)
    hidden = torch.randn(n, d, device=DEV, generator=g)
    weight = torch.randn(v, d, device=DEV, generator=g) * 0.05
    labels = torch.randint(0, v, (n,), device=DEV, generator=g)
    labels[::9] = -100

    def run():
        return [fce._run_chunks(hidden, weight, labels, -100, chunk, "autocast", grad, grad, grad) for grad in (True, False)]

    together = run()
    assert fce.group_chunks(n, chunk, v, True) == (1 if chunk == 200 else min(-(-n // chunk), 9 if n == 17000 else 99))
    monkeypatch.setattr(fce, "GROUP_BYTES", 0)
    for a, b in zip(together, run()):
        _same_bits(a, b)


def _release_memory():
    """Gives the allocator's free memory back, the rest of segments that only hold a library's
    workspace too, so that what a test then holds lies in memory of its own and a limit on what is
    reserved is a limit on what is to be had."""
    torch.cuda.synchronize()
    torch._C._cuda_clearCublasWorkspaces()
    torch.cuda.empty_cache()
    assert torch.cuda.memory_reserved(DEV) - torch.cuda.memory_allocated(DEV) < 64 << 20


def test_logits_of_several_chunks_run_one_by_one_where_memory_is_short():
    """A call that fits with one chunk's logits still does: a group whose logits cannot be had is
    run chunk by chunk, with the same bits. The limit is the process's own, set on the allocator."""
    from torchure_amd.loss import fused_linear_ce as fce

    _release_memory()
    n, d, v, chunk = 8192, 64, 16384, 1024  # 32 MiB of logits a chunk, 256 MiB together
    hidden = torch.randn(n, d, device=DEV).to(torch.bfloat16)
    weight = (torch.randn(v, d, device=DEV) * 0.05).to(torch.bfloat16)
    labels = torch.randint(0, v, (n,), device=DEV)
    assert fce.group_chunks(n, chunk, v, True) == 8
    want = fce._run_chunks(hidden, weight, labels, -100, chunk, "bf16", True, True, True)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(DEV).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(DEV) + (200 << 20)) / total, DEV)
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(256 << 20, dtype=torch.uint8, device=DEV)
        got = fce._run_chunks(hidden, weight, labels, -100, chunk, "bf16", True, True, True)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, DEV)
    _same_bits(got, want)


def _with_memory_limit(extra, call):
    """``call`` with ``extra`` bytes to be had beyond what is reserved now (the allocator's own limit
    for this process, none of the GPU's)."""
    _release_memory()
    total = torch.cuda.get_device_properties(DEV).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(DEV) + extra) / total, DEV)
        return call()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, DEV)


@pytest.mark.parametrize("n,d,v,chunk,unpadded", [
    (4096, 256, 65536, 1024, False),  # 128 MiB of logits a chunk, 512 together, 32 a grad_W
    (16320, 512, 4128, 16320, True),  # one chunk of 128 MiB, and 56 for grad_W's split sums
])
def test_forward_goes_on_where_memory_is_short_for_what_follows_the_logits(monkeypatch, n, d, v, chunk, unpadded):
    """A group's logits that can be had, and then no grad_W beside them: the call goes on with one
    chunk's logits at a time, with the same bits. And with no room for a workspace either: on the
    unpadded loop, whose grad_W is summed without splits (one ulp of bf16 off, and 2^-20 of the
    absolute sum, which is under 2^6 / n here)."""
    from torchure_amd import _native
    from torchure_amd.loss import fused_linear_ce as fce

    _release_memory()
    hidden = torch.randn(n, d, device=DEV).to(torch.bfloat16)
    weight = (torch.randn(v, d, device=DEV) * 0.05).to(torch.bfloat16).requires_grad_(True)
    labels = torch.randint(0, v, (n,), device=DEV)
    ws = _native.lib().tm_ce_grad_w_ld_workspace_bytes(fce.padded_rows(n), v, d)
    if unpadded:
        assert ws > 48 << 20
        limit = 2 * fce.padded_rows(n) * fce.padded_vocab(v) + ws // 2 + (8 << 20)
    else:
        assert fce.group_chunks(n, chunk, v, True) == 4
        limit = 560 << 20
    runs, loop = [], fce._chunks_unpadded
    monkeypatch.setattr(fce, "_chunks_unpadded", lambda *a: runs.append(1) or loop(*a))

    def call():
        return fce._FusedLinearCE.apply(hidden, weight, labels, -100, chunk)

    def grads(loss):
        loss.backward()
        got, weight.grad = weight.grad.cpu(), None
        return loss.detach().cpu(), got

    want = grads(call())
    assert not runs
    got = grads(_with_memory_limit(limit, call))
    assert len(runs) == unpadded
    assert torch.equal(got[0].view(torch.int32), want[0].view(torch.int32))
    if unpadded:
        torch.testing.assert_close(got[1].float(), want[1].float(), rtol=2.0 ** -7, atol=2.0 ** -14 / n)
    else:
        assert torch.equal(got[1].view(torch.int16), want[1].view(torch.int16))


def test_backward_goes_on_where_memory_is_short():
    """No room for the fp32 grad_W and the fp32 grad_hidden beside the chunk that waits for backward:
    grad_W is finished first and the chunk's memory serves grad_hidden, with the same bits."""
    from torchure_amd.loss import fused_linear_cross_entropy

    _release_memory()
    n, d, v = 8192, 1024, 8192  # 32 MiB for each result, 16 for the chunk's grad_W
    hidden = torch.randn(n, d, device=DEV, requires_grad=True)
    weight = (torch.randn(v, d, device=DEV) * 0.05).requires_grad_(True)
    labels = torch.randint(0, v, (n,), device=DEV)

    def loss():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            return fused_linear_cross_entropy(hidden, weight, labels, -100, n)

    def grads():
        out = hidden.grad.cpu(), weight.grad.cpu()
        hidden.grad = weight.grad = None
        return out

    loss().backward()
    want = grads()
    _release_memory()  # each of the call's buffers in memory of its own
    short = loss()
    _with_memory_limit(56 << 20, short.backward)
    for a, b in zip(grads(), want):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("vocab,ld,cols", [
    (20001, 20032, (0, 20000)),  # one thread's vector and its element past the last vector
    (20002, 20032, (20000, 20001)),
    (20001, 20001, (0, 1024)),   # rows off 16 bytes: one thread's first two elements
    (20001, 20001, (7, 19999)),
    (9, 32, (0, 8)),
    (90001, 90016, (0, 90000)),  # too long for registers
])
def test_ce_rows_f32_with_several_infinite_logits(vocab, ld, cols):
    """Two logits of +inf, wherever a thread meets them: lse and the loss are +inf as
    torch.logsumexp's, the gradient 0 but at the two, where inf - inf leaves NaN. A row that is -inf
    but for one element stays finite."""
    from torchure_amd import _native

    lib, st = _native.lib(), _native.stream_handle(DEV)
    x = torch.randn(3, ld, device=DEV)
    x[1] = x[2] = float("-inf")
    x[0, list(cols)] = float("inf")
    x[1, cols[1]] = 2.0
    x[2, list(cols)] = float("inf")
    labels = torch.tensor([vocab // 2, cols[1], vocab // 2], device=DEV)
    loss, loss_only = torch.empty(3, device=DEV), torch.empty(3, device=DEV)
    for fn, out in ((lib.tm_ce_rows_loss_f32, loss_only), (lib.tm_ce_rows_f32, loss)):
        _native.check(fn(x.data_ptr(), ld, labels.data_ptr(), 3, vocab, -100, out.data_ptr(), st), "rows")
    for out in (loss_only, loss):
        assert out[0] == float("inf") and out[1] == 0.0 and out[2] == float("inf"), out
    rest = torch.ones(vocab, dtype=torch.bool, device=DEV)
    rest[list(cols)] = False
    for r in (0, 2):
        assert x[r, list(cols)].isnan().all()
        want = torch.zeros(vocab, device=DEV)
        want[vocab // 2] = -1.0
        assert torch.equal(x[r, :vocab][rest], want[rest])
    assert (x[1, :vocab] == 0).all()
