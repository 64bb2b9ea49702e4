"""Performance cases: the work a training program gives this framework, through its public entry points.

Two families, each with a list of fixed cases and a generator of further cases of the same ranges:

- ``step``: the optimizer tail of a training step over a parameter list (``clip_grad_norm`` then
  ``AdamW.step``), on bf16 grads of working copies, on plain fp32 grads, or with two micro-steps
  accumulated into fp32 grads first;
- ``ce``: the fused linear + cross-entropy of a language-model head, forward and backward, or the
  loss alone (evaluation), for bf16 hidden states, fp32 hidden states under bf16 autocast, and
  fp32 hidden states without autocast.

``listed()`` and ``draw(rng)`` give cases (plain dicts), ``prepare`` the state a program holds
before the call, ``run`` one pass, ``exact`` the same outputs in 64 bits from plain torch.
"""

from __future__ import annotations

import contextlib
import math
import random

import torch

import torchure_amd as ta
from torchure_amd.loss import fused_linear_cross_entropy
from torchure_amd.workloads import numel, shapes_for

LR, BETAS, EPS, WEIGHT_DECAY, MAX_NORM = 3e-4, (0.9, 0.95), 1e-8, 0.1, 1.0
STEPS_DONE = 1000.0  # the optimizer is in its steady state


def listed():
    return [
        # The smallest training step: every launch and every microsecond of host work counts.
        {"name": "step-tiny", "family": "step", "params": "tiny", "grads": "bf16"},
        # A plain drop-in for torch.optim.AdamW over an irregular list (adapters, biases, odd
        # lengths), fp32 grads on the masters, no working copies.
        {"name": "step-irregular-fp32", "family": "step", "params": "list", "tensors": 400, "log2_max": 22,
         "list_seed": 5, "grads": "fp32"},
        # Gradient accumulation: two bf16 micro-steps into fp32 grads, clip, step, bf16 copies.
        {"name": "accumulate-0.6b", "family": "step", "params": "qwen3-0.6b", "grads": "accumulate"},
        # The large training step: bf16 grads, clip, AdamW, bf16 working copies rewritten.
        {"name": "step-4b", "family": "step", "params": "qwen3-4b", "grads": "bf16"},
        # The head of the tiny configuration at one short batch: latency and launches.
        {"name": "ce-tiny", "family": "ce", "rows": 512, "dim": 256, "vocab": 4096, "hidden": "bf16",
         "chunk": 1024, "copy": False, "grad": True},
        # The Qwen3-0.6B head called with every default (chunks of 1024 rows).
        {"name": "ce-0.6b-default", "family": "ce", "rows": 8192, "dim": 1024, "vocab": 151936, "hidden": "bf16",
         "chunk": 1024, "copy": False, "grad": True},
        # The trainer's call: fp32 hidden states under bf16 autocast, chunks of 4096 rows, the
        # head's working copy attached. A batch packed without padding has any number of tokens.
        {"name": "ce-0.6b-trainer-ragged", "family": "ce", "rows": 6001, "dim": 1024, "vocab": 151936,
         "hidden": "autocast", "chunk": 4096, "copy": True, "grad": True},
        # Evaluation: the loss alone, on what is left of a validation set.
        {"name": "ce-0.6b-eval", "family": "ce", "rows": 3000, "dim": 1024, "vocab": 151936, "hidden": "autocast",
         "chunk": 4096, "copy": True, "grad": False},
        # The Qwen3-4B head, chunks sized by the logits budget: the largest products.
        {"name": "ce-4b-auto", "family": "ce", "rows": 8192, "dim": 2560, "vocab": 151936, "hidden": "bf16",
         "chunk": "auto", "copy": False, "grad": True},
        # A medium vocabulary and width, as small models and most tests have.
        {"name": "ce-32k", "family": "ce", "rows": 4096, "dim": 2048, "vocab": 32768, "hidden": "bf16",
         "chunk": "auto", "copy": False, "grad": True},
        # A vocabulary with one token added to a round number, default chunks, ragged rows.
        {"name": "ce-odd-vocab", "family": "ce", "rows": 2500, "dim": 768, "vocab": 32001, "hidden": "autocast",
         "chunk": 1024, "copy": False, "grad": True},
        # Full-precision training of a small model (fp32 hidden states, no autocast).
        {"name": "ce-fp32", "family": "ce", "rows": 2048, "dim": 512, "vocab": 20008, "hidden": "fp32",
         "chunk": 1024, "copy": False, "grad": True},
    ]


def _log_uniform(rng: random.Random, lo: float, hi: float) -> int:
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng: random.Random):
    if rng.random() < 0.3:
        return {"family": "step", "params": "list", "tensors": _log_uniform(rng, 20, 1500),
                "log2_max": rng.randint(14, 23), "list_seed": rng.randrange(1 << 20),
                "grads": rng.choice(["bf16", "fp32", "accumulate"])}
    hidden = rng.choice(["bf16", "bf16", "autocast", "autocast", "autocast", "fp32"])
    rows = _log_uniform(rng, 64, 8192)
    dim = 64 * _log_uniform(rng, 4, 40)
    vocab = _log_uniform(rng, 1000, 151936)
    if rng.random() < 0.5:  # half the batches are padded to a round number of tokens
        rows = -(-rows // 256) * 256
    if rng.random() < 0.7:  # most vocabularies are padded to a round size
        vocab = -(-vocab // 64) * 64
    if hidden == "fp32":  # small models: fp32 products run far below the bf16 rate
        rows, dim, vocab = min(rows, 2048), min(dim, 1024), min(vocab, 32768)
    return {"family": "ce", "rows": rows, "dim": dim, "vocab": vocab, "hidden": hidden,
            "chunk": rng.choice([1024, 1024, 4096, "auto"]), "copy": hidden != "fp32" and rng.random() < 0.4,
            "grad": rng.random() < 0.8}


# ---------------------------------------------------------------------------- parameter lists


def _shapes(case):
    if case["params"] != "list":
        return shapes_for(case["params"])
    r = random.Random(case["list_seed"])
    out = []
    for _ in range(case["tensors"]):
        n = max(1, int(2.0 ** r.uniform(3.0, case["log2_max"])))
        if r.random() < 0.6:  # most lengths are whole vectors, the rest anything
            n = -(-n // 8) * 8
        out.append((n,) if r.random() < 0.4 else (1, n))
    return out


def _layout(shapes, align):
    """Offsets of tensors placed one after the other, each from a multiple of ``align`` elements."""
    offs, pos = [], 0
    for s in shapes:
        offs.append(pos)
        pos += -(-numel(s) // align) * align
    return offs, pos


ALIGN = 256   # elements from one tensor's start to the next one's, a multiple of this (1 KiB of fp32)
COPY_ALIGN = 8  # working copies lie in one buffer, each from a 16-byte boundary


def _view(flat, offset, shape):
    """A tensor of its own (not an autograd view) over part of ``flat``."""
    return torch.empty(0, dtype=flat.dtype, device=flat.device).set_(flat.untyped_storage(), offset, shape)


def _step_inputs(case, seed, device):
    """Flat fp32 masters and moments and flat grads of the steady state, from the seed alone; the
    places between tensors hold values too, which nothing reads or writes."""
    g = torch.Generator(device=device).manual_seed(seed)
    _, total = _layout(_shapes(case), ALIGN)

    def normal(std, dtype=torch.float32):
        return torch.empty(total, dtype=dtype, device=device).normal_(0.0, std, generator=g)

    flat = {"master": normal(0.02), "exp_avg": normal(1e-4), "exp_avg_sq": normal(1.0).abs_().mul_(1e-8)}
    n_grads = 2 if case["grads"] == "accumulate" else 1
    dtype = torch.float32 if case["grads"] == "fp32" else torch.bfloat16
    flat["grads"] = [normal(1e-3, dtype) for _ in range(n_grads)]
    return flat


def _prepare_step(case, seed):
    device = torch.device("cuda")
    shapes = _shapes(case)
    offs, _ = _layout(shapes, ALIGN)
    flat = _step_inputs(case, seed, device)
    params = [torch.nn.Parameter(_view(flat["master"], o, s)) for o, s in zip(offs, shapes)]
    opt = ta.build_optimizer(torch.nn.ParameterList(params), "adamw",
                             {"lr": LR, "weight_decay": WEIGHT_DECAY, "betas": BETAS, "eps": EPS, "fused": True})
    steps = torch.full((len(shapes),), STEPS_DONE, device=device)
    for i, (p, o, s) in enumerate(zip(params, offs, shapes)):
        opt.state[p] = {"step": _view(steps, i, ()), "exp_avg": _view(flat["exp_avg"], o, s),
                        "exp_avg_sq": _view(flat["exp_avg_sq"], o, s)}
    grads = [[_view(f, o, s) for o, s in zip(offs, shapes)] for f in flat["grads"]]
    out = {"master": flat["master"], "exp_avg": flat["exp_avg"], "exp_avg_sq": flat["exp_avg_sq"], "step": steps}
    state = {"case": case, "params": params, "opt": opt, "grads": grads, "out": out, "copies": None}
    if case["grads"] == "fp32":
        for p, g in zip(params, grads[0]):
            p.grad = g
        return state
    state["copies"] = copies = ta.attach_bf16_working_params(params)
    coffs, ctotal = _layout(shapes, COPY_ALIGN)
    out["copy"] = _view(copies[0], 0, (ctotal,))
    for o, s in zip(coffs, shapes):
        if numel(s) % COPY_ALIGN:
            out["copy"][o + numel(s): o - (-numel(s) // COPY_ALIGN) * COPY_ALIGN] = 0
    if case["grads"] == "bf16":
        for w, g in zip(copies, grads[0]):
            w.grad = g
    return state


def _run_step(state):
    params, opt = state["params"], state["opt"]
    if state["case"]["grads"] == "accumulate":
        opt.zero_grad()
        for k, micro in enumerate(state["grads"]):
            for w, g in zip(state["copies"], micro):
                w.grad = g  # as backward leaves it
            ta.optimizer.working.accumulate_grads_(params, last=k + 1 == len(state["grads"]))
    norm = ta.clip_grad_norm(params, None, MAX_NORM)
    opt.step()
    return {"norm": norm, **state["out"]}


def _exact_step(case, seed):
    device = torch.device("cuda")
    shapes = _shapes(case)
    offs, _ = _layout(shapes, ALIGN)
    flat = _step_inputs(case, seed, device)
    views = [(o, o + numel(s), s) for o, s in zip(offs, shapes)]

    def grad(a, b):
        return sum(f[a:b].double() for f in flat["grads"])

    norm = torch.zeros((), dtype=torch.float64, device=device)
    for a, b, _ in views:
        norm += grad(a, b).square().sum()
    norm = norm.sqrt()
    coef = torch.clamp(MAX_NORM / (norm + 1e-6), max=1.0)
    step = STEPS_DONE + 1
    bias1, bias2 = 1.0 - BETAS[0] ** step, 1.0 - BETAS[1] ** step
    out = {k: flat.pop(k).double() for k in ("master", "exp_avg", "exp_avg_sq")}
    for a, b, s in views:
        g = grad(a, b) * coef
        p, m, v = (out[k][a:b] for k in ("master", "exp_avg", "exp_avg_sq"))
        if len(s) >= 2:
            p.mul_(1.0 - LR * WEIGHT_DECAY)
        m.mul_(BETAS[0]).add_(g, alpha=1.0 - BETAS[0])
        v.mul_(BETAS[1]).add_(g.square_(), alpha=1.0 - BETAS[1])
        del g
        p.sub_((LR / bias1) * m / (v.sqrt().div_(math.sqrt(bias2)).add_(EPS)))
    del flat
    if case["grads"] != "fp32":
        coffs, ctotal = _layout(shapes, COPY_ALIGN)
        copy = torch.zeros(ctotal, dtype=torch.float64, device=device)
        for (a, b, _), o in zip(views, coffs):
            copy[o: o + b - a] = out["master"][a:b]
        out["copy"] = copy
    out["step"] = torch.full((len(shapes),), step, dtype=torch.float64, device=device)
    return {"norm": norm, **out}


# ---------------------------------------------------------------------------- fused linear + CE


IGNORE = -100


def _ce_inputs(case, seed, device):
    """Hidden states of about unit size (a final norm's output), a head at its usual spread, labels
    of which one in twenty is padding."""
    g = torch.Generator(device=device).manual_seed(seed)
    n, d, v = case["rows"], case["dim"], case["vocab"]
    hidden = torch.empty(n, d, device=device).normal_(0.0, 1.0, generator=g)
    if case["hidden"] == "bf16":
        hidden = hidden.to(torch.bfloat16)
    weight = torch.empty(v, d, device=device).normal_(0.0, 0.02, generator=g)
    labels = torch.randint(0, v, (n,), device=device, generator=g)
    labels[torch.rand(n, device=device, generator=g) < 0.05] = IGNORE
    labels[0] = 0  # at least one row counts
    return hidden, weight, labels


def _prepare_ce(case, seed):
    hidden, weight, labels = _ce_inputs(case, seed, torch.device("cuda"))
    weight = torch.nn.Parameter(weight)
    if case["copy"]:
        ta.attach_bf16_working_params([weight])
    return {"case": case, "hidden": hidden.requires_grad_(case["grad"]), "weight": weight, "labels": labels}


def _run_ce(state):
    case, hidden, weight = state["case"], state["hidden"], state["weight"]
    amp = torch.autocast("cuda", dtype=torch.bfloat16) if case["hidden"] == "autocast" else contextlib.nullcontext()
    if not case["grad"]:
        with torch.no_grad(), amp:
            return {"loss": fused_linear_cross_entropy(hidden, weight, state["labels"], IGNORE, case["chunk"])}
    hidden.grad = weight.grad = None
    with amp:
        loss = fused_linear_cross_entropy(hidden, weight, state["labels"], IGNORE, case["chunk"])
    loss.backward()
    return {"loss": loss.detach(), "grad_hidden": hidden.grad, "grad_weight": weight.grad}


def _exact_ce(case, seed):
    hidden, weight, labels = _ce_inputs(case, seed, torch.device("cuda"))
    if case["hidden"] != "fp32":  # the products are defined on bf16 operands
        hidden, weight = hidden.to(torch.bfloat16), weight.to(torch.bfloat16)
    h, w = hidden.double(), weight.double()
    valid = labels != IGNORE
    n_valid = int(valid.sum())
    total = torch.zeros((), dtype=torch.float64, device=h.device)
    grad_h = torch.zeros_like(h)
    grad_w = torch.zeros_like(w)
    block = 1024
    for s in range(0, case["rows"], block):
        x = h[s: s + block] @ w.t()
        ok, lab = valid[s: s + block], labels[s: s + block].clamp_min(0)[:, None]
        lse = torch.logsumexp(x, dim=1)
        total += ((lse - x.gather(1, lab)[:, 0]) * ok).sum()
        if not case["grad"]:
            continue
        x.sub_(lse[:, None]).exp_()
        x.scatter_add_(1, lab, torch.full_like(lab, -1.0, dtype=torch.float64))
        x.mul_((ok / n_valid)[:, None])
        grad_h[s: s + block] = x @ w
        grad_w += x.t() @ h[s: s + block]
    if not case["grad"]:
        return {"loss": total / n_valid}
    return {"loss": total / n_valid, "grad_hidden": grad_h, "grad_weight": grad_w}


# ---------------------------------------------------------------------------- the interface


def prepare(case, seed):
    return _prepare_step(case, seed) if case["family"] == "step" else _prepare_ce(case, seed)


def run(state):
    return _run_step(state) if state["case"]["family"] == "step" else _run_ce(state)


def exact(case, seed):
    return _exact_step(case, seed) if case["family"] == "step" else _exact_ce(case, seed)


def work(case):
    if case["family"] == "step":
        n = sum(numel(s) for s in _shapes(case))
        # grads in; master and both moments in and out; the bf16 copy out
        per = {"bf16": 2 + 24 + 2, "fp32": 4 + 24, "accumulate": 2 * 2 + 24 + 2}[case["grads"]]
        return {"bytes": n * per, "flops": 15 * n}
    n, d, v = case["rows"], case["dim"], case["vocab"]
    h_bytes = 2 if case["hidden"] == "bf16" else 4
    w_bytes = 2 if case["copy"] else 4
    read = n * d * h_bytes + v * d * w_bytes + 8 * n
    written = n * d * h_bytes + v * d * 4 if case["grad"] else 4
    return {"bytes": read + written, "flops": (6 if case["grad"] else 2) * n * d * v}


def tolerance(case):
    if case["family"] == "step":
        # fp32 state (a sum of squares in another order moves the clip by an ulp); an element of
        # the bf16 copy next to a tie may round the other way, one step of 2^-8
        return {"rel": 1e-6, "max": 1e-2} if case["grads"] != "fp32" else {"rel": 1e-6, "max": 1e-5}
    if case["hidden"] == "fp32":
        return {"rel": 1e-5, "max": 1e-3}
    # bf16 logits, softmax gradients and products; the loss alone is a mean over fp32 row losses
    return {"rel": 1e-2, "max": 0.1} if case["grad"] else {"rel": 1e-4}
