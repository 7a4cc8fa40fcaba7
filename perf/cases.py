"""The work that a user of this framework has it do, as measurable cases.

A GRASPO step goes three ways through the framework: the rollout samples one
token per row and decode step (``ops.sample``), the scoring passes turn logits
or hidden states into per-token logprobs, and the training passes run the loss
on those logprobs and their backward.  ``listed()`` holds each of them over
its range of sizes, ``draw()`` gives more of the same ranges.

A case is a dict of plain values.  ``kind`` says which entry point it calls:

- ``sample``: ``ops.sample`` over [rows, vocab] logits, as a decode loop does.
- ``score``: ``sequence_log_probs_and_entropy_from_logits`` (no gradient).
- ``policy``: ``sequence_log_probs_from_logits``, ``GRASPOLoss`` and the
  gradient of the logits.
- ``sft``: ``sft_cross_entropy_loss`` and the gradient of the logits.
- ``hidden``: ``_selected_token_log_probs_from_hidden`` over hidden states and
  the lm_head weight (no gradient).
- ``hidden_policy``: the same with ``GRASPOLoss`` and the gradients of the
  hidden states and the weight.
"""

from __future__ import annotations

import math

import torch

from graspo_amd import ops
from graspo_amd.graspo_loss import (
    GRASPOLoss,
    sequence_log_probs_and_entropy_from_logits,
    sequence_log_probs_from_logits,
)
from graspo_amd.sft_loss import sft_cross_entropy_loss
from graspo_amd.tensor_utils import _selected_token_log_probs_from_hidden

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
CLIP = 0.2
SLAB = 512  # rows made at a time, to bound the fp32 temporaries


def _sample(name, rows, vocab, dtype, temperature, top_k=0, top_p=1.0, penalty=1.0, history=0,
            mask=False):
    return dict(name=name, kind="sample", rows=rows, vocab=vocab, dtype=dtype,
                temperature=temperature, top_k=top_k, top_p=top_p, penalty=penalty,
                history=history, mask=mask)


def listed():
    return [
        # a single interactive request decoded greedily: the smallest call
        _sample("greedy_one_row", 1, 151936, "bf16", 0.0),
        # one prompt's group in the reference's own loop, which hands the
        # sampler `logits.float()` with a temperature and a top-p
        _sample("fp32_group_top_p", 8, 151936, "fp32", 0.7, top_p=0.9),
        # a rollout step of 8 prompts x group 8 with a repetition penalty
        _sample("group_rollout_penalty", 64, 151936, "bf16", 1.0, top_p=0.95, penalty=1.1,
                history=2048),
        # a rollout from the policy itself (temperature 1, nothing cut off),
        # as on-policy training samples it; a batch that fills no power of two
        _sample("plain_rollout", 96, 151936, "bf16", 1.0),
        # a large decode step over the large vocabulary
        _sample("large_decode_top_p", 256, 248320, "bf16", 0.7, top_p=0.9),
        # the same with everything on: structured output, penalty, top-k, top-p
        _sample("large_decode_masked_top_k", 256, 248320, "bf16", 0.7, top_k=64, top_p=0.9,
                penalty=1.05, history=4096, mask=True),
        # scoring one short completion
        dict(name="score_short", kind="score", batch=1, seq=61, vocab=151936, dtype="bf16"),
        # loss-side logprobs of one chunk of a rollout batch
        dict(name="score_chunk", kind="score", batch=4, seq=2048, vocab=151936, dtype="bf16"),
        # a small policy step on fp32 logits with an odd vocabulary, whose
        # rows start at every alignment
        dict(name="ragged_policy_step", kind="policy", batch=3, seq=333, vocab=50257,
             dtype="fp32"),
        # a supervised step with masked prompts
        dict(name="sft_step", kind="sft", batch=8, seq=512, vocab=151936, dtype="bf16"),
        # the production scoring pass: the fp32 copies of hidden states and
        # lm_head that the callers pass, 4 sequences of 2048 tokens
        dict(name="hidden_score", kind="hidden", batch=4, seq=2048, width=4096, vocab=248320,
             dtype="fp32"),
        # the production training pass on bf16 operands
        dict(name="hidden_policy_step", kind="hidden_policy", batch=2, seq=1024, width=4096,
             vocab=151936, dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _vocab(rng):
    v = _log_int(rng, 32000, 248320)
    # most lm_heads are padded to a multiple of 64; some vocabularies are odd
    return v if rng.random() < 0.3 else min(248320, (v + 63) // 64 * 64)


def draw(rng):
    kind = rng.choice(["sample", "sample", "sample", "score", "policy", "sft", "hidden",
                       "hidden_policy"])
    if kind == "sample":
        c = _sample("", _log_int(rng, 1, 256), _vocab(rng),
                    rng.choice(["bf16", "bf16", "bf16", "fp32", "fp16"]),
                    round(rng.uniform(0.6, 1.2), 2))
        del c["name"]
        how = rng.choice(["greedy", "plain", "top_p", "top_p", "top_k", "both"])
        if how == "greedy":
            c["temperature"] = 0.0
        if how in ("top_k", "both"):
            c["top_k"] = _log_int(rng, 5, 100)
        if how in ("top_p", "both"):
            c["top_p"] = round(rng.uniform(0.8, 0.98), 3)
        if rng.random() < 0.3:
            c["penalty"] = round(rng.uniform(1.02, 1.2), 3)
            c["history"] = _log_int(rng, 16, 4096)
        c["mask"] = rng.random() < 0.25
        return c
    v = _vocab(rng)
    if kind in ("hidden", "hidden_policy"):
        b = rng.choice([1, 2, 3, 4])
        s = _log_int(rng, 8, (8192 if kind == "hidden" else 2048) // b)
        if kind == "hidden_policy":
            v = min(v, 151936)
        return dict(kind=kind, batch=b, seq=s, width=128 * rng.randint(8, 32), vocab=v,
                    dtype=rng.choice(["fp32", "bf16"]))
    b = rng.choice([1, 2, 3, 4, 8])
    s = _log_int(rng, 9, (8192 if kind == "score" else 4096) // b)
    dtype = rng.choice(["bf16", "bf16", "fp32", "fp16"])
    if dtype == "fp32":
        s = max(9, s // 2)
    return dict(kind=kind, batch=b, seq=s, vocab=v, dtype=dtype)


# ------------------------------------------------------------------- inputs

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _logit_rows(n, V, dtype, g):
    """[n, V] logits ~ N(0, 2.5) with a few likely tokens per row (+4 to
    +10 on 16 of them), as a model's rows have."""
    x = torch.empty((n, V), dtype=DTYPES[dtype], device="cuda")
    for s in range(0, n, SLAB):
        k = min(SLAB, n - s)
        y = torch.randn((k, V), generator=g, device="cuda").mul_(2.5)
        at = torch.randint(0, V, (k, 16), generator=g, device="cuda")
        up = torch.rand((k, 16), generator=g, device="cuda") * 6.0 + 4.0
        y.scatter_(1, at, y.gather(1, at) + up)
        x[s : s + k] = y.to(x.dtype)
    return x


def _targets_of(x, g):
    """The row's largest logit for three of four rows (a policy mostly takes
    likely tokens), any token for the others."""
    t = torch.randint(0, x.shape[1], (x.shape[0],), generator=g, device="cuda")
    for s in range(0, x.shape[0], SLAB):
        top = x[s : s + SLAB].argmax(dim=1)
        pick = torch.rand(top.shape, generator=g, device="cuda") < 0.75
        t[s : s + SLAB] = torch.where(pick, top, t[s : s + SLAB])
    return t


def _mask_words(rows, V, g):
    """[rows, ceil(V/32)] int32 allow words: about 8% of the tokens and 300
    structural ones that every row allows."""
    W = (V + 31) // 32
    structural = torch.randperm(V, generator=g, device="cuda")[:300]
    weight = torch.ones(32, dtype=torch.int64, device="cuda") << torch.arange(32, device="cuda")
    words = torch.empty((rows, W), dtype=torch.int32, device="cuda")
    for s in range(0, rows, 64):
        k = min(64, rows - s)
        bits = torch.rand((k, W * 32), generator=g, device="cuda") < 0.08
        bits[:, structural] = True
        bits[:, V:] = False
        w = (bits.view(k, W, 32).to(torch.int64) * weight).sum(-1)
        words[s : s + k] = torch.where(w >= 2**31, w - 2**32, w).to(torch.int32)
    return words


def _policy_inputs(B, S, g, logp):
    """Old logprobs near ``logp``, one advantage per sequence, a mask with
    ragged ends."""
    old = logp + 0.15 * torch.randn((B, S), generator=g, device="cuda")
    adv = torch.randn((B, 1), generator=g, device="cuda")
    ends = torch.randint(max(1, S // 2), S + 1, (B, 1), generator=g, device="cuda")
    return old, adv, torch.arange(S, device="cuda").unsqueeze(0) < ends


def _rows_logprob(x, t):
    """fp32 logprobs to build old-policy logprobs from."""
    out = torch.empty(x.shape[0], dtype=torch.float32, device="cuda")
    for s in range(0, x.shape[0], SLAB):
        y = x[s : s + SLAB].float()
        out[s : s + SLAB] = y.gather(1, t[s : s + SLAB, None]).squeeze(1) - y.logsumexp(1)
    return out


def prepare(case, seed):
    g = _generator(seed)
    kind, V = case["kind"], case["vocab"]
    if kind == "sample":
        B = case["rows"]
        st = dict(logits=_logit_rows(B, V, case["dtype"], g), history=None, allow_mask=None)
        if case["history"]:
            st["history"] = torch.randint(0, V, (B, case["history"]), generator=g, device="cuda",
                                          dtype=torch.int32)
        if case["mask"]:
            st["allow_mask"] = _mask_words(B, V, g)
        # the sampler's uniforms lie on the 2^-24 grid of its own draws
        st["uniforms"] = torch.randint(0, 1 << 24, (B,), generator=g, device="cuda",
                                       dtype=torch.float32).mul_(2.0**-24)
        return dict(case=case, **st)
    B, S = case["batch"], case["seq"]
    n = B * S
    if kind in ("hidden", "hidden_policy"):
        H = case["width"]
        # normalised hidden states and a weight whose logits spread by about 2
        hid = torch.randn((n, H), generator=g, device="cuda").to(torch.bfloat16)
        w = torch.empty((V, H), dtype=torch.bfloat16, device="cuda")
        for s in range(0, V, 16384):
            w[s : s + 16384] = (torch.randn((min(16384, V - s), H), generator=g, device="cuda")
                                * (2.0 / math.sqrt(H))).to(torch.bfloat16)
        t = torch.randint(0, V, (n,), generator=g, device="cuda")
        # a token's hidden state leans to its own target's weight row
        hid = (hid.float() + w[t].float() * 2.0).to(torch.bfloat16)
        hid, w = hid.view(B, S, H).to(DTYPES[case["dtype"]]), w.to(DTYPES[case["dtype"]])
        st = dict(case=case, hidden=hid, weight=w, ids=t.view(B, S))
        if kind == "hidden_policy":
            hf = hid.reshape(n, H).float()
            # the spread of a row's normal logits gives its logsumexp closely
            logp = (hf * w[t].float()).sum(1) - math.log(V) - 2.0 / H * hf.pow(2).sum(1)
            st["old"], st["adv"], st["mask"] = _policy_inputs(B, S, g, logp.view(B, S))
            hid.requires_grad_(True)
            w.requires_grad_(True)
            st["loss"] = GRASPOLoss(CLIP)
        return st
    x = _logit_rows(n, V, case["dtype"], g)
    t = _targets_of(x, g)
    st = dict(case=case, logits=x.view(B, S, V))
    if kind == "sft":
        labels = t.view(B, S).clone()
        # labels[s + 1] is position s's target
        labels[:, 1:] = t.view(B, S)[:, :-1]
        prompt = torch.randint(1, max(2, S // 3), (B, 1), generator=g, device="cuda")
        labels[torch.arange(S, device="cuda").unsqueeze(0) < prompt] = -100
        st["labels"] = labels
        st["logits"].requires_grad_(True)
        return st
    st["ids"] = t.view(B, S)
    if kind == "policy":
        st["old"], st["adv"], st["mask"] = _policy_inputs(B, S, g, _rows_logprob(x, t).view(B, S))
        st["logits"].requires_grad_(True)
        st["loss"] = GRASPOLoss(CLIP)
    return st


# --------------------------------------------------------------------- runs

def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "sample":
        return tuple(ops.sample(
            state["logits"], temperature=c["temperature"], top_k=c["top_k"], top_p=c["top_p"],
            repetition_penalty=c["penalty"], history=state["history"],
            allow_mask=state["allow_mask"], uniforms=state["uniforms"]))
    if kind == "score":
        return sequence_log_probs_and_entropy_from_logits(state["logits"], state["ids"])
    if kind == "policy":
        lp = sequence_log_probs_from_logits(state["logits"], state["ids"])
        loss = state["loss"](lp, state["old"], state["adv"], state["mask"])
        (grad,) = torch.autograd.grad(loss, [state["logits"]])
        return lp.detach(), loss.detach(), grad
    if kind == "sft":
        loss = sft_cross_entropy_loss(state["logits"], state["labels"])
        (grad,) = torch.autograd.grad(loss, [state["logits"]])
        return loss.detach(), grad
    if kind == "hidden":
        with torch.no_grad():
            return _selected_token_log_probs_from_hidden(state["hidden"], state["weight"],
                                                         state["ids"])
    lp = _selected_token_log_probs_from_hidden(state["hidden"], state["weight"], state["ids"])
    loss = state["loss"](lp, state["old"], state["adv"], state["mask"])
    gh, gw = torch.autograd.grad(loss, [state["hidden"], state["weight"]])
    return lp.detach(), loss.detach(), gh, gw


# ------------------------------------------------------------ what it needs

def work(case):
    kind, V = case["kind"], case["vocab"]
    size = 4 if case["dtype"] == "fp32" else 2
    if kind == "sample":
        B = case["rows"]
        n = B * V
        # logits, history ids, mask words, one uniform; 7 outputs of a row
        b = n * size + B * (4 * case["history"] + 4 + 32)
        if case["mask"]:
            b += B * 4 * ((V + 31) // 32)
        return {"bytes": b, "flops": 2 * n}
    n = case["batch"] * case["seq"]
    if kind in ("hidden", "hidden_policy"):
        H = case["width"]
        b = (n * H + V * H) * size + n * 12
        f = 2 * n * H * V
        # with gradients: both operands' gradients written, two more products
        return {"bytes": 2 * b, "flops": 3 * f} if kind == "hidden_policy" else {"bytes": b,
                                                                                 "flops": f}
    b = n * V * size
    if kind == "score":
        return {"bytes": b + n * 16, "flops": 4 * n * V}
    # the logits read and their gradient written
    return {"bytes": 2 * b + n * 24, "flops": 8 * n * V}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        # ids, kept sizes and cuts are whole numbers that the sampler's
        # contract fixes; the logprobs are 32-bit sums (6e-8 off 64 bits)
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
    if kind in ("score", "hidden"):
        # 32-bit sums and products (1e-7 off 64 bits)
        return {"rel": 1e-6, "max": 1e-5}
    if kind == "hidden_policy":
        # the softmax part of the gradient goes through bf16 operands (1.7e-3
        # off 64 bits)
        return {"rel": 7e-3, "max": 1e-1}
    # a gradient rounded to the logits' type (3e-7, 2.1e-3 and 2.6e-4 off)
    return {"fp32": {"rel": 2e-6, "max": 1e-4}, "bf16": {"rel": 8e-3, "max": 1.6e-2},
            "fp16": {"rel": 1e-3, "max": 4e-3}}[case["dtype"]]


# ------------------------------------------------------------- in 64 bits

def _exact_row_sample(c, x, hist, words, u):
    """One row by the definition: penalty, mask and temperature as single
    fp32 operations, then softmax, cut and draw in 64 bits."""
    V = x.numel()
    xf = x.float()
    y = xf.clone()
    if hist is not None:
        at = hist[hist >= 0].long().unique()
        z = y[at]
        y[at] = torch.where(z < 0, z * c["penalty"], z / c["penalty"])
    if words is not None:
        bits = ((words.long() & 0xFFFFFFFF)[:, None] >> torch.arange(32, device="cuda")) & 1
        y = torch.where(bits.reshape(-1)[:V].bool(), y, float("-inf"))
    raw = xf.double()
    lse = raw.logsumexp(0)
    greedy = c["temperature"] <= 0
    if not greedy:
        y = y / torch.tensor(max(c["temperature"], 1e-6), dtype=torch.float32, device="cuda")
    top, order = y.sort(descending=True, stable=True)
    if greedy:
        return raw[order[0]] - lse, torch.zeros_like(lse), top[0].double()
    n = int((top > float("-inf")).sum())
    if 0 < c["top_k"] < n:
        n = c["top_k"]
    w = (top[:n].double() - top[0].double()).exp()
    cum = w.cumsum(0)
    if 0 < c["top_p"] < 1:
        p = torch.tensor(c["top_p"], dtype=torch.float32).double().item()
        n = int(((cum - w) <= p * cum[-1]).sum())
    total = cum[n - 1]
    r = min(n - 1, int((cum[:n] <= u.double() * total).sum()))
    return raw[order[r]] - lse, (w[r] / total).log(), top[n - 1].double()


def _exact_loss(lp, old, adv, mask):
    """GRASPOLoss and its gradient by the logprobs."""
    old, adv = old.double(), adv.double().expand_as(lp)
    lo, hi = (torch.tensor(v, dtype=torch.float32).double().item() for v in (1 - CLIP, 1 + CLIP))
    m = mask.double()
    inv = 1.0 / m.sum(1, keepdim=True).clamp_min(1)
    r = (lp - old).exp()
    a, b = r * adv, r.clamp(lo, hi) * adv
    loss = (-torch.minimum(a, b) * m * inv).sum(1).mean()
    inside = (r >= lo) & (r <= hi)
    d = torch.where((a < b) | inside, -a, torch.zeros_like(a)) * m * inv / lp.shape[0]
    return loss, d


def _exact_rows(x, t):
    """(logprob, entropy) of each row."""
    lp = torch.empty(x.shape[0], dtype=torch.float64, device="cuda")
    H = torch.empty_like(lp)
    for s in range(0, x.shape[0], SLAB):
        ls = x[s : s + SLAB].double().log_softmax(1)
        lp[s : s + SLAB] = ls.gather(1, t[s : s + SLAB, None]).squeeze(1)
        H[s : s + SLAB] = -(ls.exp() * ls).sum(1)
    return lp, H


def _exact_logit_grad(x, t, g):
    """g * (onehot - softmax), in 32 bits once computed in 64 (the rows would
    not fit otherwise)."""
    out = torch.empty(x.shape, dtype=torch.float32, device="cuda")
    for s in range(0, x.shape[0], SLAB):
        p = x[s : s + SLAB].double().softmax(1).neg_()
        p.scatter_add_(1, t[s : s + SLAB, None], torch.ones_like(p[:, :1]))
        out[s : s + SLAB] = p * g[s : s + SLAB, None]
    return out


def exact(case, seed):
    with torch.no_grad():
        return _exact(case, seed)


def _exact(case, seed):
    kind = case["kind"]
    st = prepare(case, seed)
    if kind == "sample":
        rows = [_exact_row_sample(
            case, st["logits"][b], None if st["history"] is None else st["history"][b],
            None if st["allow_mask"] is None else st["allow_mask"][b], st["uniforms"][b])
            for b in range(case["rows"])]
        lp, slp, cut = (torch.stack(v) for v in zip(*rows))
        return None, lp, slp, None, cut, None, None
    B, S, V = case["batch"], case["seq"], case["vocab"]
    if kind in ("score", "policy", "sft"):
        x = st["logits"].detach().view(B * S, V)
    if kind == "score":
        return tuple(v.view(B, S) for v in _exact_rows(x, st["ids"].view(-1)))
    if kind == "policy":
        t = st["ids"].view(-1)
        lp = _exact_rows(x, t)[0].view(B, S)
        loss, d = _exact_loss(lp, st["old"], st["adv"], st["mask"])
        return lp, loss, _exact_logit_grad(x, t, d.reshape(-1)).view(B, S, V)
    if kind == "sft":
        t = torch.full((B, S), -100, dtype=torch.int64, device="cuda")
        t[:, :-1] = st["labels"][:, 1:]
        valid = t.ne(-100)
        t = t.clamp_min(0).view(-1)
        n = valid.sum()
        lp = _exact_rows(x, t)[0].view(B, S)
        g = -valid.double() / n
        return ((lp * g).sum(), _exact_logit_grad(x, t, g.view(-1)).view(B, S, V))
    H = case["width"]
    h = st["hidden"].detach().reshape(-1, H).double()
    w, t = st["weight"].detach(), st["ids"].reshape(-1)
    parts, step = [], 8192
    for s in range(0, V, step):
        parts.append((h @ w[s : s + step].double().t()).logsumexp(1))
    lse = torch.stack(parts).logsumexp(0)
    lp = ((h * w[t].double()).sum(1) - lse)
    if kind == "hidden":
        return lp.view(B, S)
    loss, d = _exact_loss(lp.view(B, S), st["old"], st["adv"], st["mask"])
    d = d.reshape(-1, 1)
    gh = w[t].double() * d
    gw = torch.empty((V, H), dtype=torch.float32, device="cuda")
    for s in range(0, V, step):
        wc = w[s : s + step].double()
        p = ((h @ wc.t()) - lse[:, None]).exp().mul_(-d)
        gh += p @ wc
        at = ((t >= s) & (t < s + step)).nonzero().squeeze(1)
        c = p.t() @ h
        c.index_add_(0, t[at] - s, h[at] * d[at])
        gw[s : s + step] = c
    return lp.view(B, S), loss, gh.view(B, S, H), gw
