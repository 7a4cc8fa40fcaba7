"""The hidden-state path's backward on bf16 operands: weight gradients whose
target rows are summed apart in fp32 (targets shared by many tokens, both
sides of the rule that chooses it), odd token counts and vocabularies, and an
id outside the vocabulary found while the forward runs.  Against fp64."""

import pytest
import torch

from graspo_amd import ops
from graspo_amd import tensor_utils as TU

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


# 400 V = N^2 lies between 200 and 201 tokens at V = 100, and above every
# token count of the larger vocabularies
@pytest.mark.parametrize("N,V,H", [(200, 100, 128), (201, 100, 128), (1, 300, 128), (7, 2049, 256),
                                   (333, 5077, 256), (256, 4096, 384)])
@pytest.mark.parametrize("shared", [False, True])
def test_bf16_weight_gradient(N, V, H, shared):
    g = torch.Generator().manual_seed(N)
    h = (torch.randn(N, H, generator=g) * 0.5).bfloat16()
    w = (torch.randn(V, H, generator=g) * 0.3).bfloat16()
    t = torch.randint(0, V, (N,), generator=g)
    if shared:
        t = t % 3 * (V // 3)  # three targets for all tokens
    go = torch.randn(N, generator=g)
    go[N // 2] = 0.0
    hd, wd = h.to(DEV).requires_grad_(True), w.to(DEV).requires_grad_(True)
    print("hidden backward", N, V, H, shared, flush=True)
    lp = TU._selected_token_log_probs_from_hidden(hd.view(1, N, H), wd, t.to(DEV).view(1, N))
    gh, gw = torch.autograd.grad(lp, [hd, wd], go.to(DEV).view(1, N))
    hr, wr, gr = h.double(), w.double(), go.double()
    x = hr @ wr.t()
    p = (x - x.logsumexp(1, keepdim=True)).exp()
    onehot = torch.zeros_like(p).scatter_(1, t[:, None], 1.0)
    d = gr[:, None] * (onehot - p)
    for got, want, scale in ((gw, d.t() @ hr, (gr.abs()[:, None] * p).t() @ hr.abs()),
                             (gh, d @ wr, (gr.abs()[:, None] * p) @ wr.abs())):
        # each g p rounded to bf16 (2^-8), fp32 sums, one rounding of the result
        tol = 2.0 ** -8 * scale + 2.0 ** -8 * want.abs() + 1e-5
        assert float(((got.cpu().double() - want).abs() - tol).max()) <= 0.0


def test_bad_id_raises_while_the_forward_runs():
    h = torch.zeros(2, 40, 128, dtype=torch.bfloat16, device=DEV)
    w = torch.zeros(1000, 128, dtype=torch.bfloat16, device=DEV)
    t = torch.zeros(2, 40, dtype=torch.int64, device=DEV)
    for bad in (1000, -1):
        t[1, 39] = bad
        for hh, ww in ((h, w), (h.float(), w.float()), (h.half(), w.half())):
            with pytest.raises(RuntimeError, match="outside"):
                TU._selected_token_log_probs_from_hidden(hh, ww, t)
    t[1, 39] = 999
    assert bool(torch.isfinite(TU._selected_token_log_probs_from_hidden(h, w, t)).all())


def test_verdict_flags_and_targets():
    one, zero = (torch.full((1,), v, dtype=torch.int32, device=DEV) for v in (1, 0))
    t = torch.arange(5000, device=DEV)  # two workgroups of targets
    assert ops.TargetsVerdict(t, 5000).wait() == (False, False)
    assert ops.TargetsVerdict(t, 4999).wait() == (True, False)
    assert ops.TargetsVerdict(t, 5000, zero, one).wait() == (False, True)
    assert ops.TargetsVerdict(t[:0], 5000, one, zero).wait() == (False, True)
    assert ops.TargetsVerdict(t.view(2500, 2)[:, 0], 4999, zero).wait() == (False, False)
    assert ops.TargetsVerdict(t.int(), 10, zero, zero).wait() == (True, False)
