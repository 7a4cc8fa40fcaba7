"""More rows than one grid dimension holds (2^24 workgroups of 256 threads),
and a launch error while the look at the targets is still queued."""

import ctypes

import pytest
import torch
import torch.nn.functional as F

from graspo_amd import ops
from graspo_amd.graspo_loss import sequence_log_probs_from_logits
from graspo_amd.sft_loss import sft_cross_entropy_loss

DEV = torch.device("cuda:0")
# one rounding of each of a few fp32 operations on values below 16
TOL = 4e-6


@pytest.mark.gpu
@pytest.mark.parametrize("B,S", [(3, 5592407), (1, (1 << 24) + 1)])
def test_rows_past_one_grid_dimension(B, S):
    """B sequences of S - 1 shifted rows, more than 2^24 in all in the first
    case's [B, S]; the gradient covers [B, S]."""
    V = 2
    g = torch.Generator(device=DEV).manual_seed(B)
    x = torch.randn(B, S, V, generator=g, device=DEV).requires_grad_(True)
    labels = torch.randint(0, V, (B, S), generator=g, device=DEV)
    print("sft", B, S, flush=True)
    loss = sft_cross_entropy_loss(x, labels)
    (grad,) = torch.autograd.grad(loss, [x])
    xd = x.detach().double()
    lp = xd[:, :-1].log_softmax(-1).gather(-1, labels[:, 1:, None]).squeeze(-1)
    # the mean of fp32 values, each within TOL
    assert abs(float(loss.detach()) + float(lp.mean())) <= TOL
    n = B * (S - 1)
    want = torch.zeros_like(xd)
    want[:, :-1] = (xd[:, :-1].softmax(-1) - F.one_hot(labels[:, 1:], V)) / n
    assert float((grad - want).abs().max()) <= 2e-6 / n
    print("rows", B, S, flush=True)
    view = x.detach()[:, : S - 1] if B > 1 else x.detach()
    t = labels[:, : view.shape[1]]
    got = sequence_log_probs_from_logits(view, t)
    ref = view.double().log_softmax(-1).gather(-1, t[..., None]).squeeze(-1)
    assert float((got - ref).abs().max()) <= TOL
    t = t.clone()
    t[-1, -1] = V
    with pytest.raises(RuntimeError, match="invalid rows"):
        sequence_log_probs_from_logits(view, t)


def _hip():
    for line in open("/proc/self/maps"):
        if "libamdhip64" in line:
            return ctypes.CDLL(line.split()[-1])
    raise RuntimeError("no HIP runtime in this process")


@pytest.mark.gpu
@pytest.mark.parametrize("entry", ["token_logprob", "verdict"])
def test_launch_error_waits_for_the_look_at_the_targets(entry):
    """Another library's HIP error makes the launch report one: the call
    raises only when the kernel that writes the pinned words has run."""
    a = torch.randn(8192, 8192, device=DEV).to(torch.bfloat16)
    x = torch.randn(64, 1000, device=DEV)
    t = torch.zeros(64, dtype=torch.int64, device=DEV)
    torch.mm(a, a)
    ops.token_logprob(x, t)
    ops.TargetsVerdict(t, 1000).wait()
    torch.cuda.synchronize()
    for _ in range(20):  # some 20 ms ahead of the look
        torch.mm(a, a)
    ahead = torch.cuda.Event()
    ahead.record()
    assert _hip().hipSetDevice(99) != 0
    with pytest.raises(RuntimeError, match="launch error"):
        if entry == "token_logprob":
            ops.token_logprob(x, t)
        else:
            ops.TargetsVerdict(t, 1000)
    assert ahead.query()
    out = ops.token_logprob(x, t)
    assert not out.bad_target
    assert float((out.logprob - x.log_softmax(-1)[:, 0]).abs().max()) <= 2e-5
