"""The token-logprob entry points (rows cut into slices, shifted rows read in
place, ignored targets, the mean and its gradient, the host's verdict on the
targets) against fp64 torch on the CPU."""

import ctypes

import pytest
import torch
import torch.nn.functional as F

import graspo_amd
from graspo_amd import ops
from graspo_amd.graspo_loss import sequence_log_probs_from_logits
from graspo_amd.sft_loss import sft_cross_entropy_loss

DEV = torch.device("cuda:0")
REL = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 5e-6}
# fp32 partial sums of V terms and one exponential's argument below 64
LP_TOL = 2e-5


def _ref(x, t):
    ls = x.cpu().double().log_softmax(-1)
    lp = ls.gather(-1, t.cpu().long().unsqueeze(-1)).squeeze(-1)
    p = ls.exp()
    return lp, -(p * ls.nan_to_num(neginf=0.0)).sum(-1)


# 16384 and 16392 bf16 tokens are one step of a slice's stream and one vector
# more; 151936 cuts into ten slices of one row; 300 rows into seven each
@pytest.mark.gpu
@pytest.mark.parametrize("N,V", [(1, 7), (1, 16384), (1, 16392), (3, 16391), (1, 248320),
                                 (61, 151936), (300, 50257), (2049, 16392)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_slices(N, V, dtype):
    g = torch.Generator().manual_seed(N + V)
    n = min(N, 64)  # rows checked
    x = (torch.randn(n, V, generator=g) * 3).to(dtype)
    x[:, 1::3] = -float("inf")  # whole slices' maxima and moments with them
    x[0, V // 2:] = -float("inf")
    xd = x.to(DEV).repeat((N + n - 1) // n, 1)[:N].contiguous()
    t = torch.randint(0, (V + 2) // 3, (n,), generator=g) * 3
    t[0] = 0
    td = t.to(DEV).repeat((N + n - 1) // n)[:N]
    print("slices", N, V, dtype, flush=True)
    out = ops.token_logprob(xd, td, entropy=True)
    rlp, rH = _ref(x, t)
    fin = torch.isfinite(rlp)
    assert not out.bad_target
    for k in range(0, N, n):
        lp, H = out.logprob[k : k + n].cpu(), out.entropy[k : k + n].cpu()
        m = lp.numel()
        assert bool((lp[~fin[:m]] == rlp[:m][~fin[:m]]).all())
        assert float((lp - rlp[:m])[fin[:m]].abs().max()) <= LP_TOL
        assert float((H - rH[:m]).abs().max()) <= LP_TOL
    # one workgroup per row agrees, and again gives the same bits
    lp1, H1, _ = ops.logprob_entropy(xd, td)
    assert float((lp1 - out.logprob)[torch.isfinite(lp1)].abs().max()) <= LP_TOL
    again = ops.token_logprob(xd, td, entropy=True)
    assert torch.equal(again.logprob, out.logprob) and torch.equal(again.entropy, out.entropy)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N", [2, 2100])
def test_entropy_where_the_first_infinities_come_late(N, dtype):
    """Blocks before, at and after the first one that holds a -inf, in rows of
    slices and of one workgroup: single logits, a tail and a whole step."""
    V = 70001
    g = torch.Generator().manual_seed(N)
    x = (torch.randn(8, V, generator=g) * 3).to(dtype)
    for r, at in enumerate((0, 1, 16384, 40000, V - 1)):
        x[r, at] = -float("inf")
    x[5, 33000:] = -float("inf")
    x[6, 20000:60000] = -float("inf")
    t = torch.full((8,), 7)
    n = (N + 7) // 8
    out = ops.token_logprob(x.to(DEV).repeat(n, 1)[:N], t.to(DEV).repeat(n)[:N], entropy=True)
    rlp, rH = _ref(x, t)
    for k in range(0, N, 8):
        m = min(8, N - k)
        assert float((out.logprob[k : k + m].cpu() - rlp[:m]).abs().max()) <= LP_TOL
        assert float((out.entropy[k : k + m].cpu() - rH[:m]).abs().max()) <= LP_TOL


@pytest.mark.gpu
def test_non_finite_rows_in_slices():
    V = 151936
    x = torch.zeros(4, V, dtype=torch.bfloat16)
    x[0, 140000] = float("nan")
    x[1, 3] = float("inf")
    x[2] = -float("inf")
    lp = ops.token_logprob(x.to(DEV), torch.tensor([5, 5, 5, 5], device=DEV), entropy=True)
    assert bool(lp.logprob[:3].isnan().all()) and bool(lp.entropy[:3].isnan().all())
    lp1, H1, _ = ops.logprob_entropy(x.to(DEV), torch.tensor([5, 5, 5, 5], device=DEV))
    assert torch.equal(lp1.isnan(), lp.logprob.isnan())
    assert float(lp1[3]) == pytest.approx(float(lp.logprob[3]), abs=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,S,V", [(1, 2, 9), (3, 17, 4099), (2, 40, 50257), (8, 300, 1000)])
def test_sft_shifted_rows(B, S, V, dtype):
    g = torch.Generator().manual_seed(S)
    x = (torch.randn(B, S, V, generator=g) * 3).to(dtype)
    labels = torch.randint(0, V, (B, S), generator=g)
    labels[0, : S // 2 + 1] = -100 if S > 2 else labels[0, : S // 2 + 1]
    xd = x.to(DEV).requires_grad_(True)
    loss = sft_cross_entropy_loss(xd, labels.to(DEV))
    (3.0 * loss).backward()
    xr = x.double().requires_grad_(True)
    ref = F.cross_entropy(xr[:, :-1].reshape(-1, V), labels[:, 1:].reshape(-1), ignore_index=-100)
    (3.0 * ref).backward()
    assert float(loss) == pytest.approx(float(ref), abs=LP_TOL)
    err = (xd.grad.cpu().double() - xr.grad).abs() - REL[dtype] * xr.grad.abs() - 2e-7
    assert float(err.max()) <= 0.0
    assert bool((xd.grad[:, -1] == 0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
def test_sft_labels_refilled_before_the_backward(dtype):
    g = torch.Generator().manual_seed(3)
    x = torch.randn(2, 9, 500, generator=g).to(DEV).requires_grad_(True)
    labels = torch.randint(0, 500, (2, 9), generator=g).to(DEV, dtype)
    (want,) = torch.autograd.grad(sft_cross_entropy_loss(x, labels), [x])
    loss = sft_cross_entropy_loss(x, labels)
    labels.fill_(-100)
    (got,) = torch.autograd.grad(loss, [x])
    assert torch.equal(got, want) and bool(want.any())


@pytest.mark.gpu
def test_sft_ignored_rows_of_any_value():
    """A NaN in an ignored row, or token 0 at -inf there, does not reach the
    loss or the gradient, as in F.cross_entropy."""
    g = torch.Generator().manual_seed(4)
    x = torch.randn(2, 7, 300, generator=g)
    labels = torch.randint(0, 300, (2, 7), generator=g)
    labels[0, 1:4] = -100  # the targets of positions 0..2
    x[0, 0, 17] = float("nan")
    x[0, 1, 0] = float("-inf")
    x[0, 2] = float("-inf")
    x[1, 6] = float("nan")  # the last position has no target
    xd = x.to(DEV).requires_grad_(True)
    loss = sft_cross_entropy_loss(xd, labels.to(DEV))
    (grad,) = torch.autograd.grad(loss, [xd])
    keep = labels[:, 1:].ne(-100)
    ls = x[:, :-1].double().log_softmax(-1)
    ref = F.nll_loss(ls[keep], labels[:, 1:][keep])
    assert float(loss.detach()) == pytest.approx(float(ref), abs=LP_TOL)
    assert bool((grad[:, :-1][~keep.to(DEV)] == 0).all()) and bool((grad[:, -1] == 0).all())
    assert bool(grad.isfinite().all())


@pytest.mark.gpu
def test_sft_one_position_and_no_targets():
    x = torch.randn(2, 1, 64, device=DEV, requires_grad=True)
    loss = sft_cross_entropy_loss(x, torch.zeros(2, 1, dtype=torch.int64, device=DEV))
    assert bool(loss.isnan())
    (grad,) = torch.autograd.grad(loss, [x])
    assert bool((grad == 0).all())
    x = torch.randn(2, 3, 64, device=DEV, requires_grad=True)
    loss = sft_cross_entropy_loss(x, torch.full((2, 3), -100, device=DEV))
    assert bool(loss.isnan())


@pytest.mark.gpu
@pytest.mark.parametrize("n,at", [(5, 4), (9000, 0), (9000, 8999), (70000, 69999)])
def test_bad_target_raises(n, at):
    """Every word of the verdict: one to three workgroups of targets and all 16."""
    x = torch.zeros(n, 8, device=DEV)
    t = torch.zeros(n, dtype=torch.int64, device=DEV)
    assert float(sequence_log_probs_from_logits(x, t)[at]) == pytest.approx(-2.0794415, abs=1e-5)
    for bad in (8, -1):
        t[at] = bad
        with pytest.raises(RuntimeError, match="invalid rows"):
            sequence_log_probs_from_logits(x, t)
    out = ops.token_logprob(x, t, ignore_index=-1)  # not bad when ignored
    assert not out.bad_target


@pytest.mark.gpu
def test_shifted_view_and_gradient():
    g = torch.Generator().manual_seed(5)
    x = torch.randn(3, 12, 4099, generator=g).to(torch.float16)
    t = torch.randint(0, 4099, (3, 12), generator=g)
    xd = x.to(DEV).requires_grad_(True)
    lp = sequence_log_probs_from_logits(xd[:, 1:], t.to(DEV)[:, 1:])
    w = torch.randn(3, 11, generator=g)
    (lp * w.to(DEV)).sum().backward()
    xr = x.double().requires_grad_(True)
    rlp = xr[:, 1:].log_softmax(-1).gather(-1, t[:, 1:].unsqueeze(-1)).squeeze(-1)
    (rlp * w.double()).sum().backward()
    assert float((lp.detach().cpu() - rlp.detach()).abs().max()) <= LP_TOL
    err = (xd.grad.cpu().double() - xr.grad).abs() - REL[torch.float16] * xr.grad.abs() - 1e-7
    assert float(err.max()) <= 0.0


def test_arguments_and_verdict_on_the_host():
    """Bad arguments are refused before any launch, and the wait reads the
    words it is given (no GPU)."""
    L = ctypes.CDLL(graspo_amd.LIB_PATH)
    vp, i64, i32 = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int

    class Rows(ctypes.Structure):
        _fields_ = [("logits", vp), ("targets", vp), ("B", i64), ("S", i64), ("V", i64),
                    ("batch_stride", i64), ("row_stride", i64), ("target_batch_stride", i64),
                    ("target_row_stride", i64), ("ignore_index", i64), ("dtype", i32),
                    ("targets_int64", i32), ("has_ignore", i32)]

    def rows(**kw):
        r = Rows(16, 16, 2, 3, 10, 30, 10, 3, 1, 0, 1, 1, 0)
        for k, v in kw.items():
            setattr(r, k, v)
        return ctypes.byref(r)

    fwd, bwd = L.gtp_token_logprob_rows, L.gtp_token_logprob_backward
    fwd.argtypes = [vp, vp, vp, vp, vp, vp, ctypes.c_size_t, vp]
    bwd.argtypes = [vp, i64, vp, vp, vp, vp, i64, i64, vp]
    for kw in (dict(V=0), dict(row_stride=9), dict(dtype=3), dict(B=-1), dict(logits=None),
               dict(targets=None), dict(batch_stride=-1), dict(target_row_stride=-1)):
        assert fwd(rows(**kw), 16, None, None, None, None, 0, None) == 1, kw
    assert fwd(rows(B=1 << 40), 16, None, None, None, None, 0, None) == 2
    assert fwd(rows(), None, None, None, None, None, 0, None) == 1
    assert fwd(rows(B=0), None, None, None, None, None, 0, None) == 0
    assert bwd(rows(), 4, 16, 16, None, 16, 30, 10, None) == 1  # more positions than rows
    assert bwd(rows(), 3, 16, 16, None, 16, 30, 9, None) == 1
    assert bwd(rows(), 3, 16, None, None, 16, 30, 10, None) == 1
    assert bwd(rows(B=0), 3, None, None, None, None, 30, 10, None) == 0
    L.gtp_verdict_wait.argtypes = [vp, ctypes.POINTER(i32), vp]
    words, bad = (ctypes.c_uint32 * 16)(*([1] * 16)), i32(9)
    assert L.gtp_verdict_wait(words, ctypes.byref(bad), None) == 0 and bad.value == 0
    words[11] = 2
    assert L.gtp_verdict_wait(words, ctypes.byref(bad), None) == 0 and bad.value == 1
    assert L.gtp_verdict_wait(None, ctypes.byref(bad), None) == 1
