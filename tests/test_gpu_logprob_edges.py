"""Rows of the logprob and gradient kernels that do not start or end on a
16-byte boundary: an odd vocabulary's contiguous rows at every alignment,
vocabularies below one vector, and gradients written at another alignment
than the logits'.  Compared with fp64 (torch, CPU)."""

import pytest
import torch

from graspo_amd import ops

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
# one rounding of the output type, plus the fp32 exponential: its argument
# (below 64 here) is rounded once, 64 * 2^-24, and v_exp_f32 adds an ulp
REL = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 5e-6}
# fp32 sums of V terms in 256 threads' partial sums, the same exponent error
LP_TOL = 2e-5


def _rows(n, V, dtype, offset, seed):
    """n contiguous rows of V that start `offset` elements into a buffer."""
    g = torch.Generator().manual_seed(seed)
    buf = torch.empty(offset + n * V + 16, dtype=dtype, device=DEV)
    x = buf[offset : offset + n * V].view(n, V)
    x.copy_((torch.randn(n, V, generator=g) * 3).to(dtype))
    t = torch.randint(0, V, (n,), generator=g)
    t[0], t[-1] = 0, V - 1  # targets in the first and the last elements
    return x, t


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [1, 3, 9, 31, 2049, 50257])
def test_every_alignment(dtype, V):
    for offset in (0, 1, 2, 5, 7):
        print("edges", dtype, V, offset, flush=True)
        x, t = _rows(9, V, dtype, offset, V + offset)
        lp, H, st = ops.logprob_entropy(x, t.to(DEV))
        ref = x.cpu().double().log_softmax(1)
        rlp = ref.gather(1, t[:, None]).squeeze(1)
        rH = -(ref.exp() * ref).sum(1)
        assert int(st.abs().sum()) == 0
        assert float((lp.cpu() - rlp).abs().max()) <= LP_TOL
        assert float((H.cpu() - rH).abs().max()) <= LP_TOL
        g = torch.linspace(-1.5, 2.0, 9)
        g[4] = 0.0  # zeros, not read
        lse = x.cpu().double().logsumexp(1).float()
        want = -g.double()[:, None] * (x.cpu().double() - lse.double()[:, None]).exp()
        want.scatter_add_(1, t[:, None], g.double()[:, None])
        for shift in (offset, offset + 1):  # the logits' own alignment, and another
            buf = torch.full((9 * V + 32,), 7.0, dtype=dtype, device=DEV)
            out = buf[shift : shift + 9 * V].view(9, V)
            ops.logprob_backward(x, t.to(DEV), g.to(DEV), lse.to(DEV), out=out)
            err = (out.cpu().double() - want).abs() - REL[dtype] * want.abs() - 2e-7
            assert float(err.max()) <= 0.0, (offset, shift, float(err.max()))
            rest = torch.cat([buf[:shift], buf[shift + 9 * V:]])
            assert bool((rest == 7.0).all())  # nothing written outside


@pytest.mark.parametrize("V", [3, 9, 2049])
def test_split_gradient_every_alignment(V):
    for offset in (0, 1, 2, 3):
        x, t = _rows(9, V, torch.float32, offset, V + offset)
        g = torch.linspace(-1.5, 2.0, 9)
        g[4] = 0.0
        lse = x.cpu().double().logsumexp(1).float()
        hi, lo = ops.logprob_backward_split(x, t.to(DEV), g.to(DEV), lse.to(DEV))
        want = ops.logprob_backward(x, t.to(DEV), g.to(DEV), lse.to(DEV)).double()
        got = hi.double() + lo.double()
        assert float(((got - want).abs() - 2.0 ** -16 * want.abs()).max()) <= 0.0
