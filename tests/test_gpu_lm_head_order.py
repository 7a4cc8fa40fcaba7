"""The fused lm_head kernel's orders of work: up to 8, up to 16 and more token
tiles, one and two vocabulary tiles per workgroup, with and without a partial
vocabulary tile, and batches whose last workgroups have no tile, against an
fp64 evaluation.  K = 128 keeps the products small."""

import pytest
import torch

from graspo_amd import ops

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


# 1, 3, 8, 9, 13, 16 and 17 token tiles; 12800 = 50 and 12801 = 50 and one
# row of vocabulary tiles, 255 one partial tile alone, 65536 many rounds
@pytest.mark.parametrize("N", [1, 700, 2048, 2049, 3300, 4096, 4097])
@pytest.mark.parametrize("V", [255, 12800, 12801, 65536])
def test_every_tile_is_computed_once(N, V):
    g = torch.Generator(device=DEV).manual_seed(N + V)
    h = torch.randn(N, 128, generator=g, device=DEV).bfloat16()
    w = (torch.randn(V, 128, generator=g, device=DEV) * 0.2).bfloat16()
    t = torch.randint(0, V, (N,), generator=g, device=DEV)
    print("lm_head order", N, V, flush=True)
    lp, H, lse = ops.lm_head_logprob(h, w, t)
    lp2, lse2, logits, st = ops.lm_head_logprob_save(h, w, t)
    assert int(st.abs().sum()) == 0
    assert torch.equal(lse, lse2) and torch.equal(lp, lp2)
    for s in range(0, N, 1024):
        x = h[s : s + 1024].double() @ w.double().t()
        ref = x.logsumexp(1)
        # fp32 sums of V terms, exponents below 64 rounded once
        assert float((lse[s : s + 1024] - ref).abs().max()) <= 2e-5
        want = x.gather(1, t[s : s + 1024, None]).squeeze(1) - ref
        assert float((lp[s : s + 1024] - want).abs().max()) <= 2e-5
        p = (x - ref[:, None]).exp()
        ent = ref - (p * x).sum(1)
        assert float((H[s : s + 1024] - ent).abs().max()) <= 5e-5
        # products of 128 bf16 pairs summed in fp32
        assert float((logits.t()[s : s + 1024] - x).abs().max()) <= 2e-5
