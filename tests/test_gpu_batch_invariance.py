"""A token's logprob, entropy and log-sum-exp are the same bits however many
tokens are scored with it: old and new logprobs of one policy, scored in
chunks of different sizes, have a ratio of exactly 1."""

import pytest
import torch

from graspo_amd import ops

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


# 75 full vocabulary tiles and a partial one, 76 without: one token tile takes
# one vocabulary tile per workgroup, 32 take two, on 256 CUs
@pytest.mark.parametrize("V", [19300, 19456, 300])
def test_lm_head(V):
    g = torch.Generator(device=DEV).manual_seed(V)
    N = 8192
    h = torch.randn(N, 128, generator=g, device=DEV).bfloat16()
    w = (torch.randn(V, 128, generator=g, device=DEV) * 0.2).bfloat16()
    t = torch.randint(0, V, (N,), generator=g, device=DEV)
    print("lm_head", V, flush=True)
    whole = ops.lm_head_logprob(h, w, t)
    lp, lse, _, _ = ops.lm_head_logprob_save(h, w, t)
    assert torch.equal(lp, whole[0]) and torch.equal(lse, whole[2])
    for n in (1, 200, 2048, 4000):
        for s in (0, N - n):
            part = ops.lm_head_logprob(h[s : s + n], w, t[s : s + n])
            for a, b in zip(part, whole):
                assert torch.equal(a, b[s : s + n]), (n, s)
            lp, lse, _, _ = ops.lm_head_logprob_save(h[s : s + n], w, t[s : s + n])
            assert torch.equal(lp, whole[0][s : s + n]) and torch.equal(lse, whole[2][s : s + n])
