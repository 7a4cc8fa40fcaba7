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


# one chunk, exactly one and just more; ten; odd rows at every alignment; two
# steps per chunk (600001 fp32 tokens are 74 steps)
@pytest.mark.parametrize("V,N", [(7, 2100), (16384, 2100), (16392, 2100), (50257, 2100),
                                 (151936, 2100), (600001, 2060)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_token_logprob(V, N, dtype):
    g = torch.Generator(device=DEV).manual_seed(V)
    x = torch.empty(N, V, dtype=dtype, device=DEV)
    for s in range(0, N, 256):
        x[s : s + 256] = torch.randn(x[s : s + 256].shape, generator=g, device=DEV) * 3
    x[::5, V // 2 :] = -float("inf")
    t = torch.randint(0, V, (N,), generator=g, device=DEV)
    print("token_logprob", V, dtype, flush=True)
    whole = ops.token_logprob(x, t, entropy=True)
    lp, H, _ = ops.logprob_entropy(x, t)
    assert torch.equal(lp, whole.logprob) and torch.equal(H, whole.entropy)
    for n in (1, 3, 61, 300, 1500):
        for s in (0, N - n):
            part = ops.token_logprob(x[s : s + n], t[s : s + n], entropy=True)
            assert torch.equal(part.logprob, whole.logprob[s : s + n]), (n, s)
            assert torch.equal(part.entropy, whole.entropy[s : s + n]), (n, s)
            alone = ops.token_logprob(x[s : s + n], t[s : s + n])
            assert torch.equal(alone.logprob, whole.logprob[s : s + n]), (n, s)
