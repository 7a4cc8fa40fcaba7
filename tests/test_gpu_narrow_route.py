"""Which fp32 rows the drop-in samples from a bf16 copy, and that either way
gives the same tokens; the copy's exactness flag."""

import pytest
import torch

from graspo_amd import ops
from graspo_amd import tensor_utils as TU

DEV = torch.device("cuda:0")


# 13e6 and, for strided rows, 24e6 logits; vocabularies from 65536 on, in
# whole 16-byte vectors of bf16
@pytest.mark.gpu
@pytest.mark.parametrize("B,V,strided,top_p,narrow", [
    (198, 65536, False, 1.0, False), (199, 65536, False, 1.0, True),
    (199, 65536, False, 0.9, False), (199, 65540, False, 1.0, False),
    (407, 32000, False, 1.0, False), (365, 65536, True, 1.0, False),
    (367, 65536, True, 1.0, True), (2, 65536, False, 1.0, False)])
def test_route_and_tokens(B, V, strided, top_p, narrow):
    g = torch.Generator(device=DEV).manual_seed(B)
    wide = torch.randn(B, V + 8, generator=g, device=DEV).mul_(2.5).bfloat16().float()
    x = wide[:, :V] if strided else wide[:, :V].contiguous()
    u = torch.randint(0, 1 << 24, (B,), generator=g, device=DEV).float() * 2.0 ** -24
    print(B, V, strided, top_p, flush=True)
    took = TU._bf16_when_exact(x, 1.0, 0, top_p)
    assert (took.dtype == torch.bfloat16) == narrow
    assert torch.equal(took.float(), x)
    ids = TU._next_token_from_logits(x, temperature=1.0, top_p=top_p, uniforms=u)
    assert torch.equal(ids, ops.sample(x, temperature=1.0, top_p=top_p, uniforms=u).ids)
    x[B - 1, V - 1] += 2.0 ** -12  # no longer a bf16 value
    assert TU._bf16_when_exact(x, 1.0, 0, top_p).dtype == torch.float32
    ids = TU._next_token_from_logits(x, temperature=1.0, top_p=top_p, uniforms=u)
    assert torch.equal(ids, ops.sample(x, temperature=1.0, top_p=top_p, uniforms=u).ids)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 4, 1023, 1024, 1025, 8192 * 1024 + 5])
@pytest.mark.parametrize("at", ["none", "first", "last", "all"])
def test_exactness_flag(n, at):
    x = torch.randn(n, device=DEV).bfloat16().float()
    if at != "none":
        i = {"first": slice(0, 1), "last": slice(n - 1, n), "all": slice(None)}[at]
        x[i] = (x[i].view(torch.int32) | 1).view(torch.float32)
    copy, inexact = ops.to_bf16_exact(x)
    assert bool(inexact) == (at != "none")
    assert torch.equal(copy.view(torch.int16), (x.view(torch.int32) >> 16).short())
