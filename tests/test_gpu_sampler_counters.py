"""Calls of different row counts on one workspace: the arrival counters of
more than 4096 split rows (fp32 above 131072 tokens) reach into what is slot
data for a smaller call; a captured call keeps its workspace when the stream's
is outgrown."""

import ctypes

import pytest
import torch

from graspo_amd import ops
from tests import _capi

DEV = torch.device("cuda:0")


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["greedy", "greedy_unaligned", "top_k"])
def test_counters_beyond_the_fixed_region(how):
    L = _capi.lib()
    V, B = 131080, 4100
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(B, V + 4, generator=g, device=DEV)
    x = x[:, 1 : V + 1] if how == "greedy_unaligned" else x[:, :V]
    kw = dict(temperature=0.0) if how != "top_k" else dict(temperature=0.7, top_k=4)
    u = torch.rand(B, generator=g, device=DEV)
    p = _capi.SamplerParams(kw["temperature"], kw.get("top_k", 0), 1.0, 1.0)
    assert _capi.route(L, 0, B, V, T=kw["temperature"], k=kw.get("top_k", 0),
                       aligned=how != "greedy_unaligned") == (_capi.ROUTE_SPLIT_TOPK, 2)
    n = L.gtp_sample_workspace_bytes(0, B, V, ctypes.byref(p))
    ws = torch.zeros(n, dtype=torch.uint8, device=DEV)
    ref = x.argmax(1)
    first = None
    for rows in (B, 4096, B, 4099, B):
        print(how, rows, flush=True)
        args, _, _ = _capi.sample_args(x[:rows], uniforms=u, **kw)
        out = _capi.SampleBuffers(rows, DEV)
        assert L.gtp_sample_rows(*args, *out.out_args(), ws.data_ptr(), n,
                                 _capi.stream_handle()) == 0
        torch.cuda.synchronize()
        got = out.cpu()
        assert bool((got["status"] == 0).all())
        if how != "top_k":
            assert torch.equal(got["ids"], ref[:rows].cpu())
        first = first or got
        for f, v in got.items():
            if f == "logprob":  # the waves share out a slice as they go: the sum's order varies
                assert float((v - first[f][:rows]).abs().max()) <= 1e-5
            else:
                assert torch.equal(v, first[f][:rows]), f


@pytest.mark.gpu
@pytest.mark.parametrize("offset", [0, 1])
def test_captured_call_after_the_workspace_has_grown(offset):
    """Greedy rows, aligned and not: the workspace that a graph was captured
    with stays its own when a larger call on the stream has outgrown it."""
    V = 151936
    stream = torch.cuda.Stream()
    g = torch.Generator(device=DEV).manual_seed(2)
    x = torch.randn(1, V + 8, generator=g, device=DEV).bfloat16()[:, offset : offset + V]
    big = torch.randn(130, V + 8, generator=g, device=DEV).bfloat16()[:, offset : offset + V]
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        ops.sample(x, temperature=0.0)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        out = ops.sample(x, temperature=0.0)
    with torch.cuda.stream(stream):
        ids = ops.sample(big, temperature=0.0).ids
        mine = [torch.full((1 << 15,), 7, dtype=torch.uint8, device=DEV) for _ in range(64)]
    torch.cuda.synchronize()
    assert torch.equal(ids, big.argmax(1))
    for k in range(3):
        x.copy_(torch.randn(1, V, generator=g, device=DEV))
        graph.replay()
        torch.cuda.synchronize()
        assert int(out.ids) == int(x.argmax(1)), k
        assert all(bool((t == 7).all()) for t in mine)
