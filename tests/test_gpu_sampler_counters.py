"""Calls of different row counts on one workspace: the arrival counters of
more than 4096 split rows (fp32 above 131072 tokens) reach into what is slot
data for a smaller call."""

import ctypes

import pytest
import torch

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
