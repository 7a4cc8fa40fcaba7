"""The greedy kernel against the oracle, bit for bit: slice counts (one
workgroup per row and split rows), vocabularies around the slices' edges,
unaligned rows, masks, penalties, ties across slices, and rows of non-finite
or no allowed values."""

import ctypes

import numpy as np
import pytest
import torch

from tests import _capi
from tests._util import oracle_sample

DEV = torch.device("cuda:0")
INTS = ("ids", "kept", "thresh_id", "status")


def _mask(B, V, g, density):
    W = (V + 31) // 32
    bits = torch.rand(B, W * 32, generator=g) < density
    bits[:, V:] = False
    w = (bits.view(B, W, 32).long() << torch.arange(32)).sum(-1)
    return torch.where(w >= 2**31, w - 2**32, w).to(torch.int32)


def _check(x, workspace=True, **kw):
    L = _capi.lib()
    ref = oracle_sample(x, temperature=0.0, **kw)
    gk = {k: (v.to(DEV) if isinstance(v, torch.Tensor) else v) for k, v in kw.items()}
    st = x.stride(0)
    buf = torch.empty(x.storage_offset() + x.shape[0] * st + 8, dtype=x.dtype, device=DEV)
    xd = buf.as_strided(x.shape, (st, 1), x.storage_offset())
    xd.copy_(x)
    args, p, B = _capi.sample_args(xd, temperature=0.0, **gk)
    n = L.gtp_sample_workspace_bytes(_capi.DTYPE[x.dtype], B, x.shape[1], ctypes.byref(p))
    ws = torch.zeros(max(n, 256) if workspace else 0, dtype=torch.uint8, device=DEV)
    for _ in range(2):  # the second call finds the counters that the first one left
        out = _capi.SampleBuffers(B, DEV)
        assert L.gtp_sample_rows(*args, *out.out_args(), ws.data_ptr() if workspace else None,
                                 ws.numel(), _capi.stream_handle()) == 0
        torch.cuda.synchronize()
        got = out.cpu()
        for f in INTS:
            assert np.array_equal(got[f].numpy(), getattr(ref, f)), f
        assert np.array_equal(got["thresh_value"].numpy().view(np.int32)[ref.status == 0],
                              ref.thresh_value.view(np.int32)[ref.status == 0])
        # fp32 sums of up to 2^18 terms (a few 1e-6 relative), a logarithm and a
        # difference below 32 (2e-6 each); the exponents' rounding, 1e-6 a term
        a, b = got["logprob"].numpy(), ref.logprob
        assert np.array_equal(np.isnan(a), np.isnan(b))
        fin = np.isfinite(b)
        assert np.abs(a[fin] - b[fin]).max(initial=0) <= 2e-5


@pytest.mark.gpu
@pytest.mark.parametrize("B,V", [(1, 512), (3, 4103), (1, 151936), (70, 32775), (2, 262144),
                                 (257, 2055)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("extra", ["plain", "pen", "mask", "pen_mask"])
def test_greedy_matches_oracle(B, V, dtype, extra):
    print(B, V, dtype, extra, flush=True)
    g = torch.Generator().manual_seed(B * 1000 + V)
    # coarse values: exact ties of the maximum within and across slices
    x = (torch.randn(B, V + 1, generator=g) * 4).round().div(2).to(dtype)
    x = x[:, 1:] if V % 2 else x[:, :V]  # rows at odd elements
    kw = {}
    if "pen" in extra:
        kw.update(repetition_penalty=1.3 if V % 3 else 0.7,
                  history=torch.randint(-1, V, (B, 300), generator=g, dtype=torch.int32))
    if "mask" in extra:
        kw["allow_mask"] = _mask(B, V, g, 0.02)
    _check(x, **kw)


@pytest.mark.gpu
@pytest.mark.parametrize("workspace", [True, False])
@pytest.mark.parametrize("V", [513, 40003])
def test_greedy_special_rows(workspace, V):
    g = torch.Generator().manual_seed(V)
    x = torch.randn(10, V, generator=g)
    x[0, V - 1] = float("nan")
    x[1, 7] = float("inf")
    x[2] = float("-inf")
    x[3, :] = float("-inf")
    x[3, V - 2] = -3.0
    x[4] = 0.0
    x[4, ::3] = -0.0  # the two zeros tie
    x[5, 400] = float("nan")
    x[6, 11] = 3e38   # overflows under the penalty
    h = torch.full((10, 4), -1, dtype=torch.int32)
    h[6, 0] = 11
    h[7, 3] = V       # a history id beyond the vocabulary
    for rho in (1.0, 0.5):
        _check(x, workspace=workspace, history=h, repetition_penalty=rho)
    m = torch.full((10, (V + 31) // 32), -1, dtype=torch.int32)
    m[8] = 0          # nothing allowed
    m[5, 400 // 32] = 0  # the NaN is not allowed
    _check(x, workspace=workspace, history=h, repetition_penalty=0.5, allow_mask=m)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,V", [(1, 151936), (3, 50256), (2, 8192), (8, 248320)])
def test_nearly_one_hot_rows(dtype, B, V):
    """logprob = -ln(1 + r) of a small r: within the sum's rounding of 1, the
    same bits on every call, and in 16-bit types the split kernel's (top-k 1)
    where its slices lie within its pilot."""
    g = torch.Generator().manual_seed(V)
    x = torch.randn(B, V, generator=g).to(dtype)
    x[torch.arange(B), torch.randint(0, V, (B,), generator=g)] = 24.0
    got, route = _capi.sample_rows(x.to(DEV), temperature=0.0)
    assert route == _capi.ROUTE_SPLIT_TOPK
    ref = x.double().log_softmax(-1).max(-1).values
    # sums near 1, each rounded by at most 2^-24: up to 32 small terms beside
    # the largest in its thread, then 6 + 4 + 3 steps over a wave, the waves
    # and the slices; the logarithm of the result adds one more
    assert float((got["logprob"] - ref).abs().max()) <= 46 * 2.0 ** -24
    again, _ = _capi.sample_rows(x.to(DEV), temperature=0.0)
    assert torch.equal(got["logprob"], again["logprob"])
    if dtype != torch.float32 and V <= 151936:
        u = torch.full((B,), 0.25, device=DEV)
        split, _ = _capi.sample_rows(x.to(DEV), temperature=1.0, top_k=1, uniforms=u)
        for f in ("ids", "logprob", "status"):
            assert torch.equal(got[f], split[f]), f


@pytest.mark.gpu
@pytest.mark.parametrize("B", [0, 1, 3, 5])
@pytest.mark.parametrize("inference", [False, True])
def test_outputs_are_tensors_of_their_own(B, inference):
    """Each of the seven outputs is contiguous, keeps its dtype, and writing
    one in place leaves the others."""
    from graspo_amd import ops

    x = torch.randn(B, 4096, device=DEV)
    with torch.inference_mode(inference):
        out = ops.sample(x, temperature=0.0)
        assert [t.dtype for t in out] == [torch.int64, torch.float32, torch.float32, torch.int32,
                                          torch.float32, torch.int32, torch.int32]
        before = [t.clone() for t in out]
        assert torch.equal(out.ids, x.argmax(1)) and torch.equal(out.thresh_id, out.ids.int())
        for i, t in enumerate(out):
            assert t.shape == (B,) and t.is_contiguous() and t.is_inference() == inference
            v = t._version if not inference else 0
            t.fill_(77)
            assert inference or t._version == v + 1
            for j, o in enumerate(out):
                if j > i:
                    assert torch.equal(o, before[j])
    assert not any(t.requires_grad for t in out)


@pytest.mark.gpu
@pytest.mark.parametrize("kw", [dict(temperature=0.0), dict(temperature=0.8, top_k=20),
                                dict(temperature=1.0, top_p=0.9)])
def test_outputs_have_storages_of_their_own(kw):
    """They can be saved together and resized, and each is freed on its own."""
    import io

    from graspo_amd import ops

    out = ops.sample(torch.randn(3, 4096, device=DEV), **kw)
    assert len({t.untyped_storage().data_ptr() for t in out}) == 7
    for t in out:
        assert t.storage_offset() == 0
        assert t.untyped_storage().nbytes() == t.numel() * t.element_size()
    f = io.BytesIO()
    torch.save(tuple(out), f)
    f.seek(0)
    for a, b in zip(torch.load(f, weights_only=True), out):
        assert torch.equal(a.cpu(), b.cpu())
    before = [t.clone() for t in out]
    out.ids.resize_(64).fill_(-1)
    out.kept.resize_(64).fill_(-1)
    for t, b in list(zip(out, before))[1:3] + list(zip(out, before))[4:]:
        assert torch.equal(t, b)
    with torch.cuda.device(DEV):
        side = torch.cuda.Stream()
        out.logprob.record_stream(side)
