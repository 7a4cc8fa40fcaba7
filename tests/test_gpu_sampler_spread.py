"""The spread sampler (gtp_sample_rows_spread: three launches, every row over
several workgroups) against the exact oracle, bit for bit, over dtypes,
alignments, slice counts, penalties, masks, plain and top-p sampling, and rows
that it hands to the row-wise path.  The C entry point is called directly, so
that every case reaches these kernels whatever the torch op would choose; the
kernels that the op no longer takes on such batches are checked beside it."""

import ctypes

import numpy as np
import pytest
import torch

from tests import _capi
from tests._util import oracle_sample

DEV = torch.device("cuda:0")
INTS = ("ids", "kept", "thresh_id", "status")


def _lib():
    L = _capi.lib()
    L.gtp_sample_rows_spread.argtypes = L.gtp_sample_rows.argtypes
    L.gtp_sample_spread_workspace_bytes.argtypes = [ctypes.c_int64, ctypes.c_int64,
                                                    ctypes.POINTER(_capi.SamplerParams)]
    L.gtp_sample_spread_workspace_bytes.restype = ctypes.c_size_t
    return L


def _run(entry, ws_bytes, x, kw, fill):
    args, p, B = _capi.sample_args(x, **kw)
    n = ws_bytes(p, B)
    ws = torch.full((max(n, 256),), fill, dtype=torch.uint8, device=DEV)
    out = _capi.SampleBuffers(B, DEV)
    assert entry(*args, *out.out_args(), ws.data_ptr(), ws.numel(), _capi.stream_handle()) == 0
    torch.cuda.synchronize()
    return out.cpu()


def _check(what, x, general=True, **kw):
    """x on the CPU, any row stride; kw on the CPU."""
    print(what, flush=True)
    L = _lib()
    ref = oracle_sample(x, **kw)
    gk = {k: (v.to(DEV) if isinstance(v, torch.Tensor) else v) for k, v in kw.items()}
    st = x.stride(0)
    buf = torch.empty(x.storage_offset() + x.shape[0] * st + 8, dtype=x.dtype, device=DEV)
    xd = buf.as_strided(x.shape, (st, 1), x.storage_offset())
    xd.copy_(x)
    V = x.shape[1]
    calls = [("spread", L.gtp_sample_rows_spread,
              lambda p, B: L.gtp_sample_spread_workspace_bytes(B, V, ctypes.byref(p)), 0xA5)]
    if general:  # the kernel that gtp_sample_rows takes (its workspace starts at zero)
        calls.append(("general", L.gtp_sample_rows,
                      lambda p, B: L.gtp_sample_workspace_bytes(_capi.DTYPE[x.dtype], B, V,
                                                                ctypes.byref(p)), 0))
    for name, entry, bytes_of, fill in calls:
        got = _run(entry, bytes_of, xd, gk, fill)
        for f in INTS:
            assert np.array_equal(got[f].numpy(), getattr(ref, f)), (what, name, f)
        ok = ref.status == 0
        assert np.array_equal(got["thresh_value"].numpy()[ok].view(np.int32),
                              ref.thresh_value[ok].view(np.int32)), (what, name)
        # fp32 sums of up to 2^18 terms (a few 1e-6 relative), a logarithm and a
        # difference below 32 (2e-6 each); the exponents' rounding, 1e-6 a term
        for f in ("logprob", "sampled_logprob"):
            a, b = got[f].numpy()[ok], getattr(ref, f)[ok]
            fin = np.isfinite(b)
            assert np.array_equal(a[~fin], b[~fin], equal_nan=True), (what, name, f)
            assert np.abs(a[fin] - b[fin]).max(initial=0) <= 2e-5, (what, name, f)


def _u(B, g):
    return torch.randint(0, 1 << 24, (B,), generator=g).float() * 2.0 ** -24


def _mask(B, V, g, density):
    W = (V + 31) // 32
    bits = torch.rand(B, W * 32, generator=g) < density
    bits[:, V:] = False
    w = (bits.view(B, W, 32).long() << torch.arange(32)).sum(-1)
    return torch.where(w >= 2**31, w - 2**32, w).to(torch.int32)


pytest_gpu = pytest.mark.gpu


@pytest_gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("B,V,offset", [(1, 151936, 0), (3, 50257, 1), (9, 65541, 3), (40, 32000, 0),
                                        (2, 7, 0), (2, 33, 5), (5, 4103, 2), (300, 1000, 0)])
def test_dtypes_alignments_and_slices(dtype, B, V, offset):
    """16 slices down to one per row, slices that get nothing, vocabularies
    below one group of 8, rows at every alignment, tail tokens."""
    g = torch.Generator().manual_seed(B + V)
    buf = torch.zeros(offset + B * V + 8, dtype=dtype)
    x = buf.as_strided((B, V), (V, 1), offset)
    x.copy_((torch.randn(B, V, generator=g) * 3).to(dtype))
    hist = torch.randint(-1, V, (B, 70), generator=g, dtype=torch.int32)
    for kw in (dict(temperature=0.7, top_p=0.9), dict(temperature=1.0),
               dict(temperature=1.1, top_p=0.97, repetition_penalty=1.3, history=hist,
                    allow_mask=_mask(B, V, g, 0.4)),
               dict(temperature=0.5, repetition_penalty=0.8, history=hist),
               dict(temperature=0.9, top_p=0.3, allow_mask=_mask(B, V, g, 0.1))):
        _check(f"{dtype} [{B}, {V}] +{offset} {sorted(kw)}", x, general=False, uniforms=_u(B, g), **kw)


@pytest_gpu
@pytest.mark.parametrize("sigma", [0.02, 0.5, 1.5, 6.0])
def test_list_sizes_and_ties(sigma):
    """Few and many tokens in the bins of the cut and the draw, past the
    lists' capacity (the row-wise path) at the smallest spread, bf16 ties."""
    g = torch.Generator().manual_seed(7)
    for dtype in (torch.bfloat16, torch.float32):
        x = (torch.randn(4, 70000, generator=g) * sigma).to(dtype)
        for kw in (dict(temperature=1.0), dict(temperature=1.0, top_p=0.95),
                   dict(temperature=0.6, top_p=0.5)):
            for u in (0.0, 0.3, 0.999999):
                _check(f"sigma {sigma} {dtype} {kw} {u}", x,
                       uniforms=torch.full((4,), u), **kw)


@pytest_gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_handed_over(dtype):
    g = torch.Generator().manual_seed(3)
    B, V = 12, 66000
    x = (torch.randn(B, V, generator=g) * 2).to(dtype)
    x[0, 5] = float("nan")
    x[1, 65999] = float("inf")
    x[2] = -float("inf")
    x[3] = 1.25                       # one value: beyond every capacity
    x[4, 100:] = -float("inf")
    x[5] = 3e7
    x[6, 17] = 40.0                   # the rest has weight 0
    x[7, ::2] = 1.0                   # a bin with 33000 tokens
    x[8] = 0.0
    x[8, 3] = 20.0                    # weight spread below the maximum's bins
    u = _u(B, g)
    u[9] = 1.0
    fin = torch.zeros(B, dtype=torch.uint8)
    fin[10] = 1
    for kw in (dict(temperature=1.0), dict(temperature=0.8, top_p=0.9), dict(temperature=1e-7),
               dict(temperature=900.0, top_p=0.5)):
        _check(f"handed over {dtype} {kw}", x, uniforms=u, finished=fin, pad_token_id=9, **kw)
    hist = torch.randint(0, V, (B, 16), generator=g, dtype=torch.int32)
    hist[11, 3] = V
    mask = _mask(B, V, g, 0.5)
    mask[6] = 0
    for rho in (1.0, 1.5):
        _check(f"bad history, empty mask {dtype} {rho}", x, uniforms=u, temperature=0.9, top_p=0.9,
               repetition_penalty=rho, history=hist, allow_mask=mask)


@pytest_gpu
def test_repeated_calls_on_a_used_workspace_and_in_a_graph():
    """The torch op on fresh rows, and a captured call replayed between eager
    ones: the counters are cleared by the call itself."""
    from graspo_amd import ops

    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.empty(8, 151936, device=DEV)
    u = torch.empty(8, device=DEV)

    def fresh():
        x.copy_(torch.randn(x.shape, generator=g, device=DEV) * 2.5)
        u.copy_(ops.draw_uniforms(8, DEV, g))

    fresh()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ops.sample(x, temperature=0.7, top_p=0.9, uniforms=u)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.sample(x, temperature=0.7, top_p=0.9, uniforms=u)
    for _ in range(4):
        fresh()
        eager = ops.sample(x, temperature=0.7, top_p=0.9, uniforms=u)
        graph.replay()
        torch.cuda.synchronize()
        for f in ("ids", "kept", "thresh_id", "thresh_value", "status", "logprob"):
            assert torch.equal(getattr(out, f), getattr(eager, f)), f


@pytest_gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("B,V", [(4097, 40), (8200, 301)])
def test_passes_over_large_batches(dtype, B, V):
    """Two and three passes over one workspace, the last one shorter: every
    per-row argument and output moves along."""
    g = torch.Generator().manual_seed(B)
    x = (torch.randn(B, V + 3, generator=g) * 3).to(dtype)[:, 1 : V + 1]
    hist = torch.randint(-1, V, (B, 9), generator=g, dtype=torch.int32)
    hist[B - 1, 4] = V
    fin = (torch.rand(B, generator=g) < 0.1).to(torch.uint8)
    for kw in (dict(temperature=0.8), dict(temperature=0.7, top_p=0.9, repetition_penalty=1.2,
                                           history=hist, allow_mask=_mask(B, V, g, 0.6),
                                           finished=fin, pad_token_id=5)):
        _check(f"passes {dtype} [{B}, {V}] {sorted(kw)}", x, uniforms=_u(B, g), **kw)


def test_workspace_is_bounded():
    """The workspace depends on the rows of a pass and on V, not on the batch."""
    L = _lib()
    p = _capi.SamplerParams(0.7, 0, 0.9, 1.0)

    def size(B, V):
        return L.gtp_sample_spread_workspace_bytes(B, V, ctypes.byref(p))

    for V in (1, 64, 4096, 151936, 1 << 18):
        most = max(size(B, V) for B in (1, 32, 512, 4096, 4097, 8192, 65535))
        assert most <= 4096 * (16 * min(V, 4096) + 512 * 12 + 128) + 4096, V
    assert size(65535, 64) < 32 << 20 and size(65535, 151936) < 300 << 20


def test_spread_query_on_the_host():
    """Which calls the spread kernels take; arguments refused before launch."""
    L = _lib()
    P = _capi.SamplerParams

    def size(B, V, *p):
        return L.gtp_sample_spread_workspace_bytes(B, V, ctypes.byref(P(*p)))

    assert size(8, 151936, 0.7, 0, 0.9, 1.0) > 0
    assert size(8, 151936, 0.7, 151936, 1.0, 1.0) > 0  # top-k off
    assert size(8, 151936, 0.7, 50, 0.9, 1.0) == 0     # top-k
    assert size(8, 151936, 0.0, 0, 0.9, 1.0) == 0      # greedy
    assert size(8, 151936, 1025.0, 0, 0.9, 1.0) == 0
    assert size(0, 151936, 0.7, 0, 0.9, 1.0) == 0
    assert size(1 << 16, 151936, 0.7, 0, 0.9, 1.0) == 0
    assert size(8, (1 << 18) + 1, 0.7, 0, 0.9, 1.0) == 0

    def call(B=4, V=64, stride=64, T=0.7, k=0, rho=1.0, logits=16, ids=16, u=16, ws=16, n=1 << 30):
        p = P(T, k, 0.9, rho)
        return L.gtp_sample_rows_spread(logits, 1, B, V, stride, None, 0, 0, None, 0, u,
                                        ctypes.byref(p), None, 0, ids, None, None, None, None, None,
                                        None, ws, n, None)

    assert call(logits=None) == 1 and call(ids=None) == 1 and call(u=None) == 1
    assert call(stride=63) == 1 and call(rho=0.0) == 1 and call(ws=None) == 1 and call(n=64) == 1
    assert call(k=5) == 2 and call(T=0.0) == 2 and call(B=1 << 17) == 2
    assert call(B=0) == 0
