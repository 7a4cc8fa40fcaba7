"""GPU parity of the sampler kernel against the exact CPU oracle.

Ids, kept-set sizes, thresholds and statuses must be bit-exact; the two
logprob outputs within 1e-3 absolute.  Covers the four sampler workloads at
full size and the edge cases of the contract (statuses, ties, greedy,
dtypes, strided rows, odd V, the general path)."""

import numpy as np
import pytest
import torch

from graspo_amd import ops
from graspo_amd import workloads as W
from oracle import oracle as O
from tests import _capi
from tests._util import oracle_sample

pytestmark = pytest.mark.gpu
TOL = 1e-3


def _to(t, dev):
    return None if t is None else t.to(dev)


def gpu_sample(logits, route=None, **kw):
    """ops.sample's outputs on the CPU.  Where the op takes the spread kernels,
    the kernel that gtp_sample_rows takes for the same call runs too and must
    give the same bits (the logprobs within TOL).  ``route``: that kernel's."""
    dev = torch.device("cuda:0")
    kw = {k: (_to(v, dev) if isinstance(v, torch.Tensor) else v) for k, v in kw.items()}
    logits = logits.to(dev)
    out = ops.sample(logits, **kw)
    torch.cuda.synchronize()
    out = ops.SampleOutput(*[t.cpu() for t in out])
    hist = kw.get("history")
    spread = ops.sample_spread(
        logits, temperature=kw["temperature"], top_k=kw.get("top_k", 0),
        top_p=kw.get("top_p", 1.0), repetition_penalty=kw.get("repetition_penalty", 1.0),
        hist_len=0 if hist is None else hist.shape[1], has_mask=kw.get("allow_mask") is not None)
    if spread or route is not None:
        direct, took = _capi.sample_rows(logits, **kw)
        assert route is None or took == route, (took, route)
        ok = out.status == 0
        for f in ("status", "ids", "kept", "thresh_id", "thresh_value"):
            a, b = getattr(out, f), direct[f]
            if f not in ("status", "ids"):
                a, b = a[ok], b[ok]
            if f == "thresh_value":
                a, b = a.view(torch.int32), b.view(torch.int32)
            assert torch.equal(a, b), (f, took)
        for f in ("logprob", "sampled_logprob"):
            a, b = getattr(out, f)[ok], direct[f][ok]
            assert torch.allclose(a, b, rtol=0.0, atol=TOL, equal_nan=True), (f, took)
    return out


def assert_parity(g, ref, what=""):
    st = g.status.numpy()
    assert np.array_equal(st, ref.status), (what, st, ref.status)
    assert np.array_equal(g.ids.numpy(), ref.ids), (what, g.ids.numpy(), ref.ids)
    ok = ref.status == 0
    assert np.array_equal(g.kept.numpy()[ok], ref.kept[ok]), what
    assert np.array_equal(g.thresh_id.numpy()[ok], ref.thresh_id[ok]), what
    assert np.array_equal(g.thresh_value.numpy()[ok].view(np.uint32),
                          ref.thresh_value[ok].view(np.uint32)), what
    if ok.any():
        # NaN where the oracle has NaN (greedy rows holding a NaN or +inf),
        # -inf where it has -inf, within TOL elsewhere
        for got, want in ((g.logprob.numpy()[ok], ref.logprob[ok]),
                          (g.sampled_logprob.numpy()[ok], ref.sampled_logprob[ok])):
            assert np.array_equal(np.isnan(got), np.isnan(want)), what
            assert np.array_equal(np.isneginf(got), np.isneginf(want)), what
            fin = np.isfinite(want)
            if fin.any():
                assert np.abs(got[fin] - want[fin]).max() <= TOL, what


@pytest.mark.parametrize("cfg", [1, 2, 3, 5])
def test_workload_parity(cfg):
    wl = W.sampler_workload(cfg)
    print(f"workload {cfg} shape {wl.shape}", flush=True)
    ref = oracle_sample(wl.logits, **wl.kwargs())
    g = gpu_sample(wl.logits, **wl.kwargs())
    assert_parity(g, ref, f"cfg{cfg}")
    for r, t in wl.single_rows.items():
        assert int(g.ids[r]) == t


@pytest.mark.parametrize("cfg", [1, 5])
@pytest.mark.parametrize("variant", ["greedy", "top_p_only", "top_k_300", "rho_below_1"])
def test_workload_variants(cfg, variant):
    """The same inputs through the other selection paths (greedy, general
    path for top-p only / large k / rho < 1)."""
    wl = W.sampler_workload(cfg, rows=16)
    kw = wl.kwargs()
    if variant == "greedy":
        kw["temperature"] = 0.0
    elif variant == "top_p_only":
        kw["top_k"] = 0
    elif variant == "top_k_300":
        kw["top_k"] = 300
    else:
        kw["repetition_penalty"] = 0.8
    print(f"cfg {cfg} variant {variant}", flush=True)
    assert_parity(gpu_sample(wl.logits, **kw), oracle_sample(wl.logits, **kw), variant)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [1000, 1001, 4099, 32768 + 5])
def test_dtypes_and_odd_vocab(dtype, V):
    g = torch.Generator().manual_seed(V)
    x = (torch.randn(6, V, generator=g) * 3).to(dtype)
    u = W.uniforms_24(6, g, "cpu")
    hist = torch.randint(0, V, (6, 17), generator=g, dtype=torch.int32)
    for kw in (dict(temperature=0.7, top_k=20, top_p=0.9, repetition_penalty=1.1, history=hist),
               dict(temperature=1.3, top_k=0, top_p=0.8),
               dict(temperature=0.0)):
        print(dtype, V, kw.keys(), flush=True)
        assert_parity(gpu_sample(x, uniforms=u, **kw), oracle_sample(x, uniforms=u, **kw))


def test_strided_rows_last_position():
    """logits[:, -1, :] of a [B, S, V] tensor (the call-site layout)."""
    g = torch.Generator().manual_seed(1)
    full = (torch.randn(5, 3, 2000, generator=g) * 2).to(torch.bfloat16)
    u = W.uniforms_24(5, g, "cpu")
    dev = torch.device("cuda:0")
    view = full.to(dev)[:, -1, :]
    assert view.stride(0) == 3 * 2000
    out = ops.sample(view, temperature=0.9, top_k=10, uniforms=u.to(dev))
    ref = oracle_sample(full[:, -1, :].contiguous(), temperature=0.9, top_k=10, uniforms=u)
    torch.cuda.synchronize()
    assert np.array_equal(out.ids.cpu().numpy(), ref.ids)


def test_status_rows_and_padding():
    V = 300
    x = torch.zeros(8, V)
    x[0, 3] = float("nan")
    x[1, 4] = float("inf")
    bits = torch.ones(8, V, dtype=torch.bool)
    bits[2] = False
    bits[3] = False
    bits[3, 39] = True
    hist = torch.full((8, 2), -1, dtype=torch.int32)
    hist[4, 1] = V
    u = torch.full((8,), 0.5)
    u[5] = 1.0
    x[6] = float("-inf")
    x[7] = torch.arange(V, dtype=torch.float32) % 7
    fin = torch.zeros(8, dtype=torch.bool)
    fin[7] = True
    kw = dict(temperature=1.0, repetition_penalty=1.2, history=hist,
              allow_mask=W.pack_mask(bits), uniforms=u, finished=fin, pad_token_id=-5)
    assert_parity(gpu_sample(x, **kw), oracle_sample(x, **kw))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("params", [dict(temperature=0.0), dict(temperature=1.0, top_k=5),
                                    dict(temperature=1.0, top_p=0.9),
                                    dict(temperature=0.7, top_k=300, top_p=0.9)])
def test_rows_without_a_finite_value(dtype, params):
    """Rows of NaN only, NaN with -inf only, and -inf only (no finite value
    anywhere): non-finite for the first two and empty for the last, on every
    kernel the call routes to (a NaN sum must survive merges of partial
    log-sum-exps whose maxima are all -inf)."""
    V = 1000
    x = torch.randn(6, V)
    x[0] = float("nan")
    x[1] = float("-inf")
    x[1, ::3] = float("nan")
    x[2] = float("-inf")
    x[3, 17] = float("nan")
    x[4] = float("-inf")
    x[4, 999] = 2.0
    x = x.to(dtype)
    kw = dict(params, uniforms=torch.full((6,), 0.25))
    g = gpu_sample(x, **kw)
    if params["temperature"] > 0:
        assert g.status.tolist()[:4] == [1, 1, 2, 1], (dtype, params, g.status)
    else:  # greedy is torch.argmax: NaN, then +inf, win; all -inf gives id 0
        assert g.status.tolist() == [0] * 6, (dtype, g.status)
        assert g.ids.tolist() == torch.argmax(x.float(), dim=-1).tolist()
    assert_parity(g, oracle_sample(x, **kw), f"{dtype} {params}")


@pytest.mark.parametrize("top_k", [0, 1, 7, 256, 257, 5000])
def test_heavy_ties(top_k):
    """Uniform and few-valued rows: ties resolve by id (radix fallback when
    the tied bin overflows the collector)."""
    V = 20000
    x = torch.zeros(4, V, dtype=torch.bfloat16)
    x[1] = (torch.arange(V) % 3).to(torch.bfloat16)
    x[2, 100:200] = 5.0
    x[3] = (torch.arange(V) % 50).to(torch.bfloat16) * 0.25
    u = torch.tensor([0.0, 0.37, 0.999, 1 - 2**-24])
    for p in (1.0, 0.6):
        kw = dict(temperature=0.5, top_k=top_k, top_p=p, uniforms=u)
        print("ties", top_k, p, flush=True)
        assert_parity(gpu_sample(x, **kw), oracle_sample(x, **kw), f"k{top_k} p{p}")


def test_uniform_edges_and_single_allowed():
    g = torch.Generator().manual_seed(9)
    V = 151936
    x = (torch.randn(6, V, generator=g) * 2.5).to(torch.bfloat16)
    bits = torch.rand(6, V, generator=g) < 0.001
    bits[4] = False
    bits[4, 77777] = True
    bits[5] = False
    bits[5, V - 1] = True
    u = torch.tensor([0.0, 2**-24, 0.5, 1 - 2**-24, 0.25, 0.75])
    kw = dict(temperature=0.8, top_p=0.9, allow_mask=W.pack_mask(bits), uniforms=u)
    g_out = gpu_sample(x, **kw)
    assert_parity(g_out, oracle_sample(x, **kw))
    assert int(g_out.ids[4]) == 77777 and int(g_out.ids[5]) == V - 1


def test_drawn_uniforms_are_randint_over_2_to_24():
    """ops.draw_uniforms: u = randint(0, 2^24) * 2^-24 from the generator's
    state, whichever dtype randint is asked for."""
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(11)
    u = ops.draw_uniforms(4099, dev, g)
    g.manual_seed(11)
    k = torch.randint(0, 1 << 24, (4099,), device=dev, generator=g, dtype=torch.int32)
    assert u.dtype == torch.float32
    assert torch.equal(u, k.to(torch.float64).mul(2.0 ** -24).to(torch.float32))
    assert float(u.min()) >= 0.0 and float(u.max()) < 1.0


def test_deterministic_repeat():
    wl = W.sampler_workload(5, rows=32)
    a = gpu_sample(wl.logits, **wl.kwargs())
    b = gpu_sample(wl.logits, **wl.kwargs())
    assert torch.equal(a.ids, b.ids) and torch.equal(a.sampled_logprob, b.sampled_logprob)


def test_rejects_cpu_tensors_and_bad_args():
    x = torch.zeros(2, 10)
    with pytest.raises(RuntimeError):
        ops.sample(x, temperature=0.0)
    xd = x.cuda()
    with pytest.raises(RuntimeError):
        ops.sample(xd, temperature=1.0, repetition_penalty=0.0, uniforms=torch.zeros(2).cuda())
    with pytest.raises(RuntimeError):
        ops.sample(torch.zeros(2, (1 << 18) + 8).cuda(), temperature=0.0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [333, 4096, 151936])
def test_greedy_non_finite_rows_match_torch_argmax(dtype, V):
    """Greedy decoding is the reference's logits.argmax(dim=-1)
    (tensor_utils.py:658): the first NaN wins, then the first +inf, ties and
    all -inf rows go to the lowest id.  Checked against torch.argmax on the
    same device rows and against the oracle, on the row-wise kernel (V 333)
    and the split kernel (one and several slices per row)."""
    g = torch.Generator().manual_seed(V)
    B = 10
    x = torch.randn(B, V, generator=g)
    nan, inf = float("nan"), float("inf")
    x[0, [V // 3, 7, V - 2]] = nan
    x[1, [V // 2, 12]] = inf
    x[2, V // 4] = inf
    x[2, V - 30] = nan
    x[3] = -inf
    x[4] = -inf
    x[4, [V // 3, 5]] = nan
    x[5] = nan
    x[6, 17] = -inf
    x[7, [3, V - 1]] = 9.0
    x[8, V // 2] = -inf
    x[8, V // 2 + 1] = inf
    x[9, V - 1] = nan
    x = x.to(dtype)
    print(f"greedy non-finite {dtype} V={V}", flush=True)
    got = gpu_sample(x, temperature=0.0)
    want = torch.argmax(x.to("cuda:0"), dim=-1).cpu()
    assert got.status.tolist() == [0] * B, got.status
    assert torch.equal(got.ids, want), (got.ids, want)
    assert_parity(got, oracle_sample(x, temperature=0.0), "greedy non-finite")
    # the drop-in returns the same ids without raising
    from graspo_amd import tensor_utils as tu
    ids = tu._next_token_from_logits(x.to("cuda:0"), temperature=0.0, top_p=1.0)
    assert torch.equal(ids.cpu(), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_greedy_non_finite_rows_under_mask_and_penalty(dtype):
    """The argmax runs over allowed tokens with penalised values: a masked
    NaN or +inf loses, a row whose allowed tokens are all -inf returns its
    first allowed token, no allowed token is EMPTY, and a penalty can push a
    finite value to +inf (x / rho, rho < 1).  Against the oracle, on both
    kernels."""
    for V in (333, 151936):
        g = torch.Generator().manual_seed(V + 1)
        B = 6
        x = torch.randn(B, V, generator=g)
        nan, inf = float("nan"), float("inf")
        x[0, [40, 7]] = nan
        x[1, [90, 12]] = inf
        x[2] = -inf
        x[3, 100] = 3.0e38
        x[4, 200] = nan
        bits = torch.rand(B, V, generator=g) < 0.3
        bits[0, 40] = False
        bits[0, 7] = True
        bits[1, [90, 12]] = False
        bits[2] = False
        bits[2, [77, 210]] = True
        bits[3, 100] = True
        bits[5] = False
        hist = torch.full((B, 4), -1, dtype=torch.int32)
        hist[3, 0] = 100
        hist[4, 0] = 200
        x = x.to(dtype)
        kw = dict(temperature=0.0, allow_mask=W.pack_mask(bits), history=hist,
                  repetition_penalty=0.5)
        print(f"greedy non-finite masked {dtype} V={V}", flush=True)
        got = gpu_sample(x, **kw)
        ref = oracle_sample(x, **kw)
        assert ref.ids[0] == 7 and ref.ids[2] == 77 and ref.ids[3] == 100 and ref.status[5] == 2
        assert_parity(got, ref, f"greedy masked V={V}")


@pytest.mark.parametrize("kw", [dict(temperature=0.7, top_p=0.9), dict(temperature=0.7, top_p=1.0),
                                dict(temperature=1.0, top_p=0.5, repetition_penalty=1.3),
                                dict(temperature=0.7, top_k=300000, top_p=1.0)])
def test_fp32_rows_that_are_not_bf16_values_full_vocab(kw):
    """fp32 rows whose values are not bf16 values at V = 248320 (they take
    the row-wise kernel's general path): N(0, 3) with spikes, T 0.7 spreads
    the processed logits past the bins' 32-nat range, so the bottom bin
    holds most of the row; with neither top-k nor top-p the last kept rank
    is the row's last token, found without collecting that bin."""
    B, V = 24, 248320
    g = torch.Generator().manual_seed(31)
    x = torch.randn(B, V, generator=g) * 3.0
    x[:4, :3] += 12.0
    assert bool((x.to(torch.bfloat16).float() != x).any())
    u = torch.randint(0, 1 << 24, (B,), generator=g).float() * 2.0 ** -24
    if "repetition_penalty" in kw:
        kw = dict(kw, history=torch.randint(-1, V, (B, 1000), generator=g, dtype=torch.int32))
    got = gpu_sample(x, uniforms=u, **kw)
    ref = oracle_sample(x, uniforms=u, **kw)
    assert_parity(got, ref, f"fp32 full vocab {kw.get('temperature')} {kw.get('top_p')}")
