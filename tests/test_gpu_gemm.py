"""GPU tests of the matrix-core path of kvattn_gemv (batches of tokens) and of
kvattn_gemv_qkv_append on it.

Bound: FP32 sums of exact products in any order differ from the exact sum by at most
(K + 8) 2^-24 sum |w x| (the row scale, the bias and the output's rounding included in the 8),
which _bound computes for every output; float outputs are asked for, so nothing else rounds.
"""
import numpy as np
import pytest

from oracle import oracle
from test_gpu_gemv import _kv, _make, _run

pytestmark = pytest.mark.gpu


def _bound(h, B, M, K):
    W, x = np.abs(h["W"]).reshape(M, K).astype(np.float64), np.abs(h["x"]).reshape(B, K).astype(np.float64)
    s = np.ones(M) if h["scale"] is None else np.abs(h["scale"]).astype(np.float64)
    b = np.zeros(M) if h["bias"] is None else np.abs(h["bias"]).astype(np.float64)
    return (K + 8) * 2.0 ** -24 * ((x @ W.T) * s + b)


def _exact(h, B, M, K):
    y = h["x"].reshape(B, K).astype(np.float64) @ h["W"].reshape(M, K).astype(np.float64).T
    y = y if h["scale"] is None else y * h["scale"].astype(np.float64)
    return y if h["bias"] is None else y + h["bias"].astype(np.float64)


def _guarded(t):
    """The same values, followed in memory by NaNs (NaN codes)."""
    import torch
    flat = t.reshape(-1)
    fill = torch.full((4096,), 0x7F if t.dtype == torch.uint8 else float("nan"), dtype=t.dtype)
    return torch.cat([flat, fill])


@pytest.mark.parametrize("dtype", ["f32", "bf16", "int8", "fp8"])
@pytest.mark.parametrize("B,M,K", [(4, 1, 16), (8, 15, 48), (15, 16, 64), (16, 17, 80), (17, 63, 784), (33, 130, 768),
                                   (64, 40, 1040), (9, 8191, 32), (40, 33, 5136)])
def test_batch_against_float64(dev, dtype, B, M, K):
    """Tiles of 16 rows x 16 tokens that are full, one short and one over; rows of one chunk, of a
    partial last step, of fewer steps than waves and of several blocks of loads; NaNs right
    behind the weights and the tokens."""
    d, h = _make(dtype, B, M, K, seed=B * 1000 + M + K)
    d = dict(d, W=_guarded(d["W"]), x=_guarded(d["x"]))
    got, _ = _run(d, dtype, B, M, K, False, False, out_dtype="f32")
    err = np.abs(got.reshape(B, M).astype(np.float64) - _exact(h, B, M, K))
    assert np.all(err <= _bound(h, B, M, K)), float((err / _bound(h, B, M, K)).max())


@pytest.mark.parametrize("dtype", ["bf16", "int8", "fp8"])
@pytest.mark.parametrize("B,M,K", [(9, 20000, 32), (17, 20001, 144), (33, 20015, 272), (64, 20017, 528),
                                   (70, 24571, 64), (16, 65537, 48)])
def test_tall_batch_against_float64(dev, dtype, B, M, K):
    """From 20000 rows on the tokens sit in LDS: 16, 32 or 64 of them, rows in whole and partial
    tiles of 16 and in several tiles per wave (65537 rows), M not a multiple of 4, K of a partial
    block of steps, and tokens beyond one workgroup's."""
    d, h = _make(dtype, B, M, K, seed=B + M + K)
    d = dict(d, W=_guarded(d["W"]), x=_guarded(d["x"]))
    got, _ = _run(d, dtype, B, M, K, False, False, out_dtype="f32")
    bound = _bound(h, B, M, K)
    err = np.abs(got.reshape(B, M).astype(np.float64) - _exact(h, B, M, K))
    assert np.all(err <= bound), float((err / bound).max())


@pytest.mark.parametrize("out_dtype", ["f32", "bf16"])
def test_tall_batch_gelu_and_unaligned_outputs(dev, out_dtype):
    """GELU and pre_gelu from the kernel with tokens in LDS, into outputs that vector stores fit and
    into ones a single element further on: the same values."""
    import torch
    kvattn = _kv()
    B, M, K = 20, 20480, 96
    d, h = _make("bf16", B, M, K, seed=9)
    odt = torch.float32 if out_dtype == "f32" else torch.bfloat16
    dd = {k: v.to(dev) for k, v in d.items() if v is not None}
    got = []
    for shift in (0, 1):
        out, pre = (torch.full((B * M + 1,), float("nan"), dtype=odt, device=dev)[shift:shift + B * M] for _ in range(2))
        kvattn.gemv(out, dd["W"], dd["x"], B, M, K, w_dtype="bf16", bias=dd["bias"], pre_gelu=pre, gelu=True,
                    out_dtype=out_dtype)
        got.append((out.float().cpu().numpy(), pre.float().cpu().numpy()))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
    ref, rpre = oracle.gemv(h["W"], h["x"], B, M, K, bias=h["bias"], gelu=True, want_pre=True)
    tol = 1e-5 if out_dtype == "f32" else 1e-2
    for g, r in ((got[0][0], ref), (got[0][1], rpre)):
        assert np.abs(g - r.reshape(-1)).max() <= tol * np.abs(r).max()


@pytest.mark.parametrize("dtype", ["f32", "bf16", "int8", "fp8"])
def test_batch_gelu_and_pre_gelu(dev, dtype):
    B, M, K = 19, 200, 304
    d, h = _make(dtype, B, M, K, seed=77)
    got, pre = _run(d, dtype, B, M, K, True, True)
    ref, rpre = oracle.gemv(h["W"], h["x"], B, M, K, w_scale=h["scale"], bias=h["bias"], gelu=True, want_pre=True)
    tol = 1e-5 if dtype == "f32" else 1e-2     # the activations' type
    for g, r in ((got, ref), (pre, rpre)):
        g, r = g.reshape(B, M).astype(np.float64), r.reshape(B, M).astype(np.float64)
        assert np.abs(g - r).max() <= tol * np.abs(r).max()


@pytest.mark.parametrize("dtype", ["f32", "bf16", "int8"])
def test_batch_special_values(dev, dtype):
    """Infinities, NaNs, subnormal and huge activations: each token of a batch as that token
    alone (the vector units' path), NaN for NaN, infinity for infinity, and within the bound."""
    import torch
    B, M, K = 8, 48, 256
    d, h = _make(dtype, B, M, K, seed=5)
    x = d["x"].reshape(B, K).clone()
    x[1, 3], x[2, 200], x[3, 17] = float("inf"), float("nan"), float("-inf")
    x[3, 18] = float("inf")
    x[4] *= 1e-39          # subnormal activations
    x[5] *= 1e35
    x[6] = 0
    d = dict(d, x=x)
    whole, _ = _run(d, dtype, B, M, K, False, False, out_dtype="f32")
    whole = whole.reshape(B, M)
    h = dict(h, x=x.float().numpy())
    for b in range(B):
        one, _ = _run(dict(d, x=x[b].contiguous()), dtype, 1, M, K, False, False, out_dtype="f32")
        assert np.array_equal(np.isnan(one), np.isnan(whole[b])), b
        inf = np.isinf(one)
        assert np.array_equal(one[inf], whole[b][inf]), b
        if b not in (1, 2, 3):
            bound = 2 * _bound(dict(h, x=h["x"][b]), 1, M, K)[0]
            assert np.all(np.abs(one.astype(np.float64) - whole[b]) <= bound), b


@pytest.mark.parametrize("dtype", ["bf16", "int8", "fp8"])
@pytest.mark.parametrize("B,M,K", [(16, 20000, 320), (20, 20001, 320), (40, 20000, 336), (20, 20000, 704),
                                   (40, 20000, 960), (18, 65537, 80), (40, 20000, 1152), (20, 48, 336)])
def test_special_values_in_the_last_steps_of_a_row(dev, dtype, B, M, K):
    """Infinities and NaNs in a row's last step and last chunk, where the row's steps do not fill
    the blocks of the kernel with tokens in LDS (M >= 20000; 48 rows: 16 x 16 tiles): each token as
    that token alone (the vector units' path), and the other tokens within the bound.  The last
    token keeps its own infinity behind a partial step's zeros."""
    import torch
    d, h = _make(dtype, B, M, K, seed=11, with_bias=False)
    x = d["x"].reshape(B, K).clone()
    x[1, K - 1], x[2, K - 20], x[3, K - 5], x[4, 0] = float("inf"), float("-inf"), float("nan"), float("inf")
    x[B - 1, K - 16:] = float("inf")
    d = dict(d, x=x)
    whole, _ = _run(d, dtype, B, M, K, False, False, out_dtype="f32")
    whole = whole.reshape(B, M)
    special = (1, 2, 3, 4, B - 1)
    for b in special:
        one, _ = _run(dict(d, x=x[b].contiguous()), dtype, 1, M, K, False, False, out_dtype="f32")
        assert np.array_equal(np.isnan(one), np.isnan(whole[b])), b
        inf = np.isinf(one)
        assert np.array_equal(one[inf], whole[b][inf]) and (inf.any() or b in (3, B - 1)), b
    rest = [b for b in range(B) if b not in special]
    hr = dict(h, x=h["x"].reshape(B, K)[rest])
    err = np.abs(whole[rest].astype(np.float64) - _exact(hr, len(rest), M, K))
    assert np.all(err <= _bound(hr, len(rest), M, K))


@pytest.mark.parametrize("dtype,kv", [("f32", "f32"), ("bf16", "bf16"), ("int8", "bf16"), ("bf16", "int8"),
                                      ("bf16", "fp8"), ("int8", "int8"), ("fp8", "fp8")])
@pytest.mark.parametrize("B,NH", [(9, 5), (16, 12), (33, 3)])
def test_batch_qkv_append_equals_gemv_then_append(dev, dtype, kv, B, NH):
    """qkv, cache bytes and row scales bit for bit, with per-sequence lengths (one beyond maxT)."""
    import torch
    kvattn = _kv()
    HS, K, maxT = 64, 16 * 21, 40
    M = 3 * NH * HS
    d, _ = _make(dtype, B, M, K, seed=B + NH)
    W, x, bias = d["W"].to(dev), d["x"].to(dev).contiguous(), d["bias"].to(dev)
    scale = None if d.get("scale") is None else d["scale"].to(dev)
    act = torch.float32 if dtype == "f32" else torch.bfloat16
    w8 = kv in ("int8", "fp8")
    n = 2 * B * NH * maxT
    cache = torch.zeros(n * HS, dtype=torch.uint8 if w8 else act, device=dev)
    ks_a, ks_b = (torch.zeros(n, device=dev) if w8 else None for _ in range(2))
    nws = kvattn.gemv_qkv_append_workspace_bytes(B, NH)
    ws = torch.zeros(nws, dtype=torch.uint8, device=dev)
    cur = torch.tensor([(7 * b) % maxT for b in range(B - 1)] + [maxT + 5], dtype=torch.int32, device=dev)
    c_a, c_b = cache.clone(), cache.clone()
    q_a, q_b = (torch.empty(B * M, dtype=act, device=dev) for _ in range(2))
    kvattn.gemv(q_a, W, x, B, M, K, w_dtype=dtype, w_scale=scale, bias=bias)
    kvattn.kv_cache_write(c_a, q_a, B, NH, HS, maxT, kv_dtype=kv, kv_scale=ks_a, cur_len=cur, lens_per_seq=True)
    kvattn.gemv_qkv_append(q_b, W, x, B, NH, HS, K, c_b, maxT, w_dtype=dtype, kv_dtype=kv, w_scale=scale, bias=bias,
                           kv_scale=ks_b, cur_len=cur, lens_per_seq=True, workspace=ws, workspace_nbytes=nws)
    torch.cuda.synchronize()
    assert torch.equal(q_a.view(torch.uint8), q_b.view(torch.uint8))
    assert torch.equal(c_a.view(torch.uint8), c_b.view(torch.uint8))
    if w8:
        assert torch.equal(ks_a.view(torch.int32), ks_b.view(torch.int32))
    assert c_b.view(torch.uint8).any()


@pytest.mark.parametrize("dtype,kv", [("bf16", "bf16"), ("int8", "bf16"), ("bf16", "int8"), ("fp8", "fp8")])
@pytest.mark.parametrize("B", [9, 20, 33])
def test_tall_qkv_append_equals_gemv_then_append(dev, dtype, kv, B):
    """The same from 20000 rows on (105 heads), where the plain projection keeps its tokens in LDS."""
    test_batch_qkv_append_equals_gemv_then_append(dev, dtype, kv, B, 105)


def test_tall_batch_in_a_graph(dev):
    """The kernel with tokens in LDS (more than 64 KB of it) captured and replayed over new tokens,
    with eager work in between: every replay as the eager call."""
    import torch
    kvattn = _kv()
    B, M, K = 64, 20000, 768
    d, _ = _make("bf16", B, M, K, seed=3, with_bias=False)
    W, x = d["W"].to(dev), d["x"].to(dev).reshape(B, K).contiguous()
    out, ref = (torch.empty(B, M, device=dev) for _ in range(2))
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        kvattn.gemv(out, W, x, B, M, K, w_dtype="bf16", out_dtype="f32")
    for rep in range(3):
        x.copy_(x.roll(rep + 1, dims=0))
        kvattn.gemv(ref, W, x, B, M, K, w_dtype="bf16", out_dtype="f32")
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), rep
