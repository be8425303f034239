"""The one-wave-per-row projection over a few vectors: each vector's result is the one it has alone,
bit for bit (the same products in the same order), at the edges of the chunks a lane holds, with
the last wave partly beyond the rows, GELU with the pre-activation, and the cache append."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "bf16", "int8", "fp8"])
@pytest.mark.parametrize("lane_chunks", [1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 13, 16, 17])
@pytest.mark.parametrize("edge", [-16, 0])
def test_vectors_are_those_of_single_calls(dev, dtype, lane_chunks, edge):
    import torch
    from cuda_gpt2_inference_amd import kvattn
    per = {"f32": 4, "bf16": 8}.get(dtype, 16)
    K, M = 64 * per * lane_chunks + edge, 37
    # Vectors that stay with this kernel: FP32 7 over rows of 1600 < K <= 4096, else 3.
    B = 2 if dtype != "f32" else (7 if 1600 < K <= 4096 else 3)
    g = torch.Generator(device=dev)
    g.manual_seed(K)
    act = torch.float32 if dtype == "f32" else torch.bfloat16
    x = torch.randn(B, K, generator=g, device=dev).to(act)
    bias = torch.randn(M, generator=g, device=dev).to(act)
    scale = None
    if dtype in ("int8", "fp8"):
        W = torch.randint(0, 120, (M, K), generator=g, device=dev, dtype=torch.uint8)
        scale = 1e-3 * torch.rand(M, generator=g, device=dev)
    else:
        W = torch.randn(M, K, generator=g, device=dev).to(act)
    kw = dict(w_dtype=dtype, w_scale=scale, bias=bias, gelu=True)
    got = [torch.full((B, M), float("nan"), dtype=act, device=dev) for _ in range(2)]
    kvattn.gemv(got[0], W, x, B, M, K, pre_gelu=got[1], **kw)
    for b in range(B):
        one = [torch.full((1, M), float("nan"), dtype=act, device=dev) for _ in range(2)]
        kvattn.gemv(one[0], W, x[b:b + 1].contiguous(), 1, M, K, pre_gelu=one[1], **kw)
        torch.cuda.synchronize()
        for o, w in zip(one, got):
            assert torch.isfinite(o).all() and torch.equal(o[0], w[b])


@pytest.mark.parametrize("dtype,B,K", [("f32", 3, 1024), ("f32", 2, 2048), ("f32", 2, 4096), ("bf16", 2, 3072),
                                       ("bf16", 2, 2048), ("int8", 2, 4096), ("fp8", 2, 1040)])
@pytest.mark.parametrize("M", [1024, 1025, 1536, 1537, 3073, 4096, 4097])
def test_vectors_keep_their_bits_at_every_height(dev, dtype, B, K, M):
    """On either side of the heights up to which the next vector's x is requested ahead."""
    import torch
    from cuda_gpt2_inference_amd import kvattn
    g = torch.Generator(device=dev)
    g.manual_seed(K + M)
    act = torch.float32 if dtype == "f32" else torch.bfloat16
    x = torch.randn(B, K, generator=g, device=dev).to(act)
    scale = None
    if dtype in ("int8", "fp8"):
        W = torch.randint(0, 120, (M, K), generator=g, device=dev, dtype=torch.uint8)
        scale = 1e-3 * torch.rand(M, generator=g, device=dev)
    else:
        W = torch.randn(M, K, generator=g, device=dev).to(act)
    kw = dict(w_dtype=dtype, w_scale=scale, out_dtype="f32")
    got = torch.full((B, M), float("nan"), device=dev)
    kvattn.gemv(got, W, x, B, M, K, **kw)
    for b in range(B):
        one = torch.full((1, M), float("nan"), device=dev)
        kvattn.gemv(one, W, x[b:b + 1].contiguous(), 1, M, K, **kw)
        torch.cuda.synchronize()
        assert torch.isfinite(one).all() and torch.equal(one[0], got[b]), b


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_append_of_two_vectors(dev, dtype):
    import torch
    from cuda_gpt2_inference_amd import kvattn
    B, NH, maxT, K = 2, 12, 16, 768
    g = torch.Generator(device=dev)
    g.manual_seed(1)
    act = torch.float32 if dtype == "f32" else torch.bfloat16
    x = torch.randn(B, K, generator=g, device=dev).to(act)
    W = torch.randn(3 * K, K, generator=g, device=dev).to(act)
    cur = torch.tensor([3, 15], dtype=torch.int32, device=dev)
    qkv = torch.empty(B, 3 * K, dtype=act, device=dev)
    cache = torch.zeros(2, B, NH, maxT, 64, dtype=act, device=dev)
    kvattn.gemv_qkv_append(qkv, W, x, B, NH, 64, K, cache, maxT, w_dtype=dtype, cur_len=cur,
                           lens_per_seq=True)
    ref = torch.empty_like(qkv)
    kvattn.gemv(ref, W, x, B, 3 * K, K, w_dtype=dtype)
    torch.cuda.synchronize()
    assert torch.equal(qkv, ref)
    want = torch.zeros_like(cache)
    for b, t in enumerate((3, 15)):
        want[:, b, :, t] = ref[b].view(3, NH, 64)[1:]
    assert torch.equal(cache, want)


@pytest.mark.parametrize("dtype,B,M,K", [("f32", 5, 1024, 1024), ("f32", 7, 260, 1040), ("f32", 7, 1024, 1600),
                                         ("f32", 4, 1280, 1040), ("f32", 11, 37, 4096), ("f32", 4, 200, 6144),
                                         ("f32", 5, 1024, 12288), ("f32", 4, 1300, 784), ("f32", 8, 1280, 4096),
                                         ("bf16", 4, 1000, 1616),
                                         ("bf16", 3, 70, 5136), ("bf16", 4, 256, 8192), ("bf16", 3, 100, 16384),
                                         ("int8", 3, 512, 4096), ("int8", 4, 768, 8192), ("fp8", 4, 300, 16384),
                                         ("int8", 3, 64, 32768), ("fp8", 3, 1024, 6144)])
def test_few_vectors_over_few_long_rows_keep_their_bits(dev, dtype, B, M, K):
    """Where a few long rows would leave most of the chip idle as matrix-core tiles, every vector is
    the one it is alone, bit for bit."""
    import torch
    from cuda_gpt2_inference_amd import kvattn
    g = torch.Generator(device=dev)
    g.manual_seed(M + K)
    act = torch.float32 if dtype == "f32" else torch.bfloat16
    x = torch.randn(B, K, generator=g, device=dev).to(act)
    scale = None
    if dtype in ("int8", "fp8"):
        W = torch.randint(0, 120, (M, K), generator=g, device=dev, dtype=torch.uint8)
        scale = 1e-3 * torch.rand(M, generator=g, device=dev)
    else:
        W = torch.randn(M, K, generator=g, device=dev).to(act)
    kw = dict(w_dtype=dtype, w_scale=scale, out_dtype="f32")
    got = torch.full((B, M), float("nan"), device=dev)
    kvattn.gemv(got, W, x, B, M, K, **kw)
    for b in range(B):
        one = torch.full((1, M), float("nan"), device=dev)
        kvattn.gemv(one, W, x[b:b + 1].contiguous(), 1, M, K, **kw)
        torch.cuda.synchronize()
        assert torch.isfinite(one).all() and torch.equal(one[0], got[b]), b
