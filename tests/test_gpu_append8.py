"""The 8-bit append inside the attention launches (the wave quantises a row together, one element
a lane) against kvattn_cache_write: cache bytes and row scales bit for bit, whatever the row."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
HS = 64


def _rows(seed):
    """bf16 rows: normal, one large element at every place in turn, zeros, subnormals, the largest
    finite values, infinities and single NaNs."""
    import torch
    r = np.random.RandomState(seed)
    rows = [r.standard_normal(HS) for _ in range(6)]
    for c in range(HS):
        x = r.standard_normal(HS)
        x[c] *= 100.0
        rows.append(x)
    rows += [np.zeros(HS), -np.zeros(HS), 1e-39 * r.standard_normal(HS), 3e38 * np.sign(r.standard_normal(HS))]
    for special in (np.inf, -np.inf, np.nan):
        x = r.standard_normal(HS)
        x[r.randint(HS)] = special
        rows.append(x)
    return torch.from_numpy(np.stack(rows).astype(np.float32)).to(torch.bfloat16)


@pytest.mark.parametrize("kv", ["int8", "fp8"])
@pytest.mark.parametrize("maxT,cur,hint,strategy", [(64, 5, 5, "auto"), (64, 63, -1, "auto"), (512, 300, -1, "auto"),
                                                    (512, 129, 129, "lastblock"), (700, 511, 511, "split_merge"),
                                                    (640, 600, 600, "fused_single")])
def test_append8_rows(dev, kv, maxT, cur, hint, strategy):
    import torch
    from cuda_gpt2_inference_amd import kvattn
    rows = _rows(11).to(dev)
    n = rows.shape[0]
    NH, B = 1, n
    qkv = torch.empty(B, 3, NH, HS, dtype=torch.bfloat16, device=dev)
    qkv[:, 0, 0] = 0.25
    qkv[:, 1, 0] = rows
    qkv[:, 2, 0] = rows.roll(1, dims=0)
    a = torch.zeros(2, B, NH, maxT, HS, dtype=torch.uint8, device=dev)
    s_a = torch.zeros(2, B, NH, maxT, device=dev)
    b, s_b = a.clone(), s_a.clone()
    d_cur = torch.tensor([cur], dtype=torch.int32, device=dev)
    out = torch.empty(B, NH, HS, dtype=torch.bfloat16, device=dev)
    ws = kvattn.Workspace(B, NH, maxT)
    kvattn.kv_cache_write(a, qkv, B, NH, HS, maxT, kv_dtype=kv, kv_scale=s_a, cur_len=d_cur)
    kvattn.append_decode(out, qkv, b, B, NH, HS, maxT, kv_dtype=kv, kv_scale=s_b, cur_len=d_cur, len_hint=hint,
                         strategy=strategy, **ws.kwargs())
    torch.cuda.synchronize()
    assert torch.equal(a, b)
    assert torch.equal(s_a.view(torch.int32), s_b.view(torch.int32))
    assert a[:, :, :, cur].any()


@pytest.mark.parametrize("kv", ["int8", "fp8"])
@pytest.mark.parametrize("ragged", [False, True])
def test_paged_append8_rows(dev, kv, ragged):
    import torch
    from cuda_gpt2_inference_amd import kvattn
    rows = _rows(12).to(dev)
    B, NH, P, n = rows.shape[0], 1, 64, 5
    qkv = torch.stack([torch.full_like(rows, 0.25), rows, rows.roll(1, dims=0)], dim=1).reshape(B, 3, NH, HS).contiguous()
    table = torch.randperm(B * n, device=dev).to(torch.int32).view(B, n)
    pools = [torch.zeros(B * n, 2, NH, P, HS, dtype=torch.uint8, device=dev) for _ in range(2)]
    scales = [torch.zeros(B * n, 2, NH, P, device=dev) for _ in range(2)]
    lens = [(37 * i) % (P * n) for i in range(B)] if ragged else [200]
    cur = torch.tensor(lens, dtype=torch.int32, device=dev)
    pc = [kvattn.PagedCache(p, table, n, P, B * n, s) for p, s in zip(pools, scales)]
    out = torch.empty(B, NH, HS, dtype=torch.bfloat16, device=dev)
    ws = kvattn.Workspace(B, NH, P * n)
    kvattn.paged_cache_write(pc[0], qkv, B, NH, HS, kv_dtype=kv, cur_len=cur, lens_per_seq=ragged)
    kvattn.paged_decode(out, qkv, pc[1], B, NH, HS, kv_dtype=kv, cur_len=cur, lens_per_seq=ragged, append=True,
                        **ws.kwargs())
    torch.cuda.synchronize()
    assert torch.equal(pools[0], pools[1])
    assert torch.equal(scales[0].view(torch.int32), scales[1].view(torch.int32))
    assert pools[0].any()
