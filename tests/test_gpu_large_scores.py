"""Scores far beyond any softmax's range: the largest takes all the weight, so the output is its V
row, and every plan has to find that.  A score that is rounded in one place and not in another
(in the lanes of a row, or between the maximum and the distance from it) shows here, as its
error grows with the score: up to a few 2^-24 of it, in the exponent."""
import pytest

pytestmark = pytest.mark.gpu
HS = 64


@pytest.mark.parametrize("dtype", ["f32", "bf16", "int8", "fp8"])
@pytest.mark.parametrize("B,NH,maxT,hinted,ragged,strategy", [
    (1, 12, 128, True, False, "auto"), (2, 12, 250, False, False, "auto"), (1, 12, 700, True, False, "auto"),
    (1, 12, 1024, False, False, "auto"), (48, 12, 300, True, False, "auto"), (48, 12, 300, False, True, "auto"),
    (64, 12, 320, False, True, "auto"), (40, 12, 700, False, False, "auto"), (40, 12, 700, True, True, "auto"),
    (16, 12, 2048, True, False, "auto"), (3, 5, 900, False, True, "split_merge"), (3, 5, 900, False, True, "lastblock")])
def test_the_largest_score_takes_all(dev, dtype, B, NH, maxT, hinted, ragged, strategy):
    import torch
    from cuda_gpt2_inference_amd import kvattn
    g = torch.Generator(device=dev)
    g.manual_seed(B * maxT)
    act = torch.float32 if dtype == "f32" else torch.bfloat16
    x = torch.randn(2, B, NH, maxT, HS, generator=g, device=dev)
    scale = None
    if dtype in ("int8", "fp8"):
        scale = x.abs().amax(-1) / (448.0 if dtype == "fp8" else 127.0)
        y = x / scale[..., None]
        codes = y.to(torch.float8_e4m3fn) if dtype == "fp8" else y.round().to(torch.int8)
        rows, cache = codes.float().double() * scale[..., None].double(), codes.view(torch.uint8)
    else:
        cache = x.to(act)
        rows = cache.double()
    q0 = torch.randn(B, 3, NH, HS, generator=g, device=dev)
    if ragged:
        cur = torch.randint(1, maxT, (B,), generator=g, device=dev, dtype=torch.int32)
        cur[0] = maxT - 1
    else:
        cur = torch.tensor([maxT - 1], dtype=torch.int32, device=dev)
    live = torch.arange(maxT, device=dev)[None] <= (cur if ragged else cur.expand(B))[:, None]
    ws = kvattn.Workspace(B, NH, maxT)
    for mag in (1e6, 1e9, 1e15, 1e25):
        qkv = (q0 * mag).to(act)
        s = torch.einsum("bhd,bhtd->bht", qkv[:, 0].double(), rows[0]).masked_fill(~live[:, None], -float("inf"))
        top = s.topk(2, dim=-1)
        # Heads whose two largest scores FP32 products and sums tell apart with certainty: 64 products and
        # their sum, each score to (64 + 4) 2^-24 of the sum of its products' magnitudes.
        size = torch.einsum("bhd,bhtd->bht", qkv[:, 0].double().abs(), rows[0].abs()).masked_fill(~live[:, None], 0)
        sure = top.values[..., 0] - top.values[..., 1] > 2 * 68 * 2.0 ** -24 * size.amax(-1) + 8 * 150
        sure &= top.values[..., 1] > -float("inf")
        assert sure.double().mean() > 0.9, mag
        want = rows[1].gather(2, top.indices[..., :1, None].expand(-1, -1, -1, HS))[:, :, 0]
        out = torch.full((B, NH, HS), float("nan"), dtype=act, device=dev)
        kvattn.decode(out, qkv, cache, B, NH, HS, maxT, kv_dtype=dtype, kv_scale=scale, cur_len=cur, lens_per_seq=ragged,
                      len_hint=maxT - 1 if hinted else -1, strategy=strategy, **ws.kwargs())
        torch.cuda.synchronize()
        # One V row times a weight of 1 over a sum of 1, rounded to the output's type.
        ulp = 2.0 ** -22 if dtype == "f32" else 2.0 ** -8
        err = ((out.double() - want).abs() - ulp * want.abs())[sure]
        assert torch.isfinite(out[sure].float()).all() and err.max() <= 1e-30, (mag, float(err.max()))
