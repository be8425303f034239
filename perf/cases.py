"""The work a decode engine has this library do, as cases that can be timed and checked.

Five kinds of case, each through the entry points of ``cuda_gpt2_inference_amd.kvattn``:

  stack   decode attention of every layer of one token (``decode`` or ``append_decode``),
          captured once in a HIP graph and replayed, as an engine's step graph is
  attn    one decode-attention call of a batch, contiguous or paged, issued eagerly
  step    a batch's decode step without the norms, which are the engine's own: per layer the
          QKV projection with the append in its epilogue, the attention, the attention output
          projection and the two MLP projections, in one HIP graph over all layers
  mlp     the two MLP projections of one layer, eagerly (GELU and pre_gelu)
  head    the vocabulary projection with float logits, eagerly

Values are N(0, 1) for q, K, V and activations and N(0, 1/K) for weights of K columns; 8-bit
caches and weights hold row-quantised codes of such values.
"""
import math

import torch

from cuda_gpt2_inference_amd import kvattn

HD = 64
VOCAB = 50304            # the padded vocabulary of the engine's embedding table
DTYPES = ("f32", "bf16", "int8", "fp8")
ROW_BYTES = {"f32": 256, "bf16": 128, "int8": 68, "fp8": 68}     # one K or V row, with its scale
W_BYTES = {"f32": 4, "bf16": 2, "int8": 1, "fp8": 1}
MAX_KV_BYTES = 1 << 30   # attended K and V bytes of a drawn call


def _attn(name, kv, B, NH, maxT, lens, hint, append=False, page_rows=0):
    return {"name": name, "kind": "attn", "kv": kv, "B": B, "NH": NH, "maxT": maxT, "lens": lens, "hint": hint,
            "append": append, "page_rows": page_rows}


def listed():
    """lens: > 0 one attended length for the batch, 0 per-sequence lengths ~ U[1, maxT]; hint:
    the host passes the longest length; page_rows > 0: a paged cache with shuffled pages."""
    return [
        # Token 1024 of a GPT-2 sequence: the 12 attention calls of its layers, BF16 cache.
        {"name": "stack_bf16_T1024", "kind": "stack", "kv": "bf16", "B": 1, "NH": 12, "maxT": 1024, "lens": 1024,
         "hint": True, "append": False, "layers": 12},
        # A token early in a sequence on the INT8 cache, from the one graph that serves every
        # length, with the append in the attention launch: the smallest calls there are.
        {"name": "stack_int8_append_T300", "kind": "stack", "kv": "int8", "B": 1, "NH": 12, "maxT": 1024, "lens": 300,
         "hint": False, "append": True, "layers": 12},
        # One user's whole decode step in BF16 (matrix-vector projections of every layer).
        {"name": "step_bf16_b1", "kind": "step", "w": "bf16", "kv": "bf16", "B": 1, "NH": 12, "maxT": 1024,
         "lens": 777, "layers": 12},
        # A small serving batch on INT8 weights and an INT8 cache, sequences of any length.
        {"name": "step_int8_b12", "kind": "step", "w": "int8", "kv": "int8", "B": 12, "NH": 12, "maxT": 1024,
         "lens": 0, "layers": 4},
        # A full serving batch in BF16.
        {"name": "step_bf16_b64", "kind": "step", "w": "bf16", "kv": "bf16", "B": 64, "NH": 12, "maxT": 1024,
         "lens": 0, "layers": 2},
        # Logits of one sequence from the INT8 embedding table, and of a batch from the BF16 one.
        {"name": "head_int8_b1", "kind": "head", "w": "int8", "B": 1, "M": VOCAB, "K": 768},
        {"name": "head_bf16_b64", "kind": "head", "w": "bf16", "B": 64, "M": VOCAB, "K": 768},
        # The FP32 build's MLP for a few sequences.
        {"name": "mlp_f32_b5", "kind": "mlp", "w": "f32", "B": 5, "C": 768},
        # 64 ragged sequences of up to 8192 positions: the largest call, bound by memory.
        _attn("attn_bf16_ragged_8192", "bf16", 64, 12, 8192, 0, False),
        # A paged FP8 cache of a serving batch, appending.
        _attn("attn_fp8_paged_ragged", "fp8", 24, 12, 4096, 0, True, append=True, page_rows=128),
        # INT8 sequences of one length, the Infinity-Cache-sized middle.
        _attn("attn_int8_b16_T4096", "int8", 16, 12, 4096, 4096, True),
        # FP32 cache, a medium batch, an odd length.
        _attn("attn_f32_b8_T1023", "f32", 8, 12, 1024, 1023, True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("stack", "attn", "attn", "step", "step", "mlp", "head"))
    B = _log_int(rng, 1, 64)
    NH = rng.choice((12, 12, rng.randint(4, 25)))
    if kind == "stack":
        return {"kind": kind, "kv": rng.choice(DTYPES), "B": rng.choice((1, 1, 2, 4)), "NH": NH, "maxT": 1024,
                "lens": _log_int(rng, 1, 1024), "hint": rng.random() < 0.5, "append": rng.random() < 0.5,
                "layers": 12}
    if kind == "attn":
        kv = rng.choice(DTYPES)
        most = MAX_KV_BYTES // (2 * B * NH * ROW_BYTES[kv])
        maxT = 64 * max(1, _log_int(rng, 64, min(8192, most)) // 64)
        ragged, paged = rng.random() < 0.5, rng.random() < 0.4
        return {"kind": kind, "kv": kv, "B": B, "NH": NH, "maxT": maxT,
                "lens": 0 if ragged else maxT - rng.randrange(maxT // 4 + 1), "hint": rng.random() < 0.7,
                "append": rng.random() < 0.5, "page_rows": 64 if paged else 0}
    if kind == "step":
        w = rng.choice(DTYPES)
        kv = "f32" if w == "f32" else rng.choice(("bf16", "int8", "fp8"))
        ragged = rng.random() < 0.5
        maxT = _log_int(rng, 64, 1024)
        return {"kind": kind, "w": w, "kv": kv, "B": B, "NH": min(NH, 16), "maxT": maxT,
                "lens": 0 if ragged else rng.randint(1, maxT), "layers": 12 if B < 4 else 2}
    if kind == "mlp":
        return {"kind": kind, "w": rng.choice(DTYPES), "B": B, "C": 64 * NH}
    # Logits: the padded vocabulary, or any other table (odd row counts among them).
    return {"kind": kind, "w": rng.choice(DTYPES), "B": B, "M": rng.choice((VOCAB, rng.randint(8000, VOCAB))),
            "K": 64 * min(NH, 12)}


# ------------------------------------------------------------------------------------
# Inputs.
# ------------------------------------------------------------------------------------
def _act(dtype):
    return torch.float32 if dtype == "f32" else torch.bfloat16


def _encode(values, dtype):
    """Rows of `values` (last dimension) in the storage type, and their scales (8-bit)."""
    if dtype in ("f32", "bf16"):
        return values.to(_act(dtype)), None
    limit = 127.0 if dtype == "int8" else 448.0
    scale = values.abs().amax(dim=-1) / limit
    y = values / scale.clamp_min(1e-30).unsqueeze(-1)
    if dtype == "int8":
        return y.round().clamp(-127, 127).to(torch.int8).view(torch.uint8), scale
    return y.to(torch.float8_e4m3fn).view(torch.uint8), scale


def _decode64(stored, scale, dtype):
    if dtype in ("f32", "bf16"):
        return stored.double()
    codes = stored.view(torch.int8) if dtype == "int8" else stored.view(torch.float8_e4m3fn).float()
    return codes.double() * scale.double().unsqueeze(-1)


class _Source:
    """N(0, 1) values of one seed, drawn in a fixed order."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def randn(self, *shape):
        return torch.randn(shape, generator=self.g, device="cuda")

    def lens(self, case):
        """int32 lengths minus one, one for the batch or one a sequence."""
        if case["lens"]:
            return torch.tensor([case["lens"] - 1], dtype=torch.int32, device="cuda")
        return torch.randint(0, case["maxT"], (case["B"],), generator=self.g, device="cuda", dtype=torch.int32)

    def cache(self, kv, B, NH, maxT):
        """A filled cache [2, B, NH, maxT, 64] and its row scales."""
        store = torch.uint8 if kv in ("int8", "fp8") else _act(kv)
        cache = torch.empty((2, B, NH, maxT, HD), dtype=store, device="cuda")
        scale = torch.empty((2, B, NH, maxT), device="cuda") if store == torch.uint8 else None
        for part in range(2):
            for b0 in range(0, B, 8):
                c, s = _encode(self.randn(min(8, B - b0), NH, maxT, HD), kv)
                cache[part, b0:b0 + 8] = c
                if scale is not None:
                    scale[part, b0:b0 + 8] = s
        return cache, scale

    def weight(self, w, M, K):
        """(stored weights [M, K], row scales or None)."""
        return _encode(self.randn(M, K) / math.sqrt(K), w)


def _inputs(case, seed):
    """What the call reads; the same for the library and for the 64-bit result."""
    src, kind = _Source(seed), case["kind"]
    if kind in ("stack", "attn"):
        B, NH, maxT, kv = case["B"], case["NH"], case["maxT"], case["kv"]
        layers = [dict(zip(("cache", "scale"), src.cache(kv, B, NH, maxT))) for _ in range(case.get("layers", 1))]
        for d in layers:
            d["qkv"] = src.randn(B, 3, NH, HD).to(_act(kv))
        return {"layers": layers, "cur": src.lens(case)}
    w, B = case["w"], case["B"]
    act = _act(w)
    if kind == "head":
        return {"W": src.weight(w, case["M"], case["K"]), "x": src.randn(B, case["K"]).to(act)}
    C = case["C"] if kind == "mlp" else case["NH"] * HD

    def proj(M, K):
        return {"W": src.weight(w, M, K), "bias": (0.1 * src.randn(M)).to(act)}

    layers = []
    for _ in range(case.get("layers", 1)):
        d = {"x2": src.randn(B, C).to(act), "fc": proj(4 * C, C), "fcproj": proj(C, 4 * C)}
        if kind == "step":
            d.update(x=src.randn(B, C).to(act), qkv=proj(3 * C, C), att=proj(C, C))
            d["cache"], d["scale"] = src.cache(case["kv"], B, case["NH"], case["maxT"])
        layers.append(d)
    return {"layers": layers, "cur": src.lens(case) if kind == "step" else None}


def _paged(cache, scale, page_rows, seed):
    """The same rows in a pool [pages, 2, NH, page_rows, 64] whose pages are shuffled."""
    _, B, NH, maxT, _ = cache.shape
    n = maxT // page_rows
    g = torch.Generator()
    g.manual_seed(seed)
    table = torch.randperm(B * n, generator=g).to(torch.int32).cuda()
    pool = torch.empty((B * n, 2, NH, page_rows, HD), dtype=cache.dtype, device="cuda")
    pool[table.long()] = cache.view(2, B, NH, n, page_rows, HD).permute(1, 3, 0, 2, 4, 5).reshape(pool.shape)
    pscale = None
    if scale is not None:
        pscale = torch.empty((B * n, 2, NH, page_rows), device="cuda")
        pscale[table.long()] = scale.view(2, B, NH, n, page_rows).permute(1, 3, 0, 2, 4).reshape(pscale.shape)
    return kvattn.PagedCache(pool, table.view(B, n), n, page_rows, B * n, pscale)


# ------------------------------------------------------------------------------------
# What a program keeps, and one pass.
# ------------------------------------------------------------------------------------
def _len_args(case, cur, hint):
    longest = case["lens"] - 1 if case["lens"] else case["maxT"] - 1
    return {"cur_len": cur, "lens_per_seq": not case["lens"], "len_hint": longest if hint else -1}


def _gemv(out, p, x, B, w, **kw):
    W, scale = p["W"]
    kvattn.gemv(out, W, x, B, W.shape[0], W.shape[1], w_dtype=w, w_scale=scale, bias=p.get("bias"), **kw)


def prepare(case, seed):
    kind, inp = case["kind"], _inputs(case, seed)
    s = {"case": case, "inp": inp}
    B = case["B"]
    if kind == "head":
        s["logits"] = torch.empty((B, case["M"]), device="cuda")
        return s
    L = len(inp["layers"])
    if kind in ("stack", "attn"):
        act = _act(case["kv"])
        s["out"] = torch.empty((L, B, case["NH"], HD), dtype=act, device="cuda")
        s["ws"] = kvattn.Workspace(B, case["NH"], case["maxT"])
        if case.get("page_rows"):
            d = inp["layers"][0]
            s["paged"] = _paged(d.pop("cache"), d.pop("scale"), case["page_rows"], seed)
    else:
        act, C = _act(case["w"]), inp["layers"][0]["x2"].shape[1]
        for name, width in (("pre", 4 * C), ("h", 4 * C), ("mlp", C)):
            s[name] = torch.empty((L, B, width), dtype=act, device="cuda")
    if kind == "step":
        NH = case["NH"]
        for name, width in (("qkv", 3 * C), ("att", C), ("proj", C)):
            s[name] = torch.empty((L, B, width), dtype=act, device="cuda")
        s["ws"] = kvattn.Workspace(B, NH, case["maxT"])
        n = kvattn.gemv_qkv_append_workspace_bytes(B, NH)
        s["qws"] = torch.empty(n, dtype=torch.uint8, device="cuda")
        kvattn.workspace_init(s["qws"], n)
    if kind in ("stack", "step"):
        # The step graph, captured once; every token replays it.
        s["graph"] = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(s["graph"]):
            _issue(s)
    return s


def _issue(s):
    """The library calls of one pass."""
    case, inp = s["case"], s["inp"]
    kind, B = case["kind"], case["B"]
    if kind == "head":
        _gemv(s["logits"], inp, inp["x"], B, case["w"], out_dtype="f32")
        return
    for i, d in enumerate(inp["layers"]):
        if kind in ("stack", "attn"):
            kw = dict(kv_dtype=case["kv"], **_len_args(case, inp["cur"], case["hint"]), **s["ws"].kwargs())
            if "paged" in s:
                kvattn.paged_decode(s["out"][i], d["qkv"], s["paged"], B, case["NH"], HD, append=case["append"], **kw)
                continue
            call = kvattn.append_decode if case["append"] else kvattn.decode
            call(s["out"][i], d["qkv"], d["cache"], B, case["NH"], HD, case["maxT"], kv_scale=d["scale"], **kw)
            continue
        w = case["w"]
        if kind == "step":
            NH, maxT = case["NH"], case["maxT"]
            lens = _len_args(case, inp["cur"], False)
            W, wscale = d["qkv"]["W"]
            kvattn.gemv_qkv_append(s["qkv"][i], W, d["x"], B, NH, HD, NH * HD, d["cache"], maxT, w_dtype=w,
                                   kv_dtype=case["kv"], w_scale=wscale, bias=d["qkv"]["bias"], kv_scale=d["scale"],
                                   cur_len=lens["cur_len"], lens_per_seq=lens["lens_per_seq"], workspace=s["qws"],
                                   workspace_nbytes=s["qws"].numel())
            kvattn.decode(s["att"][i], s["qkv"][i], d["cache"], B, NH, HD, maxT, kv_dtype=case["kv"],
                          kv_scale=d["scale"], **lens, **s["ws"].kwargs())
            _gemv(s["proj"][i], d["att"], s["att"][i], B, w)
        _gemv(s["h"][i], d["fc"], d["x2"], B, w, gelu=True, pre_gelu=s["pre"][i])
        _gemv(s["mlp"][i], d["fcproj"], s["h"][i], B, w)


def _caches(s):
    """The caches that the pass appends to."""
    case = s["case"]
    if case["kind"] not in ("stack", "attn", "step") or not case.get("append", True):
        return []
    if "paged" in s:
        held = [(s["paged"].pages, s["paged"].page_scales)]
    else:
        held = [(d["cache"], d["scale"]) for d in s["inp"]["layers"]]
    return [t for pair in held for t in pair if t is not None]


def run(s):
    if "graph" in s:
        s["graph"].replay()
    else:
        _issue(s)
    names = ("logits", "out", "qkv", "att", "proj", "pre", "h", "mlp")
    return {**{n: s[n] for n in names if n in s}, "caches": _caches(s)}


# ------------------------------------------------------------------------------------
# What a pass cannot do without, and how far a correct one may be off.
# ------------------------------------------------------------------------------------
def work(case):
    kind, B = case["kind"], case["B"]
    total = {"bytes": 0, "flops": 0}

    def proj(w, M, K, out):
        act = 4 if w == "f32" else 2
        total["bytes"] += M * K * W_BYTES[w] + (4 * M if W_BYTES[w] == 1 else 0) + act * (B * K + M) + out * B * M
        total["flops"] += 2 * B * M * K

    def attention(kv, NH):
        rows = B * NH * (case["lens"] or (case["maxT"] + 1) // 2)   # ragged: the mean
        act = 4 if kv == "f32" else 2
        new = 2 * B * NH * (HD * act + ROW_BYTES[kv]) if case.get("append", True) else 0
        total["bytes"] += 2 * rows * ROW_BYTES[kv] + 2 * B * NH * HD * act + new
        total["flops"] += 4 * rows * HD

    if kind == "head":
        proj(case["w"], case["M"], case["K"], 4)
        return total
    for _ in range(case.get("layers", 1)):
        if kind in ("stack", "attn"):
            attention(case["kv"], case["NH"])
            continue
        w, C = case["w"], case["C"] if kind == "mlp" else case["NH"] * HD
        act = 4 if w == "f32" else 2
        if kind == "step":
            proj(w, 3 * C, C, act)
            attention(case["kv"], case["NH"])
            proj(w, C, C, act)
        proj(w, 4 * C, C, 2 * act)
        proj(w, C, 4 * C, act)
    return total


def tolerance(case):
    """About four times what sums in another order (columns of every product permuted, another
    split of the attention) were seen to differ by over these ranges: 32-bit outputs by 2.4e-7
    (norm) and 1.4e-6 (largest); 16-bit ones by 2.2e-4 and 7.6e-3, where a value sits at a
    rounding boundary and, in a step, goes on through the attention and the projection behind
    it.  Such a value can also move an appended row's scale by one step, and with it its codes."""
    if case["kind"] == "head" or case.get("w", case.get("kv")) == "f32":
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 9e-4, "max": 3e-2, "differ": 1e-3}


# ------------------------------------------------------------------------------------
# The same in 64 bits, with torch alone.
# ------------------------------------------------------------------------------------
def _attend64(q, cache, scale, kv, cur, lens_per_seq, k_new=None, v_new=None):
    """Attention of q [B, NH, 64] over rows 0 .. cur of the cache; k_new, v_new [B, NH, 64]
    replace row cur."""
    B = q.shape[0]
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    last = cur.tolist()
    for b in range(B):
        n = last[b if lens_per_seq else 0] + 1
        k, v = (_decode64(cache[p, b, :, :n], None if scale is None else scale[p, b, :, :n], kv) for p in (0, 1))
        if k_new is not None:
            k[:, n - 1], v[:, n - 1] = k_new[b], v_new[b]
        p = torch.softmax(torch.einsum("hd,htd->ht", q[b], k) / math.sqrt(HD), dim=1)
        out[b] = torch.einsum("ht,htd->hd", p, v)
    return out


def _stored64(rows, kv):
    """Rows as the cache holds them once appended."""
    return _decode64(*_encode(rows.float(), kv), kv) if kv in ("int8", "fp8") else rows


def _linear64(p, x, w):
    W = _decode64(*p["W"], w)
    y = x @ W.t()
    return y + p["bias"].double() if "bias" in p else y


def _gelu64(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def exact(case, seed):
    kind, inp = case["kind"], _inputs(case, seed)
    if kind == "head":
        return {"logits": _linear64(inp, inp["x"].double(), case["w"])}
    got = {}

    def put(name, value):
        got.setdefault(name, []).append(value)

    for d in inp["layers"]:
        if kind in ("stack", "attn"):
            q, k, v = d["qkv"].double().unbind(1)
            new = [_stored64(t, case["kv"]) for t in (k, v)] if case["append"] else []
            put("out", _attend64(q, d["cache"], d["scale"], case["kv"], inp["cur"], not case["lens"], *new))
            continue
        w = case["w"]
        if kind == "step":
            B, NH, kv = case["B"], case["NH"], case["kv"]
            qkv = _linear64(d["qkv"], d["x"].double(), w)
            q, k, v = qkv.view(B, 3, NH, HD).unbind(1)
            att = _attend64(q, d["cache"], d["scale"], kv, inp["cur"], not case["lens"], _stored64(k, kv),
                            _stored64(v, kv)).reshape(B, -1)
            put("qkv", qkv)
            put("att", att)
            put("proj", _linear64(d["att"], att, w))
        pre = _linear64(d["fc"], d["x2"].double(), w)
        put("pre", pre)
        put("h", _gelu64(pre))
        put("mlp", _linear64(d["fcproj"], got["h"][-1], w))
    return {n: torch.stack(v) for n, v in got.items()}
