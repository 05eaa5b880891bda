"""What is timed of this framework, and how its results are checked.

Each case is one pass through the public entry points (vantablack_amd.hip and
vantablack_amd.layer), as a program that serves a model calls them:

  decode         one token's attention through n_layers layers of a KvCache:
                 the slot write, RoPE where "rope" says so, and attention
                 (layer_attention / layer_attention_rope)
  prefill        one layer's attention over a prompt or a chunk of one: the
                 K/V rows written at pos0, causal attention (prefill_attention)
  gemv           one decode token through `count` projections of one shape
                 (Segment.matmul_quant)
  matmul         one projection of a prompt's tokens (Segment.matmul_batched)
  token          one token through a whole model, embedding row to logits
                 (gpu_token_step)
  prefill_layer  one layer of a model over a prompt (gpu_prefill_layer)

Inputs are made on the device from the seed alone; `exact` computes the same
results with plain torch in 64 bits.
"""
import math

import numpy as np
import torch

DEV = "cuda"
KV_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
KV_BYTES = {"f32": 4, "f16": 2, "bf16": 2}
KINDS = ("q8_0", "q4_k", "q5_k", "q6_k")
BLOCK = {"q8_0": (34, 32), "q4_k": (144, 256), "q5_k": (176, 256), "q6_k": (210, 256)}


# ------------------------------------------------------------------- cases

def _decode(n_layers, heads, n_kv, d, kv, ctx, window=0, rope="none", outliers=False, **kw):
    return dict(op="decode", n_layers=n_layers, n_heads=heads, n_kv=n_kv, head_dim=d, kv=kv, ctx=ctx, window=window,
                rope=rope, outliers=outliers, **kw)


def _prefill(heads, n_kv, d, kv, tokens, pos0=0, window=0, **kw):
    return dict(op="prefill", n_heads=heads, n_kv=n_kv, head_dim=d, kv=kv, tokens=tokens, pos0=pos0, window=window,
                **kw)


def _gemv(kind, m, k, count, **kw):
    return dict(op="gemv", kind=kind, m=m, k=k, count=count, **kw)


def _matmul(kind, m, k, tokens, **kw):
    return dict(op="matmul", kind=kind, m=m, k=k, tokens=tokens, **kw)


def _model(op, heads, n_kv, d, ffn, kv, kind, kind_alt, rope, act, **kw):
    """kind: every projection but V and down, which are kind_alt (llama.cpp's
    mixed files keep those two, and the head, at more bits)."""
    return dict(op=op, n_heads=heads, n_kv=n_kv, head_dim=d, ffn=ffn, kv=kv, kind=kind, kind_alt=kind_alt, rope=rope,
                act=act, **kw)


def listed():
    return [
        # The smallest call there is: one layer's attention for one token of a
        # TinyLlama-1.1B-shaped model, 512 positions of the f32 cache that the
        # reference itself keeps.
        _decode(1, 32, 4, 64, "f32", 512, name="decode tiny f32 512"),
        # The headline workload: a token's attention through all layers of a
        # Llama-2-7B-shaped model (no GQA), f16 cache at 8192 positions.
        _decode(32, 32, 32, 128, "f16", 8192, rope="interleaved", name="decode mha f16 8k"),
        # Mistral-7B-shaped sliding window: the cache holds 16384 positions, the
        # last 4096 are attended; 1% of the K/V channels are outliers.
        _decode(32, 32, 8, 128, "bf16", 16384, window=4096, rope="interleaved", outliers=True,
                name="decode swa bf16 4k of 16k"),
        # Gemma-shaped long context: one KV head of 256, 32768 positions.
        _decode(26, 8, 1, 256, "bf16", 32768, rope="half", name="decode mqa d256 bf16 32k"),
        # A long prompt of a Llama-3-8B-shaped model.
        _prefill(32, 8, 128, "bf16", 8192, name="prefill gqa bf16 8k"),
        # The second, ragged chunk of a Gemma-shaped prompt.
        _prefill(8, 1, 256, "f16", 2101, pos0=1995, name="prefill d256 f16 chunk"),
        # A short prompt on the reference's own f32 cache, TinyLlama-shaped.
        _prefill(32, 4, 64, "f32", 512, name="prefill tiny f32 512"),
        # Decode-time down projections of eight layers, 6-bit weights.
        _gemv("q6_k", 4096, 11008, 8, name="gemv q6_k down x8"),
        # The largest projection of a Llama-3-8B-shaped model over a prompt.
        _matmul("q4_k", 14336, 4096, 2048, name="matmul q4_k gate 2048"),
        # The tail of a chunked prompt: 33 tokens, 8-bit weights.
        _matmul("q8_0", 4096, 4096, 33, name="matmul q8_0 33 tokens"),
        # A whole decode step, TinyLlama-1.1B-shaped, mixed 4/6-bit weights.
        _model("token", 32, 4, 64, 5632, "f16", "q4_k", "q6_k", "interleaved", "silu", n_layers=22, vocab=32000,
               kind_out="q6_k", ctx=1024, name="token tiny q4_k"),
        # One whole layer of a Llama-3-8B-shaped model over a prompt.
        _model("prefill_layer", 32, 8, 128, 14336, "bf16", "q4_k", "q4_k", "half", "silu", tokens=2048, pos0=0,
               name="prefill layer 8b 2048"),
    ]


HEADS = ((32, 4, 64), (32, 32, 128), (32, 8, 128), (8, 1, 256), (16, 16, 64), (12, 4, 128), (24, 3, 64), (8, 4, 256),
         (7, 1, 128), (40, 10, 128))


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(("decode", "decode", "prefill", "prefill", "gemv", "matmul", "matmul", "token", "prefill_layer"))
    if op == "decode":
        heads, n_kv, d = rng.choice(HEADS)
        kv = rng.choice(("f32", "f16", "bf16"))
        ctx = _log(rng, 64, 32768)
        window = _log(rng, 64, 4096) if rng.random() < 0.3 else 0
        row = 2 * n_kv * d * KV_BYTES[kv]
        # no more than the headline workload's bytes, held or attended
        most = max(1, (4 << 30) // (ctx * row))
        return _decode(_log(rng, 1, min(32, most)), heads, n_kv, d, kv, ctx, window,
                       rng.choice(("none", "interleaved", "half")), rng.random() < 0.25)
    if op == "prefill":
        heads, n_kv, d = rng.choice(HEADS)
        kv = rng.choice(("f32", "f16", "bf16", "bf16"))
        tokens = _log(rng, 16, 768 if kv == "f32" else 8192)
        pos0 = _log(rng, 1, 512 if kv == "f32" else 4096) if rng.random() < 0.4 else 0
        window = _log(rng, 64, 4096) if rng.random() < 0.25 else 0
        c = _prefill(heads, n_kv, d, kv, tokens, pos0, window)
        while c["tokens"] > 16 and work(c)["flops"] > 5.4e11:
            c["tokens"] -= c["tokens"] // 4
        return c
    if op == "gemv":
        kind = rng.choice(KINDS)
        k = 256 * _log(rng, 4, 56)
        m = _log(rng, 256, 32768)
        return _gemv(kind, m, k, max(1, min(8, (512 << 20) // (m * k))))
    if op == "matmul":
        return _matmul(rng.choice(KINDS), _log(rng, 256, 14336), 256 * _log(rng, 4, 56 if rng.random() < 0.3 else 16),
                       _log(rng, 2, 2048))
    heads, n_kv, d = rng.choice(((32, 4, 64), (16, 16, 64), (32, 8, 128), (16, 4, 128), (8, 1, 256), (24, 8, 64)))
    kind = rng.choice(KINDS)
    alt = rng.choice((kind, "q6_k"))
    ffn = 256 * rng.randint(2 * heads * d // 256, 7 * heads * d // 512)
    common = (heads, n_kv, d, ffn, rng.choice(("f32", "f16", "bf16")), kind, alt,
              rng.choice(("interleaved", "half")), rng.choice(("silu", "silu", "gelu_approx")))
    if op == "token":
        return _model("token", *common, n_layers=rng.randint(2, 6), vocab=rng.randint(4000, 32000), kind_out="q6_k",
                      ctx=_log(rng, 16, 4096))
    f32 = common[4] == "f32"
    return _model("prefill_layer", *common, tokens=_log(rng, 16, 512 if f32 else 1536),
                  pos0=_log(rng, 1, 300) if rng.random() < 0.3 else 0)


# ---------------------------------------------------- quantised weights (GGUF)

def _quant(kind, m, k, g):
    """m rows of k weights as GGUF blocks (uint8 [m * bytes per row]) whose
    values have a standard deviation of about 1 / sqrt(k)."""
    bb, be = BLOCK[kind]
    n = m * (k // be)
    w = torch.randint(0, 256, (n, bb), generator=g, device=DEV, dtype=torch.uint8)
    spread = 0.5 + torch.rand(n, generator=g, device=DEV)

    def put(off, v):
        w[:, off:off + 2] = v.to(torch.float16).view(torch.uint8).reshape(n, 2)

    std = 1.0 / math.sqrt(k)
    if kind == "q8_0":
        w[:, 2:][w[:, 2:] == 128] = 127  # quantisers write -127..127
        put(0, std / 73.0 * spread)
    elif kind == "q6_k":
        sc = torch.randint(32, 128, (n, 16), generator=g, device=DEV)
        sc = torch.where(torch.rand(n, 16, generator=g, device=DEV) < 0.5, sc, -sc)
        w[:, 192:208] = sc.to(torch.int8).view(torch.uint8)
        put(208, std / (84.0 * 18.5) * spread)
    else:
        # eight 6-bit scales and mins; the mins centre the quants
        sc = torch.randint(16, 64, (n, 8), generator=g, device=DEV)
        mn = (sc + torch.randint(-3, 4, (n, 8), generator=g, device=DEV)).clamp(0, 63)
        w[:, 4:8] = (sc[:, :4] | (sc[:, 4:] >> 4) << 6).to(torch.uint8)
        w[:, 8:12] = (mn[:, :4] | (mn[:, 4:] >> 4) << 6).to(torch.uint8)
        w[:, 12:16] = ((sc[:, 4:] & 15) | (mn[:, 4:] & 15) << 4).to(torch.uint8)
        levels = 16 if kind == "q4_k" else 32
        d = std / (42.0 * levels / math.sqrt(12.0)) * spread
        put(0, d)
        put(2, d * (levels - 1) / 2)
    return w.reshape(-1)


def _dequant(kind, w, m, k):
    """The weights of _quant's blocks, float64 [m, k]."""
    bb, be = BLOCK[kind]
    b = w.reshape(-1, bb)
    n = b.shape[0]

    def half(off):
        return b[:, off:off + 2].contiguous().view(torch.float16).double()

    if kind == "q8_0":
        v = half(0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif kind == "q6_k":
        ql, qh = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 1, 32)
        q = torch.cat((ql & 15, ql >> 4), 2)  # [n, half, quadrant, 32]
        shift = torch.tensor([0, 2, 4, 6], device=DEV, dtype=torch.uint8).reshape(1, 1, 4, 1)
        q = (q | ((qh >> shift) & 3) << 4).double() - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).double().reshape(n, 2, 4, 2, 1)
        v = half(208).reshape(n, 1, 1, 1, 1) * sc * q.reshape(n, 2, 4, 2, 16)
    else:
        s = b[:, 4:16]
        sc = torch.cat((s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6) << 4), 1).double()
        mn = torch.cat((s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6) << 4), 1).double()
        qs = b[:, -128:].reshape(n, 4, 1, 32)
        q = torch.cat((qs & 15, qs >> 4), 2).reshape(n, 8, 32)
        if kind == "q5_k":
            shift = torch.arange(8, device=DEV, dtype=torch.uint8).reshape(1, 8, 1)
            q = q | ((b[:, 16:48].reshape(n, 1, 32) >> shift) & 1) << 4
        v = (half(0) * sc).unsqueeze(2) * q.double() - (half(2) * mn).unsqueeze(2)
    return v.reshape(m, k)


def _wbytes(kind, m, k):
    bb, be = BLOCK[kind]
    return m * (k // be) * bb


# ------------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _projections(c):
    dim, kv_dim, ffn = c["n_heads"] * c["head_dim"], c["n_kv"] * c["head_dim"], c["ffn"]
    a, b = c["kind"], c["kind_alt"]
    return (("q", a, dim, dim), ("k", a, kv_dim, dim), ("v", b, kv_dim, dim), ("o", a, dim, dim),
            ("gate", a, ffn, dim), ("up", a, ffn, dim), ("down", b, dim, ffn))


def _layer_weights(c, g):
    dim = c["n_heads"] * c["head_dim"]
    t = {"attn_norm": 1.0 + 0.1 * _randn(g, dim), "ffn_norm": 1.0 + 0.1 * _randn(g, dim)}
    for name, kind, m, k in _projections(c):
        t[name] = _quant(kind, m, k, g)
    return t


def _inputs(c, seed):
    """The inputs as plain tensors on the device."""
    g = _gen(seed)
    if c["op"] == "decode":
        q_dim, kv_dim, pos = c["n_heads"] * c["head_dim"], c["n_kv"] * c["head_dim"], c["ctx"] - 1
        i = {}
        gain = torch.ones(kv_dim, device=DEV)
        if c["outliers"]:
            gain[torch.rand(kv_dim, generator=g, device=DEV) < 0.01] = 20.0
        for n in ("k", "v"):
            i[n] = torch.empty(c["n_layers"], pos, kv_dim, dtype=KV_TORCH[c["kv"]], device=DEV)
            for layer in range(c["n_layers"]):
                i[n][layer] = _randn(g, pos, kv_dim) * gain
            i[n + "_cur"] = _randn(g, c["n_layers"], kv_dim) * gain
        i["q"] = _randn(g, c["n_layers"], q_dim) / math.sqrt(c["head_dim"])
        return i
    if c["op"] == "prefill":
        q_dim, kv_dim = c["n_heads"] * c["head_dim"], c["n_kv"] * c["head_dim"]
        i = {"q": _randn(g, c["tokens"], q_dim)}
        for n in ("k", "v"):
            i[n] = _randn(g, c["pos0"], kv_dim).to(KV_TORCH[c["kv"]])
            i[n + "_cur"] = _randn(g, c["tokens"], kv_dim)
        return i
    if c["op"] == "gemv":
        return {"w": [_quant(c["kind"], c["m"], c["k"], g) for _ in range(c["count"])],
                "x": _randn(g, c["count"], c["k"])}
    if c["op"] == "matmul":
        return {"w": _quant(c["kind"], c["m"], c["k"], g), "x": _randn(g, c["tokens"], c["k"])}
    dim, kv_dim = c["n_heads"] * c["head_dim"], c["n_kv"] * c["head_dim"]
    n_layers = c.get("n_layers", 1)
    rows = c["ctx"] - 1 if c["op"] == "token" else c["pos0"]
    i = {"layers": [_layer_weights(c, g) for _ in range(n_layers)]}
    for n in ("k", "v"):
        i[n] = _randn(g, n_layers, rows, kv_dim).to(KV_TORCH[c["kv"]])
    if c["op"] == "token":
        i["out_norm"] = 1.0 + 0.1 * _randn(g, dim)
        i["out"] = _quant(c["kind_out"], c["vocab"], dim, g)
        i["x"] = _randn(g, dim)
    else:
        i["x"] = _randn(g, c["tokens"], dim)
    return i


# ------------------------------------------------------------------ the passes

_context = None


def _ctx():
    """The one context that a serving program opens when it starts."""
    global _context
    if _context is None:
        import vantablack_amd as vb
        _context = vb.Context()
    return _context


class _Slab:
    """A view of a KvCache slab for torch; keeps the cache alive."""

    def __init__(self, cache, which):
        self.cache = cache
        ts = {4: "<f4", 2: "<i2"}[cache.elem_bytes]
        self.__cuda_array_interface__ = {"shape": (cache.n_layers, cache.max_seq, cache.row_elems), "typestr": ts,
                                         "data": (getattr(cache, which).ptr, False), "version": 2}


def _slab(cache, which, kv):
    t = torch.as_tensor(_Slab(cache, which), device=DEV)
    return t if kv == "f32" else t.view(KV_TORCH[kv])


def _rows(t):
    """A buffer handle for each row of t (its rows are 16-byte aligned)."""
    ctx = _ctx()
    n = t[0].numel() * t.element_size()
    return [ctx.wrap(t[r].data_ptr(), n, keepalive=t) for r in range(t.shape[0])]


def _cache(c, i, max_seq, n_layers, pos):
    from vantablack_amd import hip
    cfg = hip.LlamaConfig(c["n_heads"], c["n_kv"], c["head_dim"], max_seq,
                          c["window"] if c["window"] else hip.NO_WINDOW, rope_half=c.get("rope") == "half")
    cache = hip.KvCache(_ctx(), n_layers, c["n_kv"], c["head_dim"], max_seq, c["kv"])
    k, v = _slab(cache, "k", c["kv"]), _slab(cache, "v", c["kv"])
    k[:, :pos].copy_(i["k"])
    v[:, :pos].copy_(i["v"])
    cache.pos = pos
    return cfg, cache, k, v


def _model_state(c, i):
    """The weights in one buffer with their offsets, as the framework's layer
    functions address them, and the K/V slabs."""
    from vantablack_amd import hip
    from vantablack_amd.layer import LayerConfig, LayerOffsets
    ctx = _ctx()
    parts, at = [], 0

    def add(t):
        nonlocal at
        b = t.contiguous().view(torch.uint8).reshape(-1)
        parts.append((at, b))
        off, at = at, (at + b.numel() + 255) // 256 * 256
        return off

    kinds = {"kind_" + n: kind for n, kind, _, _ in _projections(c)}
    offs = []
    for w in i["layers"]:
        o = {n: add(w[n]) for n in ("attn_norm", "ffn_norm")}
        o.update({"w" + n: add(w[n]) for n, _, _, _ in _projections(c)})
        offs.append(LayerOffsets(**o, **kinds))
    out_norm, out = (add(i["out_norm"]), add(i["out"])) if "out" in i else (0, 0)
    blob = torch.zeros(at, dtype=torch.uint8, device=DEV)
    for off, b in parts:
        blob[off:off + b.numel()] = b
    rows = c["ctx"] - 1 if c["op"] == "token" else c["pos0"]
    max_seq = rows + c.get("tokens", 1) + 64
    lc = LayerConfig(c["n_heads"] * c["head_dim"], c["n_heads"], c["n_kv"], c["head_dim"], c["ffn"], max_seq,
                     rope_half=c["rope"] == "half", activation=c["act"], kv_dtype=hip.DTYPES[c["kv"]])
    kv = {}
    for n in ("k", "v"):
        kv[n] = torch.zeros(len(offs), max_seq, c["n_kv"] * c["head_dim"], dtype=KV_TORCH[c["kv"]], device=DEV)
        kv[n][:, :rows] = i[n]
    return {"lc": lc, "offs": offs, "out_norm": out_norm, "out": out, "pos": rows, "weights": ctx.wrap_tensor(blob),
            "kt": kv["k"], "vt": kv["v"], "k": ctx.wrap_tensor(kv["k"]), "v": ctx.wrap_tensor(kv["v"]),
            "embed": ctx.wrap_tensor(i["x"])}


def prepare(case, seed):
    from vantablack_amd import layer
    c, ctx = case, _ctx()
    i = _inputs(c, seed)
    s = {"case": c}
    if c["op"] == "decode":
        pos = c["ctx"] - 1
        s["cfg"], s["cache"], k, v = _cache(c, i, c["ctx"] + 8, c["n_layers"], pos)
        s["out"] = torch.zeros_like(i["q"])
        s["io"] = list(zip(_rows(i["q"]), _rows(i["k_cur"]), _rows(i["v_cur"]), _rows(s["out"])))
        s["k_row"], s["v_row"] = k[:, pos], v[:, pos]
    elif c["op"] == "prefill":
        end = c["pos0"] + c["tokens"]
        s["cfg"], s["cache"], k, v = _cache(c, i, end + 64, 1, c["pos0"])
        s["out"] = torch.zeros_like(i["q"])
        s["io"] = [ctx.wrap_tensor(t) for t in (i["q"], i["k_cur"], i["v_cur"], s["out"])]
        s["k_rows"], s["v_rows"] = k[0, c["pos0"]:end], v[0, c["pos0"]:end]
    elif c["op"] == "gemv":
        s["w"] = [ctx.wrap_tensor(w) for w in i["w"]]
        s["x"] = _rows(i["x"])
        s["out"] = [torch.zeros(c["m"], device=DEV) for _ in i["w"]]
        s["ob"] = [ctx.wrap_tensor(t) for t in s["out"]]
    elif c["op"] == "matmul":
        s["w"], s["x"] = ctx.wrap_tensor(i["w"]), ctx.wrap_tensor(i["x"])
        s["out"] = torch.zeros(c["tokens"], c["m"], device=DEV)
        s["ob"] = ctx.wrap_tensor(s["out"])
    elif c["op"] == "token":
        s.update(_model_state(c, i))
        s["scratch"] = layer.LayerScratch(ctx, s["lc"])
        s["logits"] = torch.zeros(c["vocab"], device=DEV)
        s["scratch"].logits = ctx.wrap_tensor(s["logits"])
    else:
        s.update(_model_state(c, i))
        s["scratch"] = layer.PrefillScratch(ctx, s["lc"], c["tokens"])
        s["x"] = torch.zeros_like(i["x"])
        s["scratch"].x.release()
        s["scratch"].x = ctx.wrap_tensor(s["x"])
    torch.cuda.synchronize()
    return s


def run(state):
    from vantablack_amd import hip, layer
    s, c = state, state["case"]
    seg = _ctx().segment()
    if c["op"] == "decode":
        attend = hip.layer_attention if c["rope"] == "none" else hip.layer_attention_rope
        for n, (q, k_cur, v_cur, out) in enumerate(s["io"]):
            attend(seg, s["cache"], s["cfg"], n, q, k_cur, v_cur, out)
        seg.commit()
        return {"out": s["out"], "k": s["k_row"], "v": s["v_row"]}
    if c["op"] == "prefill":
        q, k_cur, v_cur, out = s["io"]
        hip.prefill_attention(seg, s["cache"], s["cfg"], 0, c["tokens"], q, k_cur, v_cur, out)
        seg.commit()
        return {"out": s["out"], "k": s["k_rows"], "v": s["v_rows"]}
    if c["op"] == "gemv":
        for w, x, o in zip(s["w"], s["x"], s["ob"]):
            seg.matmul_quant(c["kind"], o, w, 0, x, c["m"], c["k"])
        seg.commit()
        return s["out"]
    if c["op"] == "matmul":
        seg.matmul_batched(c["kind"], s["ob"], s["w"], 0, s["x"], c["m"], c["k"], c["tokens"])
        seg.commit()
        return s["out"]
    sc, lc, pos = s["scratch"], s["lc"], s["pos"]
    if c["op"] == "token":
        seg.copy(sc.x, 0, s["embed"], 0, lc.dim)
        layer.gpu_token_step(seg, sc, s["weights"], s["offs"], s["k"], s["v"], lc, pos, s["out_norm"], s["out"],
                             c["kind_out"], c["vocab"])
        seg.commit()
        return {"logits": s["logits"], "k": s["kt"][:, pos], "v": s["vt"][:, pos]}
    seg.copy(sc.x, 0, s["embed"], 0, c["tokens"] * lc.dim)
    layer.gpu_prefill_layer(seg, sc, s["weights"], s["offs"][0], s["k"], s["v"], lc, 0, pos)
    seg.commit()
    end = pos + c["tokens"]
    return {"x": s["x"], "k": s["kt"][0, pos:end], "v": s["vt"][0, pos:end]}


# ----------------------------------------------------------- the work of a pass

def _pairs(tokens, pos0, window):
    """Attended (query, key) pairs."""
    if not window:
        return tokens * pos0 + tokens * (tokens + 1) // 2
    return sum(min(pos0 + b + 1, window) for b in range(tokens))


def work(case):
    c = case
    if c["op"] == "decode":
        n, q_dim, kv_dim, eb = c["n_layers"], c["n_heads"] * c["head_dim"], c["n_kv"] * c["head_dim"], KV_BYTES[c["kv"]]
        rows = min(c["ctx"], c["window"]) if c["window"] else c["ctx"]
        return {"bytes": n * (2 * rows * kv_dim * eb + 8 * kv_dim + 8 * q_dim), "flops": n * 4 * q_dim * rows}
    if c["op"] == "prefill":
        q_dim, kv_dim, eb = c["n_heads"] * c["head_dim"], c["n_kv"] * c["head_dim"], KV_BYTES[c["kv"]]
        old = min(c["pos0"], c["window"]) if c["window"] else c["pos0"]
        return {"bytes": 2 * old * kv_dim * eb + c["tokens"] * (8 * q_dim + kv_dim * (8 + 2 * eb)),
                "flops": 4 * q_dim * _pairs(c["tokens"], c["pos0"], c["window"])}
    if c["op"] == "gemv":
        return {"bytes": c["count"] * (_wbytes(c["kind"], c["m"], c["k"]) + 4 * (c["m"] + c["k"])),
                "flops": c["count"] * 2 * c["m"] * c["k"]}
    if c["op"] == "matmul":
        return {"bytes": _wbytes(c["kind"], c["m"], c["k"]) + 4 * c["tokens"] * (c["m"] + c["k"]),
                "flops": 2 * c["m"] * c["k"] * c["tokens"]}
    tokens = c.get("tokens", 1)
    n = c.get("n_layers", 1)
    pos0 = c["ctx"] - 1 if c["op"] == "token" else c["pos0"]
    dim, kv_dim, eb = c["n_heads"] * c["head_dim"], c["n_kv"] * c["head_dim"], KV_BYTES[c["kv"]]
    by = n * (sum(_wbytes(kind, m, k) for _, kind, m, k in _projections(c)) + 8 * dim +
              2 * (pos0 + tokens) * kv_dim * eb) + 8 * tokens * dim
    fl = n * (2 * tokens * sum(m * k for _, _, m, k in _projections(c)) + 4 * dim * _pairs(tokens, pos0, 0))
    if c["op"] == "token":
        by += _wbytes(c["kind_out"], c["vocab"], dim) + 4 * c["vocab"]
        fl += 2 * c["vocab"] * dim
    return {"bytes": by, "flops": fl}


# ------------------------------------------------------------- 64-bit results

def _angles(c, positions, base=10000.0):
    """Angles as the model defines them: 32-bit frequencies 1 / base^(2j/d)
    times the position, one 32-bit product."""
    d = c["head_dim"]
    f = np.float32(1) / np.power(np.float32(base), np.arange(0, d, 2, dtype=np.float32) / np.float32(d))
    f = torch.from_numpy(f.astype(np.float32)).to(DEV)
    return (torch.as_tensor(positions, device=DEV, dtype=torch.float32).unsqueeze(1) * f).double()


def _rotate(c, x, positions):
    """RoPE of x [rows, heads * head_dim], row r at positions[r]."""
    if c["rope"] == "none":
        return x
    d = c["head_dim"]
    y = x.reshape(x.shape[0], -1, d)
    t = _angles(c, positions).unsqueeze(1)
    cs, sn = torch.cos(t), torch.sin(t)
    if c["rope"] == "half":
        a, b = y[..., :d // 2], y[..., d // 2:]
        y = torch.cat((a * cs - b * sn, a * sn + b * cs), -1)
    else:
        a, b = y[..., 0::2], y[..., 1::2]
        y = torch.stack((a * cs - b * sn, a * sn + b * cs), -1)
    return y.reshape(x.shape)


def _attend(c, q, k, v, pos0, window):
    """Causal attention of q [n, heads * d] (row r at pos0 + r) over the rows of
    k, v [pos0 + n, n_kv * d], all float64."""
    n, d, heads, n_kv = q.shape[0], c["head_dim"], c["n_heads"], c["n_kv"]
    lo = max(0, pos0 - window + 1) if window else 0
    out = torch.empty_like(q)
    at = torch.arange(pos0, pos0 + n, device=DEV).unsqueeze(1)
    key = torch.arange(lo, pos0 + n, device=DEV).unsqueeze(0)
    drop = key > at
    if window:
        drop |= key <= at - window
    for h in range(heads):
        j = h * n_kv // heads
        kh, vh = (t[lo:, j * d:(j + 1) * d].contiguous() for t in (k, v))
        s = q[:, h * d:(h + 1) * d] @ kh.t().contiguous() / math.sqrt(d)
        s.masked_fill_(drop, -math.inf)
        out[:, h * d:(h + 1) * d] = torch.softmax(s, 1) @ vh
    return out


def _norm(x, w, eps=1e-5):
    return x * w.double() / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)


def _exact_layer(c, w, k, v, x, pos0):
    """One layer over x [n, dim] at pos0 ..; the new K/V rows come back rounded
    to the cache's type."""
    kv = KV_TORCH[c["kv"]]
    shape = {n: (kind, m, kk) for n, kind, m, kk in _projections(c)}

    def proj(n, t):
        return t @ _dequant(shape[n][0], w[n], *shape[n][1:]).t()

    at = range(pos0, pos0 + x.shape[0])
    xb = _norm(x, w["attn_norm"])
    q = _rotate(c, proj("q", xb), at)
    kr, vr = _rotate(c, proj("k", xb), at).to(kv), proj("v", xb).to(kv)
    a = _attend(c, q, torch.cat((k.double(), kr.double())), torch.cat((v.double(), vr.double())), pos0, 0)
    x = x + proj("o", a)
    xb = _norm(x, w["ffn_norm"])
    gate, up = proj("gate", xb), proj("up", xb)
    if c["act"] == "silu":
        h = gate * torch.sigmoid(gate) * up
    else:
        h = 0.5 * gate * (1 + torch.tanh(math.sqrt(2 / math.pi) * (gate + 0.044715 * gate ** 3))) * up
    return x + proj("down", h), kr, vr


def exact(case, seed):
    c = case
    i = _inputs(c, seed)
    kv = KV_TORCH.get(c.get("kv"))
    if c["op"] == "decode":
        pos = c["ctx"] - 1
        outs, ks, vs = [], [], []
        for n in range(c["n_layers"]):
            q = _rotate(c, i["q"][n:n + 1].double(), [pos])
            kr, vr = _rotate(c, i["k_cur"][n:n + 1].double(), [pos]).to(kv), i["v_cur"][n:n + 1].to(kv)
            k, v = (torch.cat((t, r)).double() for t, r in ((i["k"][n], kr), (i["v"][n], vr)))
            outs.append(_attend(c, q, k, v, pos, c["window"])[0])
            ks.append(kr[0])
            vs.append(vr[0])
        return {"out": torch.stack(outs), "k": torch.stack(ks), "v": torch.stack(vs)}
    if c["op"] == "prefill":
        kr, vr = i["k_cur"].to(kv), i["v_cur"].to(kv)
        k, v = (torch.cat((t, r)).double() for t, r in ((i["k"], kr), (i["v"], vr)))
        return {"out": _attend(c, i["q"].double(), k, v, c["pos0"], c["window"]), "k": kr, "v": vr}
    if c["op"] == "gemv":
        return [_dequant(c["kind"], w, c["m"], c["k"]) @ x.double() for w, x in zip(i["w"], i["x"])]
    if c["op"] == "matmul":
        return i["x"].double() @ _dequant(c["kind"], i["w"], c["m"], c["k"]).t()
    if c["op"] == "token":
        x, ks, vs = i["x"].double().unsqueeze(0), [], []
        for n, w in enumerate(i["layers"]):
            x, kr, vr = _exact_layer(c, w, i["k"][n], i["v"][n], x, c["ctx"] - 1)
            ks.append(kr[0])
            vs.append(vr[0])
        x = _norm(x, i["out_norm"])
        logits = x[0] @ _dequant(c["kind_out"], i["out"], c["vocab"], x.shape[1]).t()
        return {"logits": logits, "k": torch.stack(ks), "v": torch.stack(vs)}
    x, kr, vr = _exact_layer(c, i["layers"][0], i["k"][0], i["v"][0], i["x"].double(), c["pos0"])
    return {"x": x, "k": kr, "v": vr}


def tolerance(case):
    """About four times the distance from 64 bits that each path shows: sums of
    32 bits (1e-7 to 5e-7), f16 products in a prompt's attention (3e-4), and
    where rows rotated or projected on the way are stored in 16 bits, single
    values that round to the neighbour (at most 7e-5 f16, 6e-4 bf16 of a row's
    norm; half a unit in the last place of the value itself)."""
    c = case
    stored = {"f32": {"rel": 1e-5, "max": 2e-4}, "f16": {"rel": 3e-4, "max": 5e-3}, "bf16": {"rel": 2e-3, "max": 2e-2}}
    if c["op"] == "decode":
        return {"rel": 1e-6, "max": 2e-5} if c["rope"] == "none" else stored[c["kv"]]
    if c["op"] == "prefill":
        return {"rel": 1e-6, "max": 2e-5} if c["kv"] == "f32" else {"rel": 1.2e-3, "max": 2e-2}
    if c["op"] in ("gemv", "matmul"):
        return {"rel": 2e-6, "max": 4e-5}
    if c["op"] == "prefill_layer" and c["kv"] != "f32":
        return {"rel": 2e-3, "max": 2e-2}
    return stored[c["kv"]]
