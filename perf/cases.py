"""The attention work whose speed this library is judged by, as its users run it on one MI355X.

Kinds (`"kind"` of a case):

* ``decode``  -- one token of a decode step: a hipGraph with the attention of `layers` layers, each
  WKB into Qcur then KQKV over that layer's own cache, replayed once per token as the engine does.
  The window `n_kv` is the allocated one; the keys from `live` on are masked (the engine pads its
  window), or, with `rows` > 1, the last `rows` tokens are checked together (drafted tokens: token t
  sees the keys before it and itself).
* ``batch``   -- the same graph for a batch of `rows` sequences of different lengths that share one
  window: sequence s owns the cells [s n_kv / rows, (s + 1) n_kv / rows) and fills a part of them.
* ``layer``   -- the reference geometry's whole attention layer for one token, every weight Q8_0:
  KV-write -> WKB -> concat -> KQKV -> wv_b, `layers` of them in one graph.
* ``chunk``   -- a chunk of a prompt: `rows` tokens after `cached` cached ones, causal, called
  eagerly (WKB, KQKV and, at the reference geometry with its Q8_0 weights, concat and wv_b).

Geometries: ``base`` (KV row 576 = 512 latent + 64 rope, f32 W_kb) and ``ref`` (KV row 320 = 256
latent + 64 rope, Q8_0 W_kb and wv_b).  Caches: f16, f32 and q8 (ggml's block_q8_0).  The latent
values, q and W_kb are scaled so that the scores have a standard deviation of about 1.7, as they
have behind a normalised latent and the 1 / sqrt(d) scale.
"""
import math

import torch

import aubier_amd as A

GEOM = {"base": dict(d_n=128, d_r=64, d_lat=512), "ref": dict(d_n=64, d_r=64, d_lat=256, n_embd=4096, d_out=128)}
ROPE = dict(freq_base=1e6, freq_scale=0.25, ext_factor=1.0, attn_factor=1.0, beta_fast=32.0, beta_slow=1.0,
            eps=1e-6, n_ctx_orig=8192)
ROW_BYTES = {"f32": lambda dk: 4 * dk, "f16": lambda dk: 2 * dk, "q8": lambda dk: dk // 32 * 34}


def _case(kind, name=None, **kw):
    c = {"kind": kind, "geom": "base", "cache": "f16", "heads": 32, "rows": 1, "layers": 1}
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the first tokens of a conversation: a 256-key window, f32 cache -- launches and latency
        _case("decode", "decode_f32_256", cache="f32", n_kv=256, live=219, layers=8),
        # an f32 cache (kept for its exactness) some thousand tokens into the conversation
        _case("decode", "decode_f32_4k", cache="f32", n_kv=4096, live=3901, layers=4),
        # ordinary chat context, f16 cache
        _case("decode", "decode_f16_4k", n_kv=4096, live=4001, layers=8),
        # long context, the headline decode step
        _case("decode", "decode_f16_32k", n_kv=32768, live=32768, layers=8),
        # the longest context supported, a ragged masked tail
        _case("decode", "decode_f16_256k", n_kv=262144, live=262007, layers=2),
        # the 8-bit cache at long context
        _case("decode", "decode_q8_32k", cache="q8", n_kv=32768, live=32701, layers=8),
        # four drafted tokens verified in one call at 16K keys
        _case("decode", "verify4_f16_16k", rows=4, n_kv=16384, live=16300, layers=4),
        # eight sequences decoded together, one window of per-sequence regions
        _case("batch", "batch8_f16_32k", rows=8, n_kv=32768, layers=4),
        # the reference's own layer, all five ops, one token
        _case("layer", "layer_ref_4k", geom="ref", n_kv=4096, live=4000, layers=8),
        # a prompt's first chunk: nothing cached, causal, an odd number of tokens
        _case("chunk", "first_chunk_1000", rows=1000, cached=0, n_kv=1024),
        # a later chunk of a long prompt
        _case("chunk", "chunk_512x8k", rows=512, cached=7680, n_kv=8192),
        # a prompt chunk at the reference geometry, Q8_0 weights around the attention
        _case("chunk", "chunk_ref_500x2k", geom="ref", rows=500, cached=1500, n_kv=2048),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _padded(rng, live, most):
    # engines pad the window to a multiple of 256 or 32, or not at all
    pad = rng.choice((256, 32, 1))
    return min(most, -(-live // pad) * pad)


def draw(rng):
    kind = rng.choice(("decode", "decode", "decode", "verify", "batch", "layer", "chunk", "chunk"))
    if kind == "decode":
        cache = rng.choice(("f16", "f16", "q8", "f32"))
        live = _log(rng, 40, 8192 if cache == "f32" else 262144)
        n_kv = _padded(rng, live, 8192 if cache == "f32" else 262144)
        heads = rng.choice((16, 32, 32, 40))
        return _case("decode", cache=cache, heads=heads, n_kv=n_kv, live=live, layers=2 if live > 20000 else 4)
    if kind == "verify":
        live = _log(rng, 300, 65536)
        return _case("decode", cache=rng.choice(("f16", "f16", "q8")), rows=rng.randint(2, 15), n_kv=_padded(rng, live, 65536),
                     live=live, layers=2)
    if kind == "batch":
        rows = rng.randint(2, 15)
        return _case("batch", cache=rng.choice(("f16", "q8")), rows=rows, n_kv=rows * _log(rng, 200, 16384), layers=2)
    if kind == "layer":
        live = _log(rng, 40, 32768)
        return _case("layer", geom="ref", n_kv=_padded(rng, live, 32768), live=live, layers=4)
    geom = rng.choice(("base", "base", "ref"))
    rows = _log(rng, 16, 1024)
    cached = rng.choice((0, _log(rng, 16, 6000)))
    while (cached + rows) * rows > 3_500_000:
        cached = int(cached * 0.7)
    return _case("chunk", geom=geom, cache="f16" if geom == "ref" else rng.choice(("f16", "f16", "q8")), rows=rows, cached=cached,
                 n_kv=_padded(rng, cached + rows, 8192))


# ------------------------------------------------------------------------------------ sizes
def _lens(case):
    """Keys each row sees, and where they start."""
    n, kind = case["rows"], case["kind"]
    if kind == "batch":
        region = case["n_kv"] // n
        return [(s * region, 1 + int((region - 1) * (0.25 + 0.75 * ((s + 1) * 0.6180339887 % 1.0)))) for s in range(n)]
    if kind == "chunk":
        return [(0, case["cached"] + t + 1) for t in range(n)]
    return [(0, max(1, case["live"] - n + t + 1)) for t in range(n)]


def work(case):
    g, H, n, L = GEOM[case["geom"]], case["heads"], case["rows"], case["layers"]
    d_n, d_v = g["d_n"], g["d_lat"]
    dk = d_v + g["d_r"]
    lens = _lens(case)
    pairs = sum(c for _, c in lens)
    keys = pairs if case["kind"] == "batch" else max(c for _, c in lens)
    q8w = case["geom"] == "ref"
    by = keys * ROW_BYTES[case["cache"]](dk) + 4 * (sum(c for _, c in lens))
    by += H * d_v * (d_n // 32 * 34 if q8w else 4 * d_n) + 4 * n * H * (d_n + g["d_r"] + 2 * dk + d_v)
    fl = 2 * H * pairs * (dk + d_v) + 2 * n * H * d_v * d_n
    if q8w:
        by += H * g["d_out"] * d_v // 32 * 34 + 4 * n * H * (d_v + g["d_out"])
        fl += 2 * n * H * d_v * g["d_out"]
    if case["kind"] == "layer":
        by += dk * g["n_embd"] // 32 * 34 + 4 * g["n_embd"] + 6 * dk
        fl += 2 * dk * g["n_embd"]
    return {"bytes": L * by, "flops": L * fl}


# What another correct implementation at the same precision may differ by: about four times this
# one's distance from 64-bit results (measured: f32 cache 4e-7; f16 and q8 caches 3.8e-4, q and P in
# f16; the reference geometry 2.4e-3, where a change below f16's resolution moves some of the
# activations' int8 quants by one).
def tolerance(case):
    if case["geom"] == "ref":
        return {"rel": 1e-2}
    return {"rel": 2e-6} if case["cache"] == "f32" else {"rel": 1.5e-3}


# ------------------------------------------------------------------------------------ inputs
def _randn(gen, shape, scale=1.0):
    return torch.randn(shape, generator=gen, device="cuda") * scale


def _q8_rows(x):
    """f32 [rows, ne0] -> ggml block_q8_0 bytes [rows, ne0 / 32 * 34]."""
    rows, ne0 = x.shape
    b = x.reshape(rows, ne0 // 32, 32)
    d = b.abs().amax(dim=2) / 127.0
    q = torch.round(b / torch.where(d > 0, d, torch.ones_like(d))[:, :, None]).to(torch.int8)
    out = torch.empty((rows, ne0 // 32, 34), dtype=torch.uint8, device=x.device)
    out[:, :, :2] = d.to(torch.float16).view(torch.uint8).reshape(rows, ne0 // 32, 2)
    out[:, :, 2:] = q.view(torch.uint8)
    return out.reshape(rows, ne0 // 32 * 34)


def _q8_values(blocks):
    """block_q8_0 bytes [..., nb * 34] -> the float64 values they stand for [..., nb * 32]."""
    b = blocks.reshape(*blocks.shape[:-1], blocks.shape[-1] // 34, 34)
    d = b[..., :2].contiguous().view(torch.float16).double()
    return (d * b[..., 2:].contiguous().view(torch.int8).double()).reshape(*blocks.shape[:-1], -1)


def _mask(case):
    m = torch.full((case["rows"], case["n_kv"]), -math.inf, device="cuda")
    for t, (first, count) in enumerate(_lens(case)):
        m[t, first:first + count] = 0.0
    return m


def _inputs(case, seed):
    """Every input tensor of the case, layer by layer."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    g, H, n, n_kv = GEOM[case["geom"]], case["heads"], case["rows"], case["n_kv"]
    d_n, d_r, d_v = g["d_n"], g["d_r"], g["d_lat"]
    dk = d_v + d_r
    mask = _mask(case)
    layers = []
    for _ in range(case["layers"]):
        s = {"mask": mask}
        kc = _randn(gen, (n_kv, dk))
        if case["cache"] == "q8":
            s["kc"] = A.Q8_0(_q8_rows(kc), dk)
        else:
            s["kc"] = kc.to(torch.float16) if case["cache"] == "f16" else kc
        s["q"] = _randn(gen, (n, H, d_n + d_r))
        w = _randn(gen, (H, d_v, d_n), 1.0 / math.sqrt(d_n))
        s["w_kb"] = A.Q8_0(_q8_rows(w.view(-1, d_n)).view(H, d_v, -1), d_n) if case["geom"] == "ref" else w
        if case["geom"] == "ref":
            wv = _randn(gen, (H * g["d_out"], d_v), 1.0 / math.sqrt(d_v))
            s["wv_b"] = A.Q8_0(_q8_rows(wv).view(H, g["d_out"], -1), d_v)
        if case["kind"] == "layer":
            s["cur"] = _randn(gen, (g["n_embd"],))
            s["wkv_a"] = A.Q8_0(_q8_rows(_randn(gen, (dk, g["n_embd"]), 1.0 / math.sqrt(g["n_embd"]))), g["n_embd"])
            s["kv_norm"] = 1.0 + _randn(gen, (d_v,), 0.25)
            s["kidx"] = torch.tensor([case["live"] - 1], dtype=torch.int64, device="cuda")
            s["pos"] = torch.tensor([case["live"] - 1], dtype=torch.int32, device="cuda")
        layers.append(s)
    return layers


def _layer(case, s, w):
    """One layer's calls, on buffers that the program keeps (`w`)."""
    g = GEOM[case["geom"]]
    d_n, d_v = g["d_n"], g["d_lat"]
    if case["kind"] == "layer":
        A.ggml_m4_phase_kvwrite(s["cur"], s["wkv_a"], s["kv_norm"], s["kc"], s["kidx"], s["pos"], w["rope"], out=w["kcur"])
    A.ggml_m4_wkb(s["w_kb"], s["q"][:, :, :d_n], out=w["qcur"][:, :, :d_v])
    if case["geom"] == "ref":
        w["qcur"][:, :, d_v:].copy_(s["q"][:, :, d_n:])
    A.ggml_m4_kqkv(s["kc"], w["qcur"], s["mask"], w["scale"], out=w["kqv"], workspace=w["ws"])
    if case["geom"] == "ref":
        A.ggml_m4_phase_wvb(s["wv_b"], w["kqv"], out=w["out"])


def prepare(case, seed):
    g, H, n = GEOM[case["geom"]], case["heads"], case["rows"]
    d_n, d_r, d_v = g["d_n"], g["d_r"], g["d_lat"]
    layers = _inputs(case, seed)
    ws, bufs = None, []
    for s in layers:
        w = {"scale": 1.0 / math.sqrt(d_n + d_r), "qcur": torch.zeros((n, H, d_v + d_r), device="cuda"),
             "kqv": torch.empty((H, n, d_v), device="cuda")}
        w["qcur"][:, :, d_v:] = s["q"][:, :, d_n:]
        if case["geom"] == "ref":
            w["out"] = torch.empty((H, n, g["d_out"]), device="cuda")
        if case["kind"] == "layer":
            w["kcur"] = torch.empty((d_v + d_r,), device="cuda")
            w["rope"] = A.rope_params(n_dims=d_r, **ROPE)
        if ws is None:      # one workspace, used by the layers in turn
            ws = torch.empty(max(16, A.kqkv_workspace_bytes(s["kc"], w["qcur"], w["kqv"])), dtype=torch.uint8, device="cuda")
        w["ws"] = ws
        bufs.append(w)
    state = {"case": case, "layers": layers, "bufs": bufs, "graph": None}
    state["outs"] = [_outs(case, s, w) for s, w in zip(layers, bufs)]
    if case["kind"] != "chunk":
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):       # the first call on a stream resolves what the library keeps for it
            for s, w in zip(layers, bufs):
                _layer(case, s, w)
        side.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"], stream=side):
            for s, w in zip(layers, bufs):
                _layer(case, s, w)
    return state


def _outs(case, s, w):
    if case["kind"] == "layer":
        return {"out": w["out"], "kcur": w["kcur"], "cache": s["kc"]}
    if case["geom"] == "ref":
        return {"out": w["out"], "kqv": w["kqv"], "qcur": w["qcur"]}
    return {"kqv": w["kqv"], "qcur": w["qcur"]}


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
    else:
        for s, w in zip(state["layers"], state["bufs"]):
            _layer(state["case"], s, w)
    return state["outs"]


# ------------------------------------------------------------------------------------ in 64 bits
def _round_away(x):
    return torch.sign(x) * torch.floor(x.abs() + 0.5)


def _q8_act(x):
    """The ops' own int8 activations (part of their result): per 32 values d = max / 127, its f16
    scale times round(x / d)."""
    b = x.double().reshape(*x.shape[:-1], x.shape[-1] // 32, 32)
    d = b.abs().amax(dim=-1, keepdim=True) / 127.0
    q = _round_away(b / torch.where(d > 0, d, torch.ones_like(d)))
    return (q * d.to(torch.float16).double()).reshape(x.shape)


def _kvwrite64(case, s):
    g = GEOM[case["geom"]]
    d_r, d_v = g["d_r"], g["d_lat"]
    row = _q8_values(s["wkv_a"].blocks) @ _q8_act(s["cur"])
    lat = row[:d_v] / torch.sqrt((row[:d_v] ** 2).mean() + ROPE["eps"]) * s["kv_norm"].double()
    p = torch.arange(d_r // 2, device="cuda", dtype=torch.float64)
    ext = (case["live"] - 1) * ROPE["freq_base"] ** (-2.0 * p / d_r)

    def corr(rot):
        return d_r * math.log(ROPE["n_ctx_orig"] / (rot * 2 * math.pi)) / (2 * math.log(ROPE["freq_base"]))

    lo, hi = max(0.0, math.floor(corr(ROPE["beta_fast"]))), min(d_r - 1.0, math.ceil(corr(ROPE["beta_slow"])))
    mix = (1.0 - torch.clamp((p - lo) / max(0.001, hi - lo), 0.0, 1.0)) * ROPE["ext_factor"]
    theta = ROPE["freq_scale"] * ext * (1.0 - mix) + ext * mix
    ms = ROPE["attn_factor"] * (1.0 + 0.1 * math.log(1.0 / ROPE["freq_scale"]))
    co, si = torch.cos(theta) * ms, torch.sin(theta) * ms
    x0, x1 = row[d_v::2], row[d_v + 1::2]
    return torch.cat([lat, torch.stack([x0 * co - x1 * si, x0 * si + x1 * co], dim=1).reshape(-1)])


def exact(case, seed):
    g, H, n = GEOM[case["geom"]], case["heads"], case["rows"]
    d_n, d_r, d_v = g["d_n"], g["d_r"], g["d_lat"]
    res = []
    for s in _inputs(case, seed):
        k = _q8_values(s["kc"].blocks) if case["cache"] == "q8" else s["kc"].double()
        kcur = None
        if case["kind"] == "layer":
            kcur = _kvwrite64(case, s)
            k[case["live"] - 1] = kcur
        q = s["q"].double()
        if case["geom"] == "ref":
            wkb, qn = _q8_values(s["w_kb"].blocks), _q8_act(s["q"][:, :, :d_n])
        else:
            wkb, qn = s["w_kb"].double(), q[:, :, :d_n]
        qcur = torch.empty((n, H, d_v + d_r), dtype=torch.float64, device="cuda")
        kqv = torch.empty((H, n, d_v), dtype=torch.float64, device="cuda")
        qcur[:, :, d_v:] = q[:, :, d_n:]
        kt = k.t().contiguous()
        for h in range(H):
            qcur[:, h, :d_v] = qn[:, h] @ wkb[h].t().contiguous()
            p = torch.softmax((qcur[:, h].contiguous() @ kt) / math.sqrt(d_n + d_r) + s["mask"].double(), dim=-1)
            kqv[h] = p @ k[:, :d_v].contiguous()
        r = {"kqv": kqv, "qcur": qcur}
        if case["geom"] == "ref":
            wv = _q8_values(s["wv_b"].blocks)
            r["out"] = torch.stack([_q8_act(kqv[h]) @ wv[h].t().contiguous() for h in range(H)])
        if case["kind"] == "layer":
            r = {"out": r["out"], "kcur": kcur, "cache": k}
        res.append(r)
    return res
