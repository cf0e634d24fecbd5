"""Cases that stand for the work this library does for its users, for timing and comparing.

One generation step of a causal-chunk video DiT calls, per layer: the fused q/k norm + RoPE (and
K/V commit), the chunk's self-attention over the KV cache, and the cross-attention to the text
context; the fp8 cache adds its quantiser. Each is a case through its own entry point, at the
sizes of the 1.3B (12 heads x 128) and 14B (40 heads x 128) models: 1560 tokens per latent frame
at 480p (30 x 52), 3600 at 720p (45 x 80), 1 or 3 frames per chunk. One whole layer is there too.

listed() names them, draw() gives more of the same ranges (odd and ragged sizes, other head
counts as a tensor-parallel rank has them, windows, segments, both pairings of q's scale).
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "lingbot-world-v2_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import lbw_amd  # noqa: E402

D = 128
EPS = 1e-6
BF16 = torch.bfloat16


def listed():
    return [
        # the smallest chunk call: 1.3B 480p, one frame over itself and two cached ones, through
        # the drop-in attention() with the flat cache's window (q not pre-scaled)
        {"name": "attn_13b_480p_1f_over_2f", "kind": "attn", "batch": 1, "heads": 12, "q": 1560,
         "keys": 4680, "segs": 1, "lo": 0, "pre": False},
        # 1.3B 480p, three frames over six cached ones and themselves: cache + chunk in place
        {"name": "attn_13b_480p_3f_over_6f", "kind": "attn", "batch": 1, "heads": 12, "q": 4680,
         "keys": 14040, "segs": 2, "lo": 0, "pre": True},
        # one tensor-parallel rank of eight of the 14B model, 720p, a full flat cache
        {"name": "attn_14b_720p_5heads", "kind": "attn", "batch": 1, "heads": 5, "q": 3600,
         "keys": 46800, "segs": 1, "lo": 0, "pre": True},
        # 14B 720p, one frame over twelve cached ones and itself: the headline chunk
        {"name": "attn_14b_720p_1f_over_12f", "kind": "attn", "batch": 1, "heads": 40, "q": 3600,
         "keys": 46800, "segs": 1, "lo": 0, "pre": True},
        # the long horizon: 14B 720p over 24 cached frames and itself in an fp8 cache
        {"name": "attn_fp8_14b_720p_1f_over_24f", "kind": "attn_fp8", "batch": 1, "heads": 40,
         "q": 3600, "keys": 90000, "segs": 1, "pre": True},
        # a chunk's K and V into their fp8 cache slots, 14B 720p
        {"name": "kv_quant_14b_720p", "kind": "quant", "batch": 1, "heads": 40, "tokens": 3600},
        # q/k norm + RoPE of a chunk with its K and V committed to the cache, 14B 720p, from the
        # fused QKV projection
        {"name": "qk_rows_14b_720p", "kind": "qk_rows", "heads": 40, "f": 1, "h": 45, "w": 80,
         "extra": 0, "start": 12},
        # the same with head-major, d-major outputs (N-major caches), 14B 480p three frames
        {"name": "qk_dmajor_14b_480p", "kind": "qk_dmajor", "heads": 40, "f": 3, "h": 30, "w": 52,
         "extra": 0, "start": 18},
        # cross-attention to the whole 512-row text context, 14B 480p three frames
        {"name": "cross_14b_480p_512", "kind": "cross", "batch": 1, "heads": 40, "q": 4680,
         "ctx": 512, "valid": 512, "mode": "all"},
        # cross-attention with the context's padding masked, 1.3B 480p three frames
        {"name": "cross_13b_480p_300of512", "kind": "cross", "batch": 1, "heads": 12, "q": 4680,
         "ctx": 512, "valid": 300, "mode": "masked"},
        # the chained calls over a chunk list: partials of each call merged into one running
        # triple, the last call normalises; 1.3B 480p, one frame, three chunks
        {"name": "chain_13b_480p_3chunks", "kind": "chain", "batch": 1, "heads": 12, "q": 1560,
         "keys": 4680, "segs": 3},
        # a whole self-attention layer over the chunked cache (projections, norm + RoPE + commit,
        # attention, output projection): 1.3B 480p, three frames, three chunk slots
        {"name": "layer_13b_480p_chunked", "kind": "layer", "heads": 12, "f": 3, "h": 30, "w": 52,
         "slots": 3, "start": 15},
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["attn", "attn", "attn", "attn_fp8", "quant", "qk_rows", "qk_dmajor",
                       "cross", "cross", "chain", "layer"])
    heads = rng.choice([2, 3, 5, 10, 12, 20, 24, 40])
    if kind in ("attn", "attn_fp8"):
        top = 46800 if kind == "attn" else 90000
        q = _log(rng, 300, 4680)
        keys = _log(rng, max(q, 1500), top)
        # no more than the largest listed case of its kind
        keys = max(q, min(keys, 40 * 3600 * top // (heads * q)))
        segs = rng.choice([1, 1, 2, 3, 4])
        c = {"kind": kind, "batch": 1, "heads": heads, "q": q, "keys": keys, "segs": segs,
             "pre": rng.random() < 0.6}
        if kind == "attn":
            c["lo"] = rng.randrange(1, 500) if segs == 1 and rng.random() < 0.4 else 0
        return c
    if kind == "quant":
        return {"kind": kind, "batch": rng.choice([1, 2]), "heads": heads,
                "tokens": _log(rng, 300, 4680)}
    if kind in ("qk_rows", "qk_dmajor"):
        f, h, w = rng.choice([1, 1, 2, 3]), rng.randrange(15, 46), rng.randrange(20, 53)
        return {"kind": kind, "heads": heads, "f": f, "h": h, "w": w,
                "extra": rng.choice([0, 0, 1, 13, 64]), "start": rng.randrange(0, 60)}
    if kind == "cross":
        mode = rng.choice(["all", "masked", "dedup"])
        ctx = rng.choice([512, 512, 512, rng.randrange(80, 512)])
        valid = ctx if mode == "all" else rng.randrange(20, ctx)
        return {"kind": kind, "batch": 1 if mode == "dedup" else rng.choice([1, 1, 2]),
                "heads": heads, "q": _log(rng, 300, 4680), "ctx": ctx, "valid": valid,
                "mode": mode}
    if kind == "chain":
        q = _log(rng, 300, 3600)
        segs = rng.choice([2, 3, 4])
        return {"kind": kind, "batch": 1, "heads": rng.choice([2, 3, 5, 12]), "q": q,
                "keys": q * segs + rng.randrange(0, 100), "segs": segs}
    return {"kind": "layer", "heads": rng.choice([2, 5, 8, 12]), "f": rng.choice([1, 2, 3]),
            "h": rng.randrange(15, 31), "w": rng.randrange(20, 53), "slots": rng.choice([2, 3, 4]),
            "start": rng.randrange(0, 30)}


# ---- sizes

def _lens(case):
    """Segment lengths of a cache + chunk list: the chunk last, the cached keys in even parts."""
    n, keys, q = case["segs"], case["keys"], case["q"]
    if n == 1:
        return [keys]
    last = q if keys - q >= n - 1 else keys // n
    rest, k = keys - last, n - 1
    return [rest // k + (1 if i < rest % k else 0) for i in range(k)] + [last]


def _tokens(case):
    return case["f"] * case["h"] * case["w"] + case.get("extra", 0)


def work(case):
    kind, h = case["kind"], case["heads"]
    c = h * D
    b = case.get("batch", 1)
    if kind in ("attn", "chain"):
        q, k = case["q"], case["keys"]
        return {"bytes": b * 2 * (2 * q + 2 * k) * c, "flops": 4 * b * q * k * c}
    if kind == "attn_fp8":
        q, k = case["q"], case["keys"]
        return {"bytes": b * (2 * 2 * q * c + 2 * k * c + 2 * 4 * h * (k // 64 + 1)),
                "flops": 4 * b * q * k * c}
    if kind == "cross":
        # identical padding rows are one weighted row of the deduplicated form
        q, k = case["q"], case["valid"] + (case["mode"] == "dedup")
        return {"bytes": b * 2 * (2 * q + 2 * k) * c, "flops": 4 * b * q * k * c}
    if kind == "quant":
        t = case["tokens"]
        return {"bytes": 2 * b * (3 * t * c + 4 * h * ((t + 63) // 64)), "flops": 0}
    t = _tokens(case)
    if kind == "qk_rows":
        return {"bytes": 12 * c * t, "flops": 0}
    if kind == "qk_dmajor":
        return {"bytes": 8 * c * t, "flops": 0}
    k = t * case["slots"]
    return {"bytes": 2 * (2 * t * c + 4 * c * c + 2 * k * c),
            "flops": 8 * t * c * c + 4 * t * k * c}


def tolerance(case):
    kind = case["kind"]
    if kind == "quant":
        return "exact"
    return {"rel": TOL[kind], "max": MAX[kind]}


# about four times the error against exact(), which is also what another correct order of sums or
# another rounding of P shows: one bf16 rounding of the output (2^-9 of each value at most, 1.6e-3
# rel) and, in the attention, P rounded to bf16
TOL = {"attn": 1e-2, "attn_fp8": 1e-2, "cross": 1e-2, "chain": 1e-2, "qk_rows": 8e-3,
       "qk_dmajor": 8e-3, "layer": 1.5e-2}
MAX = {"attn": 0.1, "attn_fp8": 0.1, "cross": 0.1, "chain": 0.1, "qk_rows": 0.04,
       "qk_dmajor": 0.04, "layer": 0.15}


# ---- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _q_k_v(case, g, lens):
    """q and k as RMSNorm and its gammas leave them (unit variance, heads of different sharpness),
    v as its projection gives it."""
    b, h = case.get("batch", 1), case["heads"]
    gain = 0.8 + 1.2 * torch.rand(h, 1, generator=g, device="cuda")
    q = _randn(g, b, case["q"], h, D) * gain
    if case.get("pre"):
        q = q * lbw_amd.prescaled_q_scale(D)
    ks = [_randn(g, b, n, h, D).to(BF16) for n in lens]
    vs = [_randn(g, b, n, h, D).to(BF16) for n in lens]
    return q.to(BF16), ks, vs


def _quantised(x):
    """The fp8 cache's format: e4m3 codes [B, L, H, D] and one power-of-two scale per (batch, head,
    64 tokens), the smallest 2^k that brings the block's largest magnitude to 448 at most."""
    b, n, h, d = x.shape
    blocks = (n + 63) // 64
    pad = torch.zeros(b, blocks * 64, h, d, dtype=torch.float32, device=x.device)
    pad[:, :n] = x.float()
    t = pad.view(b, blocks, 64, h, d)
    amax = t.abs().amax(dim=(2, 4))                                    # [B, blocks, H]
    mant, expo = torch.frexp(amax / 448.0)                             # amax / 448 = mant 2^expo
    k = torch.where(mant == 0.5, expo - 1, expo).clamp(min=-126)
    scale = torch.where(amax > 0, torch.ldexp(torch.ones_like(amax), k), torch.ones_like(amax))
    codes = (t / scale[:, :, None, :, None]).to(torch.float8_e4m3fn).view(torch.uint8)
    codes = codes.view(b, blocks * 64, h, d)[:, :n].contiguous()
    return codes, scale.permute(0, 2, 1).contiguous()


def _dequantised(codes, scale):
    n = codes.shape[1]
    s = scale.permute(0, 2, 1).repeat_interleave(64, dim=1)[:, :n]
    return codes.view(torch.float8_e4m3fn).float() * s[..., None]


def prepare(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    s = {"case": case}
    if kind == "attn":
        lens = _lens(case)
        if case["lo"]:
            lens = [lens[0] + case["lo"]]   # a flat cache whose window starts at `lo`
        s["q"], s["k"], s["v"] = _q_k_v(case, g, lens)
    elif kind == "attn_fp8":
        s["q"], ks, vs = _q_k_v(case, g, _lens(case))
        s["segs"] = [(lbw_amd.Fp8KV(*_quantised(k)), lbw_amd.Fp8KV(*_quantised(v)))
                     for k, v in zip(ks, vs)]
    elif kind == "chain":
        s["q"], ks, vs = _q_k_v(case, g, _lens(case))
        s["segs"] = list(zip(ks, vs))
    elif kind == "cross":
        s["q"], (k,), (v,) = _q_k_v(case, g, [case["ctx"]])
        n = case["valid"]
        if n < case["ctx"]:   # the projected zero padding: identical rows
            k[:, n:] = k[:, -1:].clone()
            v[:, n:] = v[:, -1:].clone()
        s["k"], s["v"] = k, v
        if case["mode"] == "masked":
            s["k_lens"] = torch.full((case["batch"],), n, dtype=torch.int32, device="cuda")
    elif kind == "quant":
        b, t, h = case["batch"], case["tokens"], case["heads"]
        blocks = (t + 63) // 64
        s["x"], s["slots"] = [], []
        for _ in range(2):
            s["x"].append(_randn(g, b, t, h, D).to(BF16))
            s["slots"].append(lbw_amd.Fp8KV(
                torch.zeros(b, t, h, D, dtype=torch.uint8, device="cuda"),
                torch.ones(b, h, blocks, dtype=torch.float32, device="cuda")))
    else:
        _prepare_rows(case, g, s)
    return s


def _vectors(g, c):
    """q and k biases and RMSNorm gammas."""
    return [(0.1 * _randn(g, c)).to(BF16), (0.1 * _randn(g, c)).to(BF16),
            (1 + 0.1 * _randn(g, c)).to(BF16), (1 + 0.1 * _randn(g, c)).to(BF16)]


def _prepare_rows(case, g, s):
    h = case["heads"]
    c, t = h * D, _tokens(case)
    s["bq"], s["bk"], s["gq"], s["gk"] = _vectors(g, c)
    s["freqs"] = lbw_amd.wan_rope_freqs(D)
    grid = (case["f"], case["h"], case["w"])
    if case["kind"] == "layer":
        s["x"] = _randn(g, 1, t, c).to(BF16)
        s["w"] = [(_randn(g, c, c) / math.sqrt(c)).to(BF16) for _ in range(4)]
        s["bv"], s["bo"] = (0.1 * _randn(g, c)).to(BF16), (0.1 * _randn(g, c)).to(BF16)
        wq, wk, wv, wo = s["w"]
        s["layer"] = lbw_amd.WanSelfAttention(wq, s["bq"], wk, s["bk"], wv, s["bv"], wo, s["bo"],
                                              s["gq"], s["gk"], heads=h, eps=EPS,
                                              freqs=s["freqs"])
        n = case["slots"]
        s["chunks"] = {"k": [_randn(g, 1, t, h, D).to(BF16) for _ in range(n)],
                       "v": [_randn(g, 1, t, h, D).to(BF16) for _ in range(n)]}
        s["index"] = n + 1   # every slot written before, the sink and a rotated one among them
        s["grid"] = grid
        s["dest"], s["leading"] = lbw_amd.chunk_routing(s["index"], n)
        return
    s["qkv"] = _randn(g, t, 3 * c).to(BF16)
    s["tabs"] = lbw_amd.causal_rope_tables(s["freqs"], grid, case["start"], device="cuda")
    if case["kind"] == "qk_rows":
        s["q_out"] = torch.empty(t, c, dtype=BF16, device="cuda")
        # the slot is the end of a flat cache
        s["cache_k"] = torch.zeros(1, t + 64, h, D, dtype=BF16, device="cuda")
        s["cache_v"] = torch.zeros(1, t + 64, h, D, dtype=BF16, device="cuda")


# ---- one pass

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "attn":
        if case["pre"]:
            lo = case["lo"]
            return lbw_amd.attention_segments(
                s["q"], list(zip(s["k"], s["v"])), kv_lo=lo, kv_hi=lo + case["keys"],
                softmax_scale=lbw_amd.PRESCALED_SOFTMAX_SCALE)
        if case["segs"] == 1:
            lo = case["lo"]
            return lbw_amd.attention(s["q"], s["k"][0], s["v"][0], kv_lo=lo,
                                     kv_hi=lo + case["keys"])
        return lbw_amd.exact_attention_chunks(s["q"], s["k"], s["v"])
    if kind == "attn_fp8":
        return lbw_amd.attention_fp8kv(
            s["q"], s["segs"],
            softmax_scale=lbw_amd.PRESCALED_SOFTMAX_SCALE if case["pre"] else None)
    if kind == "chain":
        state = None
        for seg in s["segs"][:-1]:
            state = lbw_amd.attention_chain(s["q"], [seg], state)
        return lbw_amd.attention_chain(s["q"], [s["segs"][-1]], state, normalize=True)
    if kind == "cross":
        return lbw_amd.cross_attention(
            s["q"], s["k"], s["v"], k_lens=s.get("k_lens"),
            n_distinct=case["valid"] if case["mode"] == "dedup" else None)
    if kind == "quant":
        out = []
        for x, slot in zip(s["x"], s["slots"]):
            lbw_amd.quantize_kv_fp8(x, out=slot)
            out += [slot.codes, slot.scales]
        return out
    if kind == "qk_rows":
        t, c = s["q_out"].shape
        ks, vs = s["cache_k"][0, 64:].view(t, c), s["cache_v"][0, 64:].view(t, c)
        qkv = s["qkv"]
        lbw_amd.qk_norm_rope_(qkv[:, :c], qkv[:, c:2 * c], s["bq"], s["bk"], s["gq"], s["gk"],
                              s["tabs"], EPS, case["heads"], q_out=s["q_out"], k_out=ks,
                              v=qkv[:, 2 * c:], v_out=vs, q_scale=lbw_amd.prescaled_q_scale(D))
        return [s["q_out"], ks, vs]
    if kind == "qk_dmajor":
        return list(lbw_amd.qk_norm_rope_t3(s["qkv"], s["bq"], s["bk"], s["gq"], s["gk"],
                                            s["tabs"], EPS))
    y = s["layer"].forward_chunked(s["x"], s["grid"], case["start"], s["chunks"], s["index"])
    return [y, s["chunks"]["k"][s["dest"]], s["chunks"]["v"][s["dest"]]]


# ---- the same in 64 bits

def _attention64(q, k, v, scale):
    """softmax(scale q k^T) v per head, q [B, Lq, H, D] -> float64 of that shape."""
    b, lq, h, d = q.shape
    lk = k.shape[1]
    out = torch.empty(b, lq, h, d, dtype=torch.float64, device=q.device)
    step = max(64, min(lq, (1 << 27) // lk))
    for i in range(b):
        for j in range(h):
            kt = k[i, :, j].double().t().contiguous()
            vj = v[i, :, j].double().contiguous()
            for r in range(0, lq, step):
                sc = (q[i, r:r + step, j].double() @ kt) * scale
                out[i, r:r + step, j] = torch.softmax(sc, dim=-1) @ vj
    return out


def _norm_rope64(x, bias, gamma, case, scale):
    """RMSNorm and the 3-D rotation of rows [L, C] -> float64 [L, C]."""
    t, c = x.shape
    h = c // D
    y = x.double() + bias.double()
    y = y / torch.sqrt((y * y).mean(dim=1, keepdim=True) + EPS) * gamma.double()
    f, gh, gw = case["f"], case["h"], case["w"]
    n = f * gh * gw
    pairs = D // 2
    s1 = pairs // 3
    s0 = pairs - 2 * s1
    dev = x.device
    row = torch.arange(n, device=dev)
    pos = [row // (gh * gw) + case["start"], (row // gw) % gh, row % gw]
    ang = []
    for p, m in zip(pos, (s0, s1, s1)):
        inv = 10000.0 ** (-torch.arange(m, dtype=torch.float64, device=dev) / m)
        ang.append(p.double()[:, None] * inv[None])
    ang = torch.cat(ang, dim=1)[:, None, :]                            # [n, 1, pairs]
    z = y[:n].view(n, h, pairs, 2)
    co, si = ang.cos(), ang.sin()
    rot = torch.stack([z[..., 0] * co - z[..., 1] * si, z[..., 0] * si + z[..., 1] * co], dim=-1)
    return torch.cat([rot.reshape(n, c), y[n:]], dim=0) * scale


def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    scale = 1.0 / math.sqrt(D)
    pre = math.log(2.0) if case.get("pre") else scale
    if kind == "attn":
        lo, hi = case["lo"], case["lo"] + case["keys"]
        return _attention64(s["q"], torch.cat(s["k"], 1)[:, lo:hi], torch.cat(s["v"], 1)[:, lo:hi],
                            pre)
    if kind == "attn_fp8":
        # over the keys and values that the cache holds
        k = torch.cat([_dequantised(a.codes, a.scales) for a, _ in s["segs"]], 1)
        v = torch.cat([_dequantised(a.codes, a.scales) for _, a in s["segs"]], 1)
        return _attention64(s["q"], k, v, pre)
    if kind == "chain":
        return _attention64(s["q"], torch.cat([k for k, _ in s["segs"]], 1),
                            torch.cat([v for _, v in s["segs"]], 1), scale)
    if kind == "cross":
        n = case["valid"] if case["mode"] == "masked" else case["ctx"]
        return _attention64(s["q"], s["k"][:, :n], s["v"][:, :n], scale)
    if kind == "quant":
        return [t for x in s["x"] for t in _quantised(x)]
    c = case["heads"] * D
    if kind in ("qk_rows", "qk_dmajor"):
        qkv = s["qkv"]
        rows = kind == "qk_rows"
        q = _norm_rope64(qkv[:, :c], s["bq"], s["gq"], case,
                         lbw_amd.prescaled_q_scale(D) if rows else scale)
        k = _norm_rope64(qkv[:, c:2 * c], s["bk"], s["gk"], case, 1.0)
        if rows:
            return [q, k, qkv[:, 2 * c:].double()]
        t = qkv.shape[0]
        return [z.view(t, case["heads"], D).permute(1, 2, 0).contiguous() for z in (q, k)]
    x = s["x"][0].double()
    wq, wk, wv, wo = (w.double() for w in s["w"])
    t = x.shape[0]
    q = _norm_rope64(x @ wq.t(), s["bq"], s["gq"], case, 1.0).view(1, t, -1, D)
    k = _norm_rope64(x @ wk.t(), s["bk"], s["gk"], case, 1.0).view(1, t, -1, D)
    v = (x @ wv.t() + s["bv"].double()).view(1, t, -1, D)
    ks = [s["chunks"]["k"][i].double() for i in s["leading"]] + [k]
    vs = [s["chunks"]["v"][i].double() for i in s["leading"]] + [v]
    o = _attention64(q, torch.cat(ks, 1), torch.cat(vs, 1), scale).view(t, c)
    return [(o @ wo.t() + s["bo"].double()).view(1, t, c), k, v]
