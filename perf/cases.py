"""What a user of this framework has it do, as cases that can be timed and checked.

The framework is the quantized linear path of a decoder: GGUF-quantized weights (Q4_K, Q5_K, Q6_K, Q8_0,
IQ4_XS; F16 / F32 for small ones), re-tiled at load time or used as uploaded, one token at a time (decode),
2 to 16 rows (speculative verification) and up to 64 rows a call (prefill), the token_embd gather, and the
vocab product with its candidate selection.  A case names one such step; `draw` gives steps of the same
kinds over the sizes, types, layouts and row counts that the entry points take.

A case's "path":
  matvec   one weight, one token: y = W x (+ residual), x fp32 or gated by a sigmoid and quantized first
  multi    several weights on one fp32 token in one call (q / k / v, the SSM pair)
  ffn      silu(gate x) * (up x), quantized by the product, then down with the residual
  layer    a decoder layer's linears captured once in a HIP graph and replayed, as a decode loop does
  matmul   M fp32 rows quantized, then one or several weights on them in one call
  vocab    the LM head on one token, its exact top-k and the sampled token
  embed    rows of the embedding table by device ids
  exactvec one weight on an fp32 token with exact dequantization (or F16 / F32 weights)
"""
import importlib

import numpy as np
import torch

m27q = importlib.import_module("mono-qwen27_amd").m27q

TYPES = {"Q4_K": m27q.Q4_K, "Q5_K": m27q.Q5_K, "Q6_K": m27q.Q6_K, "Q8_0": m27q.Q8_0, "IQ4_XS": m27q.IQ4_XS,
         "F16": m27q.F16, "F32": m27q.F32}
BLOCK = {"Q4_K": 256, "Q5_K": 256, "Q6_K": 256, "Q8_0": 32, "IQ4_XS": 256, "F16": 1, "F32": 1}
BLOCK_BYTES = {"Q4_K": 144, "Q5_K": 176, "Q6_K": 210, "Q8_0": 34, "IQ4_XS": 136, "F16": 2, "F32": 4}
LAYOUTS = {"tiled": m27q.TILED, "gguf": m27q.GGUF}
IQ4_VALUES = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)
STD = 0.02  # of the weights


def listed():
    return [
        # the draft model's projection, the smallest call of a decode loop: latency and host cost
        {"name": "draft_proj_m1", "path": "matvec", "types": "Q8_0", "rows": "2048", "K": 2048, "layout": "tiled",
         "M": 1, "residual": False, "gated": False},
        # an attention block's q / k / v on one token
        {"name": "attn_qkv_m1", "path": "multi", "types": "Q4_K,Q4_K,Q4_K", "rows": "6144,1024,1024", "K": 5120,
         "layout": "tiled", "M": 1},
        # the feed-forward block on one token
        {"name": "ffn_block_m1", "path": "ffn", "types": "Q4_K,Q6_K", "rows": "17408,5120", "K": 5120,
         "layout": "tiled", "M": 1},
        # a decoder layer's linears as a decode loop replays them
        {"name": "decode_layer_m1", "path": "layer", "types": "Q4_K,Q4_K,Q6_K", "rows": "8192,6144,17408", "K": 5120,
         "layout": "tiled", "M": 1},
        # the SSM block's pair of mixed types, weights used as they lie in the checkpoint
        {"name": "ssm_pair_m1_gguf", "path": "multi", "types": "Q6_K,Q5_K", "rows": "10240,6144", "K": 5120,
         "layout": "gguf", "M": 1},
        # next-token choice over the whole vocabulary
        {"name": "vocab_top64", "path": "vocab", "types": "Q6_K", "rows": "248320", "K": 5120, "layout": "tiled",
         "M": 1, "k": 64},
        # the embedding rows of a prompt
        {"name": "embed_512", "path": "embed", "types": "Q6_K", "rows": "248320", "K": 5120, "layout": "tiled",
         "M": 512},
        # speculative verification: a few rows on q / k / v
        {"name": "verify_qkv_m4", "path": "matmul", "types": "Q4_K,Q4_K,Q4_K", "rows": "6144,1024,1024", "K": 5120,
         "layout": "tiled", "M": 4, "residual": False},
        # speculative verification: a full batch of rows on gate / up
        {"name": "verify_gate_up_m16", "path": "matmul", "types": "Q4_K,Q4_K", "rows": "17408,17408", "K": 5120,
         "layout": "tiled", "M": 16, "residual": False},
        # prefill, the most rows a call takes: gate / up, and down with the residual
        {"name": "prefill_gate_up_m64", "path": "matmul", "types": "Q4_K,Q4_K", "rows": "17408,17408", "K": 5120,
         "layout": "tiled", "M": 64, "residual": False},
        {"name": "prefill_down_m64", "path": "matmul", "types": "Q6_K", "rows": "5120", "K": 17408,
         "layout": "tiled", "M": 64, "residual": True},
        # the draft model's prefill tail: an odd number of rows, weights as they lie in the checkpoint
        {"name": "draft_prefill_m37_gguf", "path": "matmul", "types": "Q8_0,Q8_0", "rows": "6144,6144", "K": 2048,
         "layout": "gguf", "M": 37, "residual": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _blocks(rng, lo, hi, block):
    return block * _log_int(rng, max(1, lo // block), hi // block)


def draw(rng):
    """One more case of the same ranges: any quantized type, either layout, odd and ragged sizes."""
    path = rng.choice(["matvec", "multi", "ffn", "layer", "matmul", "matmul", "matmul", "vocab", "embed", "exactvec"])
    t = rng.choice(["Q4_K", "Q4_K", "Q6_K", "Q6_K", "Q5_K", "Q8_0", "Q8_0", "IQ4_XS"])
    layout = rng.choice(["tiled", "tiled", "gguf"])
    K = _blocks(rng, 512, 17408, BLOCK[t])
    if path == "matvec":
        return {"path": path, "types": t, "rows": str(_log_int(rng, 48, 17408)), "K": K, "layout": layout, "M": 1,
                "residual": rng.random() < 0.5, "gated": rng.random() < 0.3}
    if path == "multi":
        K = _blocks(rng, 1024, 6144, 256)
        n = rng.choice([2, 3, 4])
        ts = [t] * n if rng.random() < 0.6 else [rng.choice(["Q4_K", "Q5_K", "Q6_K", "Q8_0"]) for _ in range(n)]
        return {"path": path, "types": ",".join(ts), "rows": ",".join(str(_log_int(rng, 256, 10240)) for _ in ts),
                "K": K, "layout": layout, "M": 1}
    if path == "ffn":
        t, down = rng.choice([("Q4_K", "Q6_K"), ("Q4_K", "Q4_K"), ("Q5_K", "Q6_K"), ("Q8_0", "Q8_0")])
        K = 256 * _log_int(rng, 4, 20)
        return {"path": path, "types": "%s,%s" % (t, down), "rows": "%d,%d" % (256 * _log_int(rng, 8, 68), K), "K": K,
                "layout": layout, "M": 1}
    if path == "layer":
        t, down = rng.choice([("Q4_K", "Q6_K"), ("Q5_K", "Q6_K"), ("Q8_0", "Q8_0")])
        K = 256 * _log_int(rng, 4, 20)
        q = 256 * _log_int(rng, 4, 24)
        return {"path": path, "types": "%s,%s,%s" % (t, t, down),
                "rows": "%d,%d,%d" % (q + 2 * max(32, q // 6), q, 256 * _log_int(rng, 8, 68)), "K": K,
                "layout": layout, "M": 1}
    if path == "matmul":
        n = rng.choice([1, 1, 2, 3])
        res = n == 1 and rng.random() < 0.5
        hi = 17408 if K <= 6144 else 6144
        rows = [_log_int(rng, 64, hi) for _ in range(n)]
        return {"path": path, "types": ",".join([t] * n), "rows": ",".join(str(r) for r in rows), "K": K,
                "layout": layout, "M": _log_int(rng, 2, 64), "residual": res}
    if path == "vocab":
        return {"path": path, "types": rng.choice(["Q6_K", "Q8_0", "Q4_K"]), "rows": str(_log_int(rng, 32000, 160001)),
                "K": 256 * _log_int(rng, 4, 20), "layout": layout, "M": 1, "k": rng.choice([1, 20, 40, 64])}
    if path == "embed":
        return {"path": path, "types": rng.choice([t, "F16"]), "rows": str(_log_int(rng, 8192, 151936)),
                "K": 256 * _log_int(rng, 4, 20), "layout": "gguf" if rng.random() < 0.3 else "tiled",
                "M": _log_int(rng, 1, 2048)}
    t = rng.choice([t, "F16", "F32"])
    return {"path": path, "types": t, "rows": str(_log_int(rng, 48, 6144)), "K": 256 * _log_int(rng, 2, 24),
            "layout": layout, "M": 1}


# ---------------------------------------------------------------------------------- weights --
# N(0, STD) values rounded to each block format; `_values` gives the same blocks' exact values in 64 bits.

def _f16(x):
    return x.to(torch.float16)


def _nz(x):
    return torch.where(x == 0, torch.ones_like(x), x)


def _quantize(t, w):
    """fp32 [n, K] -> the fields of its blocks."""
    n = w.shape[0]
    if t in ("F16", "F32"):
        return {"w": _f16(w) if t == "F16" else w}
    if t in ("Q4_K", "Q5_K"):
        top = 15 if t == "Q4_K" else 31
        g = w.view(n, -1, 8, 32)
        lo, hi = g.amin(-1).clamp(max=0), g.amax(-1)
        s, m = (hi - lo) / top, -lo
        d, dm = _f16(s.amax(-1) / 63), _f16(m.amax(-1) / 63)
        sc = torch.round(s / _nz(d.float())[..., None]).clamp(0, 63)
        mn = torch.round(m / _nz(dm.float())[..., None]).clamp(0, 63)
        q = torch.round((g + (dm.float()[..., None] * mn)[..., None]) / _nz(d.float()[..., None] * sc)[..., None])
        return {"d": d, "dm": dm, "sc": sc.to(torch.uint8), "mn": mn.to(torch.uint8), "q": q.clamp(0, top).to(torch.uint8)}
    if t == "Q6_K":
        g = w.view(n, -1, 16, 16)
        far = g.gather(-1, g.abs().argmax(-1, keepdim=True)).squeeze(-1)
        s = far / -32
        d = _f16(s.abs().amax(-1) / 127)
        sc = torch.round(s / _nz(d.float())[..., None]).clamp(-128, 127)
        q = torch.round(g / _nz(d.float()[..., None] * sc)[..., None]).clamp(-32, 31)
        return {"d": d, "sc": sc.to(torch.int8), "q": q.to(torch.int8)}
    if t == "Q8_0":
        g = w.view(n, -1, 32)
        d = _f16(g.abs().amax(-1) / 127)
        return {"d": d, "q": torch.round(g / _nz(d.float())[..., None]).clamp(-127, 127).to(torch.int8)}
    g = w.view(n, -1, 8, 32)  # IQ4_XS
    s = g.abs().amax(-1) / 120
    d = _f16(s.amax(-1) / 31)
    sc = torch.round(s / _nz(d.float())[..., None]).clamp(-32, 31)
    v = torch.tensor(IQ4_VALUES, dtype=torch.float32, device=w.device)
    x = (g / _nz(d.float()[..., None] * sc)[..., None]).contiguous()
    return {"d": d, "sc": sc.to(torch.int8), "q": torch.bucketize(x, (v[1:] + v[:-1]) / 2).to(torch.uint8)}


def _values(t, f):
    """The blocks' exact values, float64 [n, K]."""
    if t in ("F16", "F32"):
        return f["w"].double()
    n = f["d"].shape[0]
    d = f["d"].double()
    if t in ("Q4_K", "Q5_K"):
        x = (d[..., None] * f["sc"])[..., None] * f["q"] - (f["dm"].double()[..., None] * f["mn"])[..., None]
    elif t == "Q8_0":
        x = d[..., None] * f["q"]
    elif t == "Q6_K":
        x = (d[..., None] * f["sc"])[..., None] * f["q"]
    else:
        v = torch.tensor(IQ4_VALUES, dtype=torch.float64, device=d.device)
        x = (d[..., None] * f["sc"])[..., None] * v[f["q"].long()]
    return x.reshape(n, -1)


def _bytes(x):
    return x.contiguous().view(torch.uint8)


def _pack(t, f):
    """The blocks' GGUF bytes, uint8 [n, row bytes]."""
    if t in ("F16", "F32"):
        return _bytes(f["w"])
    n, q = f["d"].shape[0], f["q"]
    d = _bytes(f["d"][..., None])
    if t in ("Q4_K", "Q5_K"):
        sc, mn = f["sc"], f["mn"]
        lo, hi = slice(0, 4), slice(4, 8)
        scales = torch.cat([sc[..., lo] | (sc[..., hi] >> 4 << 6), mn[..., lo] | (mn[..., hi] >> 4 << 6),
                            (sc[..., hi] & 15) | ((mn[..., hi] & 15) << 4)], -1)
        nib = q & 15
        qs = (nib[..., 0::2, :] | (nib[..., 1::2, :] << 4)).flatten(-2)
        parts = [d, _bytes(f["dm"][..., None]), scales]
        if t == "Q5_K":
            bits = torch.zeros_like(q[..., 0, :])
            for j in range(8):
                bits |= (q[..., j, :] >> 4) << j
            parts.append(bits)
        parts.append(qs)
    elif t == "Q8_0":
        parts = [d, _bytes(q)]
    elif t == "Q6_K":
        b = (q + 32).to(torch.uint8).view(*q.shape[:2], 2, 4, 32)  # half, quarter, position
        ql = torch.cat([(b[..., k, :] & 15) | ((b[..., k + 2, :] & 15) << 4) for k in (0, 1)], -1).flatten(-2)
        qh = torch.zeros_like(b[..., 0, :])
        for k in range(4):
            qh |= (b[..., k, :] >> 4) << (2 * k)
        parts = [ql, qh.flatten(-2), _bytes(f["sc"]), d]
    else:
        ls = (f["sc"].to(torch.int32) + 32)
        sh = torch.zeros_like(ls[..., 0])
        for j in range(8):
            sh |= (ls[..., j] >> 4) << (2 * j)
        sl = ((ls[..., 0::2] & 15) | ((ls[..., 1::2] & 15) << 4)).to(torch.uint8)
        qs = (q[..., :16] | (q[..., 16:] << 4)).flatten(-2)
        parts = [d, torch.stack([sh & 255, sh >> 8], -1).to(torch.uint8), sl, qs]
    return torch.cat(parts, -1).reshape(n, -1)


def _fields(t, rows, K, seed, device):
    """The fields of a weight's blocks, a run of rows at a time (the same ones for the same arguments)."""
    gen = torch.Generator(device).manual_seed(seed)
    step = max(1, (1 << 26) // K)
    for r0 in range(0, rows, step):
        n = min(step, rows - r0)
        yield r0, _quantize(t, torch.randn((n, K), generator=gen, device=device) * STD)


def _specs(case):
    """(type, rows, K) of each weight."""
    ts, rows, K = case["types"].split(","), [int(r) for r in case["rows"].split(",")], case["K"]
    if case["path"] == "ffn":  # gate, up, down
        return [(ts[0], rows[0], K), (ts[0], rows[0], K), (ts[1], rows[1], rows[0])]
    if case["path"] == "layer":  # q, k, v, o, gate, up, down
        q, kv, inner = rows[1], (rows[0] - rows[1]) // 2, rows[2]
        return [(ts[0], q, K), (ts[0], kv, K), (ts[0], kv, K), (ts[1], K, q), (ts[0], inner, K), (ts[0], inner, K),
                (ts[2], K, inner)]
    return [(t, r, K) for t, r in zip(ts, rows)]


def _weights(case, seed):
    out = []
    for i, (t, rows, K) in enumerate(_specs(case)):
        host = np.empty((rows, K // BLOCK[t] * BLOCK_BYTES[t]), np.uint8)
        for r0, f in _fields(t, rows, K, 1000 * seed + i, "cuda"):
            b = _pack(t, f)
            host[r0:r0 + b.shape[0]] = b.cpu().numpy()
        layout = m27q.GGUF if t in ("F16", "F32") else LAYOUTS[case["layout"]]
        out.append(m27q.Weight.upload(host, TYPES[t], K // BLOCK[t], rows, layout))
    return out


# ------------------------------------------------------------------------------- activations --

def _normal(seed, which, *shape):
    return np.random.default_rng([seed, which]).standard_normal(shape).astype(np.float32)


def _inputs(case, seed):
    """The fp32 host arrays of a case, the same for prepare and exact."""
    p, specs, M = case["path"], _specs(case), case["M"]
    if p == "embed":
        ids = np.random.default_rng([seed, 9]).integers(0, specs[0][1], M)
        return {"ids": ids.astype(np.int32)}
    x = {"x": _normal(seed, 1, M, specs[0][2])}
    if case.get("gated") or p == "layer":
        x["gate"] = _normal(seed, 2, M, specs[3][2] if p == "layer" else specs[0][2])
    if p == "layer":
        x["attn"] = _normal(seed, 3, M, specs[3][2])
    if case.get("residual") or p in ("ffn", "layer"):
        x["res"] = _normal(seed, 4, M, specs[-1][1])
    if p == "vocab":
        x["u"] = np.random.default_rng([seed, 5]).random(1).astype(np.float32)
    return x


def _decode_layer(s):
    w = s["w"]
    m27q.matvec_multi(w[:3], s["x"], s["ys"][:3])
    m27q.quant_act(s["attn"], s["aq"], gate=s["gate"])
    m27q.matvec_q8(w[3], s["aq"], s["ys"][3], residual=s["res"])
    m27q.ffn_swiglu(w[4], w[5], s["x"], s["ys"][4], yq=s["hq"])
    m27q.matvec_q8(w[6], s["hq"], s["ys"][5], residual=s["res"])


def prepare(case, seed):
    p, specs, M, K = case["path"], _specs(case), case["M"], case["K"]
    s = {"case": case, "path": p, "w": _weights(case, seed)}
    for k, v in _inputs(case, seed).items():
        s[k] = torch.from_numpy(v).cuda()
    new = lambda *shape: torch.empty(shape, dtype=torch.float32, device="cuda")  # noqa: E731
    if p == "embed":
        s["ys"] = [new(M, K)]
    elif p == "ffn":
        s["ys"] = [new(1, specs[0][1]), new(1, specs[2][1])]
        s["hq"] = m27q.Act(1, specs[0][1])
    elif p == "layer":
        s["ys"] = [new(1, specs[i][1]) for i in (0, 1, 2, 3, 4, 6)]
        s["aq"], s["hq"] = m27q.Act(1, specs[3][2]), m27q.Act(1, specs[6][2])
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _decode_layer(s)
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            _decode_layer(s)
    else:
        s["ys"] = [new(M, r) for _, r, _ in specs]
    if p == "matmul" or case.get("gated"):
        s["xq"] = m27q.Act(M, K)
    if p == "vocab":
        n, k = specs[0][1], case["k"]
        s["idx"] = torch.empty(k, dtype=torch.int32, device="cuda")
        s["val"] = new(k)
        s["token"] = torch.empty(1, dtype=torch.int32, device="cuda")
        s["scratch"] = torch.empty(m27q.topk_scratch_bytes(n, k), dtype=torch.uint8, device="cuda")
    return s


def run(s):
    p, w, ys = s["path"], s["w"], s["ys"]
    if p == "matvec":
        if "xq" in s:
            m27q.quant_act(s["x"], s["xq"], gate=s.get("gate"))
            m27q.matvec_q8(w[0], s["xq"], ys[0], residual=s.get("res"))
        else:
            m27q.matvec(w[0], s["x"], ys[0], residual=s.get("res"))
    elif p == "multi":
        m27q.matvec_multi(w, s["x"], ys)
    elif p == "ffn":
        m27q.ffn_swiglu(w[0], w[1], s["x"], ys[0], yq=s["hq"])
        m27q.matvec_q8(w[2], s["hq"], ys[1], residual=s["res"])
    elif p == "layer":
        s["graph"].replay()
    elif p == "matmul":
        m27q.quant_act(s["x"], s["xq"])
        if len(w) == 1:
            m27q.matmul_q8(w[0], s["xq"], ys[0], residual=s.get("res"))
        else:
            m27q.matmul_q8_multi(w, s["xq"], ys)
    elif p == "vocab":
        k = s["case"]["k"]
        m27q.matvec(w[0], s["x"], ys[0])
        m27q.topk(ys[0], k, s["idx"], s["val"], s["scratch"])
        m27q.sample(s["idx"], s["val"], k, 0.8, 0.05, 0.95, s["u"], s["token"])
        return {"logits": ys[0], "idx": s["idx"], "val": s["val"], "token": s["token"]}
    elif p == "embed":
        m27q.embed_rows(w[0], s["ids"], ys[0])
    else:
        m27q.matvec_f32(w[0], s["x"], ys[0])
    return ys


# ------------------------------------------------------------------------------------ checks --

def work(case):
    specs, M, p = _specs(case), case["M"], case["path"]
    if p == "embed":
        t, _, K = specs[0]
        return {"bytes": M * (K // BLOCK[t] * BLOCK_BYTES[t] + 4 * K + 4), "flops": 0}
    b = sum(r * (K // BLOCK[t]) * BLOCK_BYTES[t] for t, r, K in specs)
    b += sum(4 * v.size for v in _inputs(case, 0).values()) + 4 * M * sum(r for _, r, _ in specs)
    return {"bytes": b, "flops": 2 * M * sum(r * K for _, r, K in specs)}


def tolerance(case):
    p = case["path"]
    if p == "embed":
        return "exact"  # dequantization is bit-exact
    if p == "ffn" or p == "layer":
        # the hidden activations are quantized between two products: a last-bit difference in one of them
        # can move its code by one, a 127th of its group's largest
        return {"rel": 1e-3}
    if case.get("gated"):
        return {"rel": 1e-3}  # the same for the gated values
    if p == "vocab":
        return {"rel": 2e-6, "differ": 0.05}  # neighbours closer than the logits' last bits may swap
    return {"rel": 2e-6}  # exact integer sums per group, combined in 32 bits (measured 1e-7 to 5e-7)


def _codes(x):
    """The values an int8 activation buffer stands for: d = max / 127 per 32, codes round(x / d) half away from zero."""
    g = x.reshape(x.shape[0], -1, 32)
    d = np.abs(g).max(-1, keepdims=True) / np.float32(127)
    inv = np.divide(np.float32(1), d, out=np.zeros_like(d), where=d > 0)
    v = (g * inv).astype(np.float64)
    q = np.clip(np.sign(v) * np.floor(np.abs(v) + 0.5), -127, 127)
    return torch.from_numpy((q * d.astype(np.float64)).reshape(x.shape)).cuda()


def _product(spec, seed, which, x):
    t, rows, K = spec
    y = torch.empty((x.shape[0], rows), dtype=torch.float64, device="cuda")
    for r0, f in _fields(t, rows, K, 1000 * seed + which, "cuda"):
        v = _values(t, f)
        y[:, r0:r0 + v.shape[0]] = x @ v.t().contiguous()
    return y


def _sample(val, u):
    """The token's rank for top-k logits val: softmax at 0.8, min_p 0.05, top_p 0.95, the pick at u."""
    p = torch.softmax((val - val[0]) / 0.8, 0)
    p = p[p >= p[0] * float(np.float32(0.05))]
    run_ = torch.cumsum(p, 0)
    n = int((run_ < float(np.float32(0.95))).sum().item()) + 1
    run_ = run_[:n]
    return int((run_ < float(u) * run_[-1]).sum().item())


def exact(case, seed):
    p, specs = case["path"], _specs(case)
    a = _inputs(case, seed)
    res = torch.from_numpy(a["res"]).cuda().double() if "res" in a else 0
    if p == "embed":
        t, rows, K = specs[0]
        ids = torch.from_numpy(a["ids"]).cuda().long()
        out = torch.empty((len(ids), K), dtype=torch.float64, device="cuda")
        for r0, f in _fields(t, rows, K, 1000 * seed, "cuda"):
            n = (f["w"] if "w" in f else f["d"]).shape[0]
            at = ((ids >= r0) & (ids < r0 + n)).nonzero().flatten()
            if len(at):
                out[at] = _values(t, {k: v[ids[at] - r0] for k, v in f.items()})
        return [out]
    x = a["x"]
    if p == "exactvec":
        return [_product(specs[0], seed, 0, torch.from_numpy(x).cuda().double())]
    if case.get("gated"):
        x = (x.astype(np.float64) / (1 + np.exp(-a["gate"].astype(np.float64)))).astype(np.float32)
    xq = _codes(x)
    if p == "vocab":
        y = _product(specs[0], seed, 0, xq)
        val, idx = torch.topk(y[0], case["k"])
        return {"logits": y, "idx": idx.int(), "val": val, "token": idx[_sample(val, a["u"][0])][None].int()}
    if p in ("ffn", "layer"):
        at = 4 if p == "layer" else 0
        g, u = (_product(specs[at + i], seed, at + i, xq) for i in (0, 1))
        h = g / (1 + torch.exp(-g)) * u
        y = _product(specs[at + 2], seed, at + 2, _codes(h.float().cpu().numpy())) + res
        if p == "ffn":
            return [h, y]
        att = (a["attn"].astype(np.float64) / (1 + np.exp(-a["gate"].astype(np.float64)))).astype(np.float32)
        o = _product(specs[3], seed, 3, _codes(att)) + res
        return [_product(specs[i], seed, i, xq) for i in range(3)] + [o, h, y]
    return [_product(sp, seed, i, xq) + res for i, sp in enumerate(specs)]
