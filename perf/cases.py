"""Performance cases of the quantized-linear library: what its users run.

Each case is a dict of plain values; `kind` selects the call:

  linear     one eager rt_hip_linear_forward on a weight of any format, any number of rows
  layer      the seven projections of a transformer layer, several layers (decode batches replay a captured
             graph, prefill calls eagerly; single-row formats with entry points of their own too)
  token      one decode token through the fused launches a decode loop issues, captured as one graph
  engine     one step of the decode engine (one token, or a batch of tokens to verify)
  flux       a FLUX block's linears: QKV, MLP-in, MLP-out on the image and text tokens, with bias
  attention  FLUX's unmasked attention
  lm_head    the BF16 output projection with the greedy token
  quantize   f32 weights to Q4_K blocks at load, and the blocks back to bf16

Weights and inputs are synthetic: N(0, 0.02) weights encoded to the storage formats here, N(0, 1) activations.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _rt():
    name = "rich_triplet_cpp_amd"
    if name not in sys.modules:
        path = os.path.join(ROOT, "rich-triplet-cpp_amd", "__init__.py")
        spec = importlib.util.spec_from_file_location(name, path, submodule_search_locations=[os.path.dirname(path)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
        mod.rt_hip.init(0)
    return sys.modules[name].rt_hip


def listed():
    return [
        # the smallest call: one row through one projection with its bias, as a program's eager loop issues it
        {"name": "linear_row", "kind": "linear", "fmt": "q4k", "m": 1, "n": 3072, "k": 3072, "bias": True},
        # GGUF Q4_0 weights at a small decode batch (4 rows), 4096-wide layers
        {"name": "layer_q4_0_m4", "kind": "layer", "fmt": "q4_0", "m": 4, "hidden": 4096, "kv": 1024, "ffn": 11008,
         "layers": 2},
        # speculative verify: 8 rows through Llama-3.2-3B's Q4_K projections
        {"name": "layer_verify_m8", "kind": "layer", "fmt": "q4k", "m": 8, "hidden": 3072, "kv": 1024, "ffn": 8192,
         "layers": 4},
        # the decode loop of the fused launches: Llama-3.2-3B, Q4_K_M mix, 1024 cached positions
        {"name": "token_llama3b", "kind": "token", "hidden": 3072, "heads": 24, "kv_heads": 8, "ffn": 8192,
         "layers": 28, "vocab": 128256, "wide": 14, "ctx": 1024},
        # the decode engine, one token with the logits on the host: the same model at another position
        {"name": "engine_llama3b", "kind": "engine", "arch": "llama", "hidden": 3072, "heads": 24, "kv_heads": 8,
         "head_dim": 128, "ffn": 8192, "layers": 28, "vocab": 128256, "wide": 14, "ctx": 777, "batch": 1},
        # the engine verifying five tokens at once: Gemma-3-4B's layers (12 of 34, a shorter vocabulary: the
        # upload of all of it would take longer than everything else here)
        {"name": "engine_gemma_batch5", "kind": "engine", "arch": "gemma3", "hidden": 2560, "heads": 8,
         "kv_heads": 4, "head_dim": 256, "ffn": 10240, "layers": 12, "vocab": 65536, "wide": 0, "ctx": 1100,
         "batch": 5},
        # prefill of a 512-token prompt, Llama-3.2-3B's Q4_K projections
        {"name": "prefill_q4k_512", "kind": "layer", "fmt": "q4k", "m": 512, "hidden": 3072, "kv": 1024,
         "ffn": 8192, "layers": 1},
        # prefill of an odd prompt on BF16 weights, hidden 1152 and ffn 6912 (Gemma-3-1B's)
        {"name": "prefill_bf16_333", "kind": "layer", "fmt": "bf16", "m": 333, "hidden": 1152, "kv": 256,
         "ffn": 6912, "layers": 1},
        # FLUX at 1024 x 1024: 4096 image and 512 text tokens
        {"name": "flux_4608", "kind": "flux", "m": 4608, "hidden": 3072, "a_bf16": True},
        # FLUX attention at 1024 x 1024: 4096 image and 256 text tokens
        {"name": "attention_4352", "kind": "attention", "t": 4352, "heads": 24, "head_dim": 128},
        # the largest decode projection: a 262144-token BF16 lm_head and its argmax
        {"name": "lm_head_262144", "kind": "lm_head", "n": 262144, "k": 1152},
        # loading: an MLP weight encoded to Q4_K and widened again
        {"name": "quantize_mlp", "kind": "quantize", "n": 8192, "k": 3072},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "layer", "layer", "layer", "token", "engine", "flux", "attention", "attention",
                       "lm_head", "quantize"])
    if kind == "linear":
        fmt = rng.choice(["q4k", "bf16", "q4_0", "q4mat"])
        return {"kind": kind, "fmt": fmt, "m": _log_int(rng, 1, 700), "n": _log_int(rng, 700, 12288),
                "k": 256 * rng.randint(4, 40), "bias": rng.random() < 0.5}
    if kind == "layer":
        fmt = rng.choice(["q4k", "q4k", "bf16", "q4_0", "q4mat", "q6k", "q8"])
        m = 1 if fmt in ("q6k", "q8") else rng.choice([rng.randint(1, 8), _log_int(rng, 9, 1024)])
        hidden = 256 * rng.randint(4, 16)
        if fmt == "bf16" and rng.random() < 0.5:
            hidden = 128 * rng.randint(7, 24)
        ffn = 256 * (rng.randint(12, 32) if fmt in ("q6k", "q8") else rng.randint(12, 44))
        return {"kind": kind, "fmt": fmt, "m": m, "hidden": hidden, "kv": 64 * rng.randint(4, 20), "ffn": ffn,
                "layers": rng.randint(2, 4) if m <= 8 else 1}
    if kind == "token":
        kv = rng.choice([4, 8])
        heads = kv * rng.choice([2, 3, 4])
        layers = rng.randint(4, 28)
        return {"kind": kind, "hidden": 128 * heads, "heads": heads, "kv_heads": kv, "ffn": 256 * rng.randint(12, 32),
                "layers": layers, "vocab": _log_int(rng, 20000, 128256), "wide": rng.randint(0, layers // 2),
                "ctx": _log_int(rng, 16, 4000)}
    if kind == "engine":
        arch = rng.choice(["llama", "gemma3"])
        d = 256 if arch == "gemma3" else rng.choice([64, 128])
        kv = rng.choice([2, 4] if d == 256 else [4, 8])
        layers = rng.randint(4, 12)
        return {"kind": kind, "arch": arch, "hidden": 256 * rng.randint(6, 12), "heads": kv * rng.choice([2, 3, 4]),
                "kv_heads": kv, "head_dim": d, "ffn": 256 * rng.randint(12, 40), "layers": layers,
                "vocab": _log_int(rng, 16000, 65536), "wide": 0 if arch == "gemma3" else rng.randint(0, layers // 2),
                "ctx": _log_int(rng, 16, 3000), "batch": rng.choice([1, 1, rng.randint(2, 8)])}
    if kind == "flux":
        return {"kind": kind, "m": _log_int(rng, 300, 4608), "hidden": 256 * rng.randint(4, 12),
                "a_bf16": rng.random() < 0.5}
    if kind == "attention":
        return {"kind": kind, "t": _log_int(rng, 100, 4352), "heads": rng.randint(4, 24),
                "head_dim": rng.choice([128, 128, 128, 64, 8 * rng.randint(4, 16)])}
    if kind == "lm_head":
        return {"kind": kind, "n": _log_int(rng, 30000, 262144), "k": 128 * rng.randint(6, 20)}
    return {"kind": "quantize", "n": _log_int(rng, 500, 8192), "k": 256 * rng.randint(4, 16)}


# ------------------------------------------------------------------- formats --

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _q4k_blocks(w):
    """Q4_K blocks of w [n, k]: per 32 values scale = (max - min) / 15 and min, both 6-bit against the
    super-block's largest (a simple encoder: the distributions are those of real blocks)."""
    n, k = w.shape
    s = w.reshape(n * (k // 256), 8, 32)
    lo = (-s.amin(-1)).clamp_min(0)
    sc = (s.amax(-1) + lo) / 15
    d, dm = (sc.amax(-1) / 63).half(), (lo.amax(-1) / 63).half()
    df, dmf = d.float()[:, None], dm.float()[:, None]
    sv = torch.where(df > 0, torch.round(sc / df.clamp_min(1e-30)), torch.zeros_like(sc)).clamp(0, 63)
    mv = torch.where(dmf > 0, torch.round(lo / dmf.clamp_min(1e-30)), torch.zeros_like(lo)).clamp(0, 63)
    step = (df * sv)[..., None]
    q = torch.where(step > 0, torch.round((s + (dmf * mv)[..., None]) / step.clamp_min(1e-30)), torch.zeros_like(s))
    q = q.clamp(0, 15).to(torch.uint8).reshape(-1, 4, 2, 32)
    sv, mv = sv.to(torch.uint8), mv.to(torch.uint8)
    out = torch.empty((n * (k // 256), 144), dtype=torch.uint8, device=w.device)
    out[:, 0:2] = d[:, None].view(torch.uint8)
    out[:, 2:4] = dm[:, None].view(torch.uint8)
    out[:, 4:8] = sv[:, :4] | ((sv[:, 4:] >> 4) << 6)
    out[:, 8:12] = mv[:, :4] | ((mv[:, 4:] >> 4) << 6)
    out[:, 12:16] = (sv[:, 4:] & 15) | ((mv[:, 4:] & 15) << 4)
    out[:, 16:] = (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(-1, 128)
    return out.reshape(-1)


def _q4k_values(blocks, n, k):
    b = blocks.reshape(-1, 144)
    d = b[:, 0:2].contiguous().view(torch.float16).double()
    dm = b[:, 2:4].contiguous().view(torch.float16).double()
    p = b[:, 4:16].to(torch.int32)
    sv = torch.cat([p[:, 0:4] & 63, (p[:, 8:12] & 15) | ((p[:, 0:4] >> 6) << 4)], 1).double()
    mv = torch.cat([p[:, 4:8] & 63, (p[:, 8:12] >> 4) | ((p[:, 4:8] >> 6) << 4)], 1).double()
    qs = b[:, 16:].reshape(-1, 4, 32)
    q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
    return ((d * sv)[..., None] * q - (dm * mv)[..., None]).reshape(n, k)


def _q4_0_blocks(w):
    """GGUF Q4_0 blocks: d = absmax / 7 in f16, values d (q - 8)."""
    n, k = w.shape
    b = w.reshape(n * (k // 32), 32)
    d = (b.abs().amax(-1) / 7).half()
    q = (torch.round(b / d.float()[:, None].clamp_min(1e-30)).clamp(-8, 7) + 8).to(torch.uint8)
    out = torch.empty((b.shape[0], 18), dtype=torch.uint8, device=w.device)
    out[:, 0:2] = d[:, None].view(torch.uint8)
    out[:, 2:] = q[:, :16] | (q[:, 16:] << 4)
    return out.reshape(-1)


def _q4_0_values(blocks, n, k):
    b = blocks.reshape(-1, 18)
    d = b[:, 0:2].contiguous().view(torch.float16).double()
    q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8
    return (d * q).reshape(n, k)


def _q4mat_parts(w):
    """Q4Mat: packed signed nibbles (even element low) and one f32 scale per 32 values."""
    b = w.reshape(-1, 32)
    s = b.abs().amax(-1) / 7
    q = torch.round(b / s[:, None].clamp_min(1e-30)).clamp(-8, 7).to(torch.int32) & 15
    packed = (q[:, 0::2] | (q[:, 1::2] << 4)).to(torch.uint8).reshape(-1)
    return packed, s


def _q4mat_values(packed, scales, n, k):
    p = packed.reshape(-1, 16).to(torch.int32)
    q = torch.stack([p & 15, p >> 4], -1).reshape(-1, 32)
    q = torch.where(q > 7, q - 16, q).double()
    return (q * scales.double()[:, None]).reshape(n, k)


def _q6k_blocks(g, n, k):
    """GGUF Q6_K blocks of about N(0, 0.02): random quants and scales, d = 2^-14."""
    nb = n * (k // 256)
    b = torch.randint(0, 256, (nb, 210), dtype=torch.uint8, device="cuda", generator=g)
    b[:, 192:208] = torch.randint(10, 28, (nb, 16), dtype=torch.uint8, device="cuda", generator=g)
    b[:, 208], b[:, 209] = 0x00, 0x04
    return b.reshape(-1)


def _q6k_values(blocks, n, k):
    """The weights as they are used: decoded, then widened to bf16."""
    b = blocks.reshape(-1, 210).to(torch.int32)
    ql, qh, sc = b[:, :128].reshape(-1, 2, 64), b[:, 128:192].reshape(-1, 2, 32), b[:, 192:208].reshape(-1, 2, 8)
    q = torch.stack([(ql[..., :32] & 15) | ((qh & 3) << 4), (ql[..., 32:] & 15) | (((qh >> 2) & 3) << 4),
                     (ql[..., :32] >> 4) | (((qh >> 4) & 3) << 4), (ql[..., 32:] >> 4) | ((qh >> 6) << 4)], 2) - 32
    sc = torch.where(sc > 127, sc - 256, sc).reshape(-1, 2, 4, 2, 1)
    v = (q.reshape(-1, 2, 4, 2, 16) * sc).float() * 2.0 ** -14
    return v.to(torch.bfloat16).double().reshape(n, k)


def _bf16_bits(w):
    return w.to(torch.bfloat16).view(torch.int16)


def _weight(g, fmt, n, k):
    """Device bytes of a random weight: a tensor (q4mat: the packed bytes and the scales)."""
    if fmt == "q6k":
        return _q6k_blocks(g, n, k)
    w = torch.randn((n, k), device="cuda", generator=g) * 0.02
    if fmt == "bf16":
        return _bf16_bits(w)
    return {"q4k": _q4k_blocks, "q8": _q4k_blocks, "q4_0": _q4_0_blocks, "q4mat": _q4mat_parts}[fmt](w)


def _values(fmt, w, n, k):
    if fmt == "bf16":
        return w.view(torch.bfloat16).double().reshape(n, k)
    if fmt == "q4mat":
        return _q4mat_values(w[0], w[1], n, k)
    return {"q4k": _q4k_values, "q8": _q4k_values, "q4_0": _q4_0_values, "q6k": _q6k_values}[fmt](w, n, k)


def _weight_bytes(fmt, n, k):
    return n * k * {"q4k": 144 / 256, "q8": 144 / 256, "q4_0": 18 / 32, "q4mat": 20 / 32, "q6k": 210 / 256, "bf16": 2}[fmt]


def _device_form(rt, fmt, w, n, k):
    """What the entry points of `fmt` read: made once at load."""
    if fmt == "q4mat":
        return rt.q4mat_upload(w[0].cpu().numpy(), w[1].cpu().numpy(), n, k)
    if fmt == "q8":
        return rt.q4k_tile(w, n, k)
    return rt.q6k_tile(w, n, k) if fmt == "q6k" else w


def _linear(rt, fmt, w, x, n, k, bias, y):
    if fmt == "q8":
        return rt.gemv_q4k_q8(w, x, n, k, tiled=True, y=y)
    if fmt == "q6k":
        return rt.gemv_q6k_tiled(w, x, n, k, y=y)
    code = {"q4k": rt.Q4K, "bf16": rt.BF16, "q4_0": rt.Q4_0, "q4mat": rt.Q4MAT}[fmt]
    return rt.linear_forward(code, w, x, n, k, bias=bias, y=y)


def _exact_linear(fmt, w, x, n, k):
    v = _values(fmt, w, n, k)
    if fmt != "q8":
        return x.double() @ v.T
    # activations to int8 per 32 values, the minimum's term on the unquantized sums
    b = x.reshape(-1, 32)
    scale = b.abs().amax(-1, keepdim=True) / 127.0
    r = b * (1.0 / scale)
    q = torch.sign(r) * torch.floor(r.abs() + 0.5)
    xq = (q.clamp(-128, 127).double() * scale.double()).reshape(-1)
    z = w.reshape(-1, 144).clone()
    z[:, 16:] = 0
    mins = _q4k_values(z.reshape(-1), n, k)
    return ((v - mins) @ xq + mins @ x.double().reshape(-1)).reshape(1, n)


def _capture(fn):
    """fn's launches as one graph (run once eagerly first: workspaces grow outside a capture)."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        fn()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn()
    return graph


# ----------------------------------------------------------------- inputs --
# _inputs(case, seed): the data both prepare() and exact() start from.

def _projections(case):
    h, kv, f = case["hidden"], case["kv"], case["ffn"]
    return [("q", h, h, "attn"), ("k", kv, h, "attn"), ("v", kv, h, "attn"), ("o", h, h, "o"), ("gate", f, h, "mlp"),
            ("up", f, h, "mlp"), ("down", h, f, "act")]


def _layer_inputs(case, seed):
    g = _gen(seed)
    m = case["m"]
    for _ in range(case["layers"]):
        x = {nm: torch.randn((m, case["ffn"] if nm == "act" else case["hidden"]), device="cuda", generator=g)
             for nm in ("attn", "o", "mlp", "act")}
        for _, n, k, nm in _projections(case):
            yield n, k, x[nm], _weight(g, case["fmt"], n, k)


def _flux_shapes(case):
    h = case["hidden"]
    return [(3 * h, h), (4 * h, h), (h, 4 * h)]


def _flux_inputs(case, seed):
    g = _gen(seed)
    for n, k in _flux_shapes(case):
        a = torch.randn((case["m"], k), device="cuda", generator=g)
        yield (n, k, a.to(torch.bfloat16) if case["a_bf16"] else a, _weight(g, "q4k", n, k),
               0.1 * torch.randn((n,), device="cuda", generator=g))


def _attention_inputs(case, seed):
    g = _gen(seed)
    w = case["heads"] * case["head_dim"]
    q, k, v = (torch.randn((case["t"], w), device="cuda", generator=g) for _ in range(3))
    return q * 1.5, k * 1.5, v


def _inv_freq(d, theta):
    return torch.tensor([1.0 / theta ** (2.0 * i / d) for i in range(d // 2)], dtype=torch.float32, device="cuda")


def _model(case, seed):
    """Weights of a token / engine case: per layer a dict of (format, bytes, n, k), the norms, caches and head."""
    g = _gen(seed)
    gemma = case.get("arch") == "gemma3"
    h, f, d = case["hidden"], case["ffn"], case.get("head_dim", 128)
    nq, nkv = case["heads"] * d, case["kv_heads"] * d

    def norm(n):
        return (0.0 if gemma else 1.0) + 0.1 * torch.randn((n,), device="cuda", generator=g)

    layers = []
    for li in range(case["layers"]):
        vf = "bf16" if li < case["wide"] else "q4k"
        lay = {nm: (fm, _weight(g, fm, n, k), n, k)
               for nm, fm, n, k in [("q", "q4k", nq, h), ("k", "q4k", nkv, h), ("v", vf, nkv, h), ("o", "q4k", h, nq),
                                    ("gate", "q4k", f, h), ("up", "q4k", f, h), ("down", vf, h, f)]}
        lay["attn_norm"], lay["ffn_norm"] = norm(h), norm(h)
        if gemma:
            lay["post_attn_norm"], lay["post_ffn_norm"] = norm(h), norm(h)
            lay["q_norm"], lay["k_norm"] = norm(d), norm(d)
        lay["kv"] = torch.randn((2, case["ctx"], nkv), device="cuda", generator=g)
        if gemma:  # cached in f16
            lay["kv"] = lay["kv"].half().float()
        layers.append(lay)
    embed = _bf16_bits(0.5 * torch.randn((case["vocab"], h), device="cuda", generator=g))
    head = ("bf16", embed, case["vocab"], h) if gemma else ("q4k", _weight(g, "q4k", case["vocab"], h), case["vocab"], h)
    tokens = torch.randint(0, case["vocab"], (case.get("batch", 1),), device="cuda", generator=g)
    return {"layers": layers, "embed": embed, "out_norm": norm(h), "head": head, "tokens": tokens.cpu().tolist()}


_GEMMA = {"rope_theta": 1e6, "rope_theta_local": 1e4, "rope_freq_scale": 0.125, "rope_freq_scale_local": 1.0,
          "sliding_window": 1024, "global_every": 6, "attn_scale": 1.0 / 16.0}
_LLAMA_THETA = 500000.0


def _exact_model(case, model):
    """Logits [batch, vocab] and the new cache rows [layers, 2, batch, kv] in float64."""
    gemma = case.get("arch") == "gemma3"
    d = case.get("head_dim", 128)
    nq, nkv, ctx = case["heads"], case["kv_heads"], case["ctx"]
    eps = 1e-6 if gemma else 1e-5
    add = 1.0 if gemma else 0.0

    def norm(x, gamma):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * (gamma.double() + add)

    def mm(x, w):
        return x @ _values(w[0], w[1], w[2], w[3]).T

    tok = torch.tensor(model["tokens"], device="cuda")
    b = tok.numel()
    pos = torch.arange(ctx, ctx + b, device="cuda", dtype=torch.float64)
    x = model["embed"].view(torch.bfloat16)[tok].double() * (float(np.float32(math.sqrt(case["hidden"]))) if gemma else 1.0)
    rows = []
    for li, lay in enumerate(model["layers"]):
        glob = gemma and li % _GEMMA["global_every"] == _GEMMA["global_every"] - 1
        n1 = norm(x, lay["attn_norm"])
        q, k, v = mm(n1, lay["q"]).view(b, nq, d), mm(n1, lay["k"]).view(b, nkv, d), mm(n1, lay["v"]).view(b, nkv, d)
        if gemma:
            q, k = norm(q, lay["q_norm"]), norm(k, lay["k_norm"])
            theta = _GEMMA["rope_theta" if glob else "rope_theta_local"]
            fs = _GEMMA["rope_freq_scale" if glob else "rope_freq_scale_local"]
            inv = torch.tensor([fs / theta ** (2.0 * i / d) for i in range(d // 2)], dtype=torch.float64, device="cuda")
        else:
            inv = _inv_freq(d, _LLAMA_THETA).double()
        ang = (pos[:, None] * inv)[:, None, :]
        cos, sin = torch.cos(ang), torch.sin(ang)

        def rope(t):
            if gemma:
                p, r = t[..., : d // 2], t[..., d // 2:]
                return torch.cat([p * cos - r * sin, p * sin + r * cos], -1)
            p, r = t[..., 0::2], t[..., 1::2]
            return torch.stack([p * cos - r * sin, p * sin + r * cos], -1).flatten(-2)

        q, k = rope(q), rope(k)
        if gemma:
            k, v = k.half().double(), v.half().double()
        rows.append(torch.stack([k.reshape(b, -1), v.reshape(b, -1)]))
        kc = torch.cat([lay["kv"][0].double(), k.reshape(b, -1)]).view(-1, nkv, d).repeat_interleave(nq // nkv, 1)
        vc = torch.cat([lay["kv"][1].double(), v.reshape(b, -1)]).view(-1, nkv, d).repeat_interleave(nq // nkv, 1)
        s = (q.transpose(0, 1) @ kc.permute(1, 2, 0)) * (_GEMMA["attn_scale"] if gemma else 1.0 / math.sqrt(d))
        at = torch.arange(kc.shape[0], device="cuda")[None, :]
        mine = torch.arange(ctx, ctx + b, device="cuda")[:, None]
        hide = at > mine
        if gemma and not glob:
            hide = hide | (at <= mine - _GEMMA["sliding_window"])
        p = torch.softmax(s.masked_fill(hide, -math.inf), -1)
        ao = mm((p @ vc.transpose(0, 1)).transpose(0, 1).reshape(b, nq * d), lay["o"])
        x = x + (norm(ao, lay["post_attn_norm"]) if gemma else ao)
        n2 = norm(x, lay["ffn_norm"])
        gt, up = mm(n2, lay["gate"]), mm(n2, lay["up"])
        act = torch.nn.functional.gelu(gt, approximate="tanh") if gemma else torch.nn.functional.silu(gt)
        dn = mm(act * up, lay["down"])
        x = x + (norm(dn, lay["post_ffn_norm"]) if gemma else dn)
    return mm(norm(x, model["out_norm"]), model["head"]), x, torch.stack(rows)


# ---------------------------------------------------------------- prepare --

def _prepare_token(rt, case, seed):
    model = _model(case, seed)
    h, f, ctx, hd = case["hidden"], case["ffn"], case["ctx"], 128
    nq, nkv = case["heads"], case["kv_heads"]
    kv = nkv * hd
    new = lambda n: torch.empty((1, n), device="cuda")  # noqa: E731
    layers = []
    for lay in model["layers"]:
        cache = torch.empty((2, ctx + 1, kv), device="cuda")
        cache[:, :ctx] = lay["kv"]
        out = {"kc": cache[0], "vc": cache[1], "g1": lay["attn_norm"], "g2": lay["ffn_norm"], "wide": lay["v"][0] == "bf16"}
        for nm in ("q", "k", "v", "o", "gate", "up", "down"):
            fm, w, n, k = lay[nm]
            out[nm] = rt.q4k_tile(w, n, k) if fm == "q4k" else w
        layers.append(out)
    head, gf = rt.q4k_tile(model["head"][1], case["vocab"], h), model["out_norm"]
    embed = model["embed"].view(torch.bfloat16)[torch.tensor(model["tokens"], device="cuda")].float()
    which = torch.zeros(1, dtype=torch.int64, device="cuda")
    resid, q, attn, gate, up, logits = new(h), new(h), new(h), new(f), new(f), new(case["vocab"])
    inv, eps, scale = _inv_freq(hd, _LLAMA_THETA), 1e-5, 1.0 / math.sqrt(hd)

    def step():
        torch.index_select(embed, 0, which, out=resid)
        for lay in layers:
            kr, vr = lay["kc"][ctx:ctx + 1], lay["vc"][ctx:ctx + 1]
            if lay["wide"]:
                rt.gemv_q4k_tiled_bf16_rmsnorm([lay["q"], lay["k"]], [h, kv], lay["v"], kv, resid, lay["g1"], eps, h,
                                               ys=[q, kr], yb=vr, rope=(inv, ctx, hd, 0x3))
            else:
                rt.gemv_q4k_tiled_rmsnorm_rope([lay["q"], lay["k"], lay["v"]], resid, lay["g1"], eps, [h, kv, kv], h, inv,
                                               ctx, hd, 0x3, ys=[q, kr, vr])
            rt.attention_decode(q, lay["kc"], lay["vc"], ctx + 1, nq, nkv, scale, out=attn)
            rt.gemv_q4k_tiled_residual(lay["o"], attn, resid, h, h)
            rt.gemv_q4k_tiled_rmsnorm_multi([lay["gate"], lay["up"]], resid, lay["g2"], eps, [f, f], h, ys=[gate, up])
            rt.gemv_swiglu_residual(rt.BF16 if lay["wide"] else rt.Q4K, lay["down"], gate, up, resid, h, f)
        rt.gemv_q4k_tiled_rmsnorm_multi([head], resid, gf, eps, [case["vocab"]], h, ys=[logits])

    outs = {"logits": logits, "x": resid, "k": [lay["kc"][ctx:ctx + 1] for lay in layers],
            "v": [lay["vc"][ctx:ctx + 1] for lay in layers]}
    return {"graph": _capture(step), "outs": outs, "keep": (layers, head, gf, embed, which, q, attn, gate, up, inv)}


def _prepare_engine(rt, case, seed):
    model = _model(case, seed)
    gemma = case["arch"] == "gemma3"
    cfg = dict(arch=rt.ARCH_GEMMA3 if gemma else rt.ARCH_LLAMA, n_layers=case["layers"], hidden=case["hidden"],
               n_heads=case["heads"], n_kv_heads=case["kv_heads"], head_dim=case["head_dim"], ffn=case["ffn"],
               vocab=case["vocab"], max_seq=case["ctx"] + 64, norm_eps=1e-6 if gemma else 1e-5,
               rope_theta=_LLAMA_THETA, rope_theta_local=0.0, rope_freq_scale=1.0, rope_freq_scale_local=1.0,
               rope_half=0, sliding_window=0, global_every=0, attn_scale=0.0,
               embed_scale=math.sqrt(case["hidden"]) if gemma else 0.0, kv_f16=1 if gemma else 0,
               max_batch=case["batch"] if case["batch"] > 1 else 0)
    if gemma:
        cfg.update(_GEMMA, rope_half=1)
    dec = rt.Decoder(**cfg)
    fmts = {"q4k": rt.Q4K, "bf16": rt.BF16}
    names = {"q": rt.T_Q, "k": rt.T_K, "v": rt.T_V, "o": rt.T_O, "gate": rt.T_GATE, "up": rt.T_UP, "down": rt.T_DOWN}
    norms = {"attn_norm": rt.T_ATTN_NORM, "ffn_norm": rt.T_FFN_NORM, "post_attn_norm": rt.T_POST_ATTN_NORM,
             "post_ffn_norm": rt.T_POST_FFN_NORM, "q_norm": rt.T_Q_NORM, "k_norm": rt.T_K_NORM}
    for li, lay in enumerate(model["layers"]):
        for nm, t in names.items():
            dec.set(li, t, fmts[lay[nm][0]], lay[nm][1].cpu().numpy())
        for nm, t in norms.items():
            if nm in lay:
                dec.set(li, t, rt.F32, lay[nm].cpu().numpy())
        kv = lay["kv"].cpu().numpy()
        dec.set_kv(li, kv[0], kv[1], case["ctx"])
    embed = model["embed"].cpu().numpy()
    dec.set(-1, rt.T_EMBED, rt.BF16, embed)
    dec.set(-1, rt.T_OUTPUT_NORM, rt.F32, model["out_norm"].cpu().numpy())
    dec.set(-1, rt.T_LM_HEAD, fmts[model["head"][0]], embed if gemma else model["head"][1].cpu().numpy())
    return {"dec": dec, "tokens": model["tokens"], "pos": case["ctx"]}


def prepare(case, seed):
    rt = _rt()
    kind = case["kind"]
    if kind == "linear":
        g = _gen(seed)
        m, n, k = case["m"], case["n"], case["k"]
        x = torch.randn((m, k), device="cuda", generator=g)
        w = _device_form(rt, case["fmt"], _weight(g, case["fmt"], n, k), n, k)
        bias = 0.1 * torch.randn((n,), device="cuda", generator=g) if case["bias"] else None
        return {"fn": lambda: _linear(rt, case["fmt"], w, x, n, k, bias, None)}
    if kind == "layer":
        items = [(x, _device_form(rt, case["fmt"], w, n, k), n, k, torch.empty((case["m"], n), device="cuda"))
                 for n, k, x, w in _layer_inputs(case, seed)]

        def layer():
            return [_linear(rt, case["fmt"], w, x, n, k, None, y) for x, w, n, k, y in items]

        if case["m"] > 8:
            return {"fn": layer}
        return {"graph": _capture(layer), "outs": [it[4] for it in items], "keep": items}
    if kind == "token":
        return _prepare_token(rt, case, seed)
    if kind == "engine":
        return _prepare_engine(rt, case, seed)
    if kind == "flux":
        items = [(a, w, n, k, bias, torch.empty((case["m"], n), device="cuda"))
                 for n, k, a, w, bias in _flux_inputs(case, seed)]
        return {"fn": lambda: [rt.gemm(rt.Q4K, a, w, n, k, bias=bias, c=c) for a, w, n, k, bias, c in items]}
    if kind == "attention":
        q, k, v = _attention_inputs(case, seed)
        out = torch.empty_like(q)
        return {"fn": lambda: rt.flux_attention(q, k, v, case["heads"], case["head_dim"], out=out)}
    if kind == "lm_head":
        g = _gen(seed)
        n, k = case["n"], case["k"]
        w, x = _weight(g, "bf16", n, k), torch.randn((1, k), device="cuda", generator=g)
        y = torch.empty((1, n), device="cuda")
        return {"fn": lambda: rt.gemv_bf16_argmax(w, x, n, k, y=y)}
    g = _gen(seed)
    n, k = case["n"], case["k"]
    w = torch.randn((n, k), device="cuda", generator=g) * 0.02

    def load():
        blocks = rt.quantize_q4k(w)
        return blocks, rt.dequant_q4k(blocks, n, k, bf16=True)

    return {"fn": load}


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outs"]
    if "dec" in state:
        if len(state["tokens"]) == 1:
            return state["dec"].step(state["tokens"][0], state["pos"], argmax=True)
        return state["dec"].step_batch(state["tokens"], state["pos"])
    return state["fn"]()


# ------------------------------------------------------- work and accuracy --

def _mm_work(fmt, m, n, k, x=True):
    return np.array([_weight_bytes(fmt, n, k) + (4 * m * k if x else 0) + 4 * m * n, 2 * m * n * k], dtype=float)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        t = _mm_work(case["fmt"], case["m"], case["n"], case["k"])
    elif kind == "layer":
        t = case["layers"] * sum(_mm_work(case["fmt"], case["m"], n, k, nm in ("q", "o", "gate", "down"))
                                 for nm, n, k, _ in _projections(case))
    elif kind in ("token", "engine"):
        d, b = case.get("head_dim", 128), case.get("batch", 1)
        h, f, nq, nkv = case["hidden"], case["ffn"], case["heads"] * d, case["kv_heads"] * d
        gemma = case.get("arch") == "gemma3"
        t = np.zeros(2)
        for li in range(case["layers"]):
            vf = "bf16" if li < case["wide"] else "q4k"
            seen = case["ctx"]
            if gemma and li % _GEMMA["global_every"] != _GEMMA["global_every"] - 1:
                seen = min(seen, _GEMMA["sliding_window"] - 1)
            for fm, n, k in [("q4k", nq, h), ("q4k", nkv, h), (vf, nkv, h), ("q4k", h, nq), ("q4k", f, h),
                             ("q4k", f, h), (vf, h, f)]:
                t += [_weight_bytes(fm, n, k), 2 * b * n * k]
            t += [2 * (seen + b) * nkv * (2 if gemma else 4), 4 * b * (seen + b) * nq]
        t += [_weight_bytes("bf16" if gemma else "q4k", case["vocab"], h) + b * (4 * case["vocab"] + 2 * h),
              2 * b * case["vocab"] * h]
    elif kind == "flux":
        t = sum(_mm_work("q4k", case["m"], n, k, False) + [(2 if case["a_bf16"] else 4) * case["m"] * k, 0]
                for n, k in _flux_shapes(case))
    elif kind == "attention":
        w = case["heads"] * case["head_dim"]
        t = np.array([16 * case["t"] * w, 4 * case["t"] * case["t"] * w], dtype=float)
    elif kind == "lm_head":
        t = _mm_work("bf16", 1, case["n"], case["k"])
    else:
        nk = case["n"] * case["k"]
        t = np.array([nk * (4 + 144 / 256 + 2), 0], dtype=float)
    return {"bytes": float(t[0]), "flops": float(t[1])}


def tolerance(case):
    """About four times what the path is off a float64 result (measured at the listed and drawn cases)."""
    kind = case["kind"]
    if kind == "quantize":
        return "exact"  # bytes and bf16 bits
    if kind == "flux" or (kind in ("linear", "layer") and case["m"] > 8):
        return {"rel": 1e-2, "max": 0.06}  # operands rounded to bf16: 2.4e-3
    if kind in ("token", "engine"):
        return {"rel": 3e-5, "max": 4e-4, "differ": 0.0}  # f32 through all layers: 7.5e-6
    if kind == "attention":
        return {"rel": 6e-6, "max": 2e-4}  # f32 scores and sums: 1.6e-6
    return {"rel": 3e-6, "max": 4e-5, "differ": 0.0}  # f32 sums: 7e-7


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        g = _gen(seed)
        m, n, k = case["m"], case["n"], case["k"]
        x = torch.randn((m, k), device="cuda", generator=g)
        y = _exact_linear(case["fmt"], _weight(g, case["fmt"], n, k), x, n, k)
        return y + (0.1 * torch.randn((n,), device="cuda", generator=g)).double() if case["bias"] else y
    if kind == "layer":
        return [_exact_linear(case["fmt"], w, x, n, k) for n, k, x, w in _layer_inputs(case, seed)]
    if kind == "token":
        logits, x, rows = _exact_model(case, _model(case, seed))
        return {"logits": logits, "x": x, "k": list(rows[:, 0]), "v": list(rows[:, 1])}
    if kind == "engine":
        logits = _exact_model(case, _model(case, seed))[0]
        return (logits[0], None) if case["batch"] == 1 else logits
    if kind == "flux":
        return [a.double() @ _values("q4k", w, n, k).T + bias.double() for n, k, a, w, bias in _flux_inputs(case, seed)]
    if kind == "attention":
        q, k, v = _attention_inputs(case, seed)
        d = case["head_dim"]
        out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
        for h in range(case["heads"]):
            c = slice(h * d, (h + 1) * d)
            p = torch.softmax(q[:, c].double() @ k[:, c].double().T / math.sqrt(d), -1)
            out[:, c] = p @ v[:, c].double()
        return out
    if kind == "lm_head":
        g = _gen(seed)
        n, k = case["n"], case["k"]
        w, x = _weight(g, "bf16", n, k), torch.randn((1, k), device="cuda", generator=g)
        return _exact_linear("bf16", w, x, n, k), None, None
    return None
