"""Performance cases: the work a program gives this library, through its public entry points.

What a user of the library runs, in the order it happens in a serving process:
loading weights (quantize-on-load), prefill (seq > 1) projections on int4 weights, batch-1
decode projections in both precisions, small-batch decode projections, the lm_head, and
whole greedy decode steps.  Shapes are the Llama-3.2-1B / 3.2-3B / 3.1-8B layer shapes the
benchmark names, weights N(0, 0.02) int4 group-quantized, activations N(0, 1) with 0.5% of
the channels at 20 sigma (the benchmark's distributions).

A case is a dict; `kind` selects the path:
  gemv     one projection of one token (gpu_layer.project)
  layer    the seven projections of one layer for one token, Q/K/V (and gate/up) grouped
  batch    the seven projections of one layer for m <= 16 tokens, W4A8, per-row quantization
  head     the lm_head for m <= 16 tokens, W4A8
  prefill  the seven projections of one layer for m prompt tokens (gemm_w4a16_ws)
  load     quantize-on-load of the seven matrices of one layer
  decode   one greedy token through a whole decoder (DecodeModel, captured HIP graph)
"""
from __future__ import annotations

import math

import numpy as np
import torch

from nve_amd import hip_kernels as hk
from nve_amd.decode import DecodeModel, ModelShape
from nve_amd.gpu_layer import GpuW4, project

DEV = "cuda"
VOCAB = 128256
# hidden, query rows, key/value rows, ffn
DIMS = {"1b": (2048, 2048, 512, 8192), "3b": (3072, 3072, 1024, 8192), "8b": (4096, 4096, 1024, 14336)}
DT = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def dims(case):
    """hidden, query rows, key/value rows and ffn of the case's layer; drawn cases have an ffn of their own."""
    h, q, kv, f = DIMS[case["shape"]]
    return h, q, kv, case.get("ffn", f)


def mats(case):
    """(name, N, K) of a layer's seven projections."""
    h, q, kv, f = dims(case)
    return [("q", q, h), ("k", kv, h), ("v", kv, h), ("o", h, q), ("gate", f, h), ("up", f, h), ("down", h, f)]


def listed():
    return [
        # the smallest call: one 1B q_proj for one token, activations quantized then multiplied
        {"name": "gemv_1b_w4a8", "kind": "gemv", "n": 2048, "k": 2048, "precision": "w4a8", "dtype": "f16"},
        # one decode token through an 8B layer's projections in W4A16, bf16 activations
        {"name": "layer_8b_w4a16", "kind": "layer", "shape": "8b", "precision": "w4a16", "dtype": "bf16"},
        # small-batch decode: eight sequences through an 8B layer, one bf16 scale per row
        {"name": "batch_8b_m8", "kind": "batch", "shape": "8b", "m": 8, "per_token": True},
        # the logits of eight sequences (8B lm_head, group scales): ends every batched decode step
        {"name": "head_8b_m8", "kind": "head", "n": VOCAB, "k": 4096, "m": 8, "per_token": False},
        # a short prompt (one question) through an 8B layer
        {"name": "prefill_8b_m40", "kind": "prefill", "shape": "8b", "m": 40, "dtype": "f16", "awq": False},
        # a paragraph of odd length through a 3B layer, bf16
        {"name": "prefill_3b_m197", "kind": "prefill", "shape": "3b", "m": 197, "dtype": "bf16", "awq": False},
        # a medium prompt through an AWQ-quantized 8B layer
        {"name": "prefill_8b_m300_awq", "kind": "prefill", "shape": "8b", "m": 300, "dtype": "f16", "awq": True},
        # a page of text through an 8B layer
        {"name": "prefill_8b_m512", "kind": "prefill", "shape": "8b", "m": 512, "dtype": "f16", "awq": False},
        # a long prompt (one prefill chunk) through an 8B layer, bf16
        {"name": "prefill_8b_m2048", "kind": "prefill", "shape": "8b", "m": 2048, "dtype": "bf16", "awq": False},
        # loading one 8B layer of a bf16 checkpoint
        {"name": "load_8b_bf16", "kind": "load", "shape": "8b", "dtype": "bf16", "mode": "plain"},
        # loading one 3B layer of a bf16 checkpoint with AWQ scales (the k-quant search)
        {"name": "load_3b_awq", "kind": "load", "shape": "3b", "dtype": "bf16", "mode": "kquant"},
        # one greedy token through four layers of the 3B decoder and its head, one layer W4A16, 512 cached
        # positions (four, since through all 28 layers an int8 code that one rounding moved grows to 3% of
        # the last keys, and two correct results could no longer be told from wrong ones)
        {"name": "decode_3b_4_layers", "kind": "decode", "shape": "3b", "layers": 4, "context": 512, "w4a16": 0.3},
    ]


def _log(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "prefill", "prefill", "layer", "batch", "head", "gemv", "load", "decode"])
    shape, ffn = rng.choice(["1b", "3b", "8b"]), 128 * _log(rng, 24, 111)
    if kind == "prefill":
        return {"kind": kind, "shape": shape, "ffn": ffn, "m": _log(rng, 2, 2047),
                "dtype": rng.choice(["f16", "bf16"]), "awq": rng.random() < 0.25}
    if kind == "layer":
        p = rng.choice(["w4a16", "w4a8"])
        return {"kind": kind, "shape": shape, "ffn": ffn, "precision": p,
                "dtype": rng.choice(["f16", "bf16"])}
    if kind == "batch":
        return {"kind": kind, "shape": shape, "ffn": ffn, "m": rng.randint(2, 16),
                "per_token": rng.random() < 0.5}
    if kind == "head":
        return {"kind": kind, "n": _log(rng, 32000, VOCAB), "k": rng.choice([2048, 3072, 4096]),
                "m": rng.randint(1, 16), "per_token": rng.random() < 0.5}
    if kind == "gemv":
        return {"kind": kind, "n": _log(rng, 300, 20000), "k": 32 * _log(rng, 16, 448),
                "precision": rng.choice(["w4a16", "w4a8"]), "dtype": rng.choice(["f16", "bf16"])}
    if kind == "load":
        return {"kind": kind, "shape": shape, "ffn": ffn, "dtype": rng.choice(["f32", "bf16", "f16"]),
                "mode": rng.choice(["plain", "plain", "awq", "kquant"])}
    return {"kind": kind, "shape": "3b", "ffn": ffn, "layers": rng.randint(1, 4), "context": _log(rng, 64, 6000),
            "w4a16": rng.choice([0.0, 0.3, 1.0])}


# ---- inputs ----------------------------------------------------------------------------
class _Rand:
    """Seeded device random inputs; the same calls in the same order give the same tensors."""

    def __init__(self, seed: int):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def dense(self, n, k):
        return torch.randn((n, k), generator=self.g, device=DEV).mul_(0.02)

    def w4(self, n, k):
        """Packed int4 weights of an N(0, 0.02) matrix: nibbles u8 [n, k/2] (byte j of a
        32-block = element j | element j + 16 << 4), scales f32 [n, k/32]."""
        b = self.dense(n, k).view(n, k // 32, 32)
        s = b.abs().amax(-1) / 7
        q = b.div_(s[..., None]).round_().clamp_(-8, 7).add_(8).to(torch.uint8)
        return (q[..., :16] | (q[..., 16:] << 4)).reshape(n, k // 2).contiguous(), s.contiguous()

    def acts(self, m, k, dtype):
        x = torch.randn((m, k), generator=self.g, device=DEV)
        out = torch.rand(k, generator=self.g, device=DEV) < 0.005
        sign = torch.where(torch.rand(k, generator=self.g, device=DEV) < 0.5, -20.0, 20.0)
        return torch.where(out, sign, x).to(dtype)

    def awq(self, k):
        return torch.rand(k, generator=self.g, device=DEV).mul_(1.5).add_(0.5)

    def norm(self, n):
        return (1.0 + 0.1 * torch.randn(n, generator=self.g, device=DEV)).to(torch.bfloat16)


def _decode_parts(case, seed):
    """Shape, packed weights (Hugging Face names), per-layer importance and first token."""
    h, q, kv, f = dims(case)
    s = ModelShape(hidden=h, layers=case["layers"], heads=q // 128, kv_heads=kv // 128, head_dim=128, ffn=f,
                   vocab=VOCAB)
    r = _Rand(seed)
    w = {}
    src = {"q": "self_attn.q_proj", "k": "self_attn.k_proj", "v": "self_attn.v_proj", "o": "self_attn.o_proj",
           "gate": "mlp.gate_proj", "up": "mlp.up_proj", "down": "mlp.down_proj"}
    for i in range(s.layers):
        p = f"model.layers.{i}."
        w[p + "input_layernorm.weight"] = r.norm(h)
        w[p + "post_attention_layernorm.weight"] = r.norm(h)
        for nm, n, k in mats(case):
            w[p + src[nm] + ".weight"] = r.w4(n, k)
    w["model.norm.weight"] = r.norm(h)
    w["model.embed_tokens.weight"] = torch.randn((VOCAB, h), generator=r.g, device=DEV).to(torch.bfloat16)
    w["lm_head.weight"] = r.w4(VOCAB, h)
    rng = np.random.default_rng(seed)
    imp = np.zeros(s.layers)
    imp[rng.choice(s.layers, size=int(round(case["w4a16"] * s.layers)), replace=False)] = 1.0
    return s, w, imp, int(rng.integers(VOCAB))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        s, w, imp, token = _decode_parts(case, seed)
        w = {k: GpuW4(v[0], v[1], None, v[0].shape[0], v[0].shape[1] * 2) if isinstance(v, tuple) else v
             for k, v in w.items()}
        ctx = case["context"]
        model = DecodeModel(s, max_seq=256 * (ctx // 256 + 2), prefill=ctx, importance=imp, seed=seed, weights=w)
        model.start(token)
        model.capture()
        return {"case": case, "model": model, "token": token}
    r = _Rand(seed)
    if kind == "gemv":
        nib, sc = r.w4(case["n"], case["k"])
        return {"case": case, "w": GpuW4(nib, sc, None, case["n"], case["k"]),
                "x": r.acts(1, case["k"], DT[case["dtype"]])}
    if kind == "head":
        nib, sc = r.w4(case["n"], case["k"])
        return {"case": case, "w": GpuW4(nib, sc, None, case["n"], case["k"]),
                "x": r.acts(case["m"], case["k"], torch.float16)}
    if kind == "load":
        w = [r.dense(n, k).to(DT[case["dtype"]]) for _, n, k in mats(case)]
        awq = [r.awq(k) if case["mode"] != "plain" else None for _, _, k in mats(case)]
        return {"case": case, "w": w, "awq": awq}
    # layer, batch, prefill: a layer's weights and the inputs of its four input points
    h, q, kv, f = dims(case)
    ws = {}
    for nm, n, k in mats(case):
        nib, sc = r.w4(n, k)
        ws[nm] = GpuW4(nib, sc, r.awq(k) if case.get("awq") else None, n, k)
    m = case.get("m", 1)
    dt = DT[case.get("dtype", "f16")]
    st = {"case": case, "w": ws, "x": {"qkv": r.acts(m, h, dt), "o": r.acts(m, q, dt), "ffn": r.acts(m, h, dt),
                                       "down": r.acts(m, f, dt)}}
    if kind == "prefill":  # one workspace for the layer, as a serving process keeps it
        need = max(hk.gemm_w4a16_workspace_bytes(m, n, k) for _, n, k in mats(case))
        st["ws"] = torch.empty(max(need, 256), dtype=torch.uint8, device=DEV)
    return st


INPUT = {"q": "qkv", "k": "qkv", "v": "qkv", "o": "o", "gate": "ffn", "up": "ffn", "down": "down"}


# ---- one pass --------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "gemv":
        w = state["w"]
        return project(state["x"], w, case["precision"] == "w4a8")
    if kind == "head":
        w = state["w"]
        xq, xs = hk.quantize_q8_rows(state["x"], per_token=case["per_token"])
        return hk.matvec_w4a8_batched(xq, xs, w.nibbles, w.scales, w.n, w.k)
    if kind == "load":
        kq = case["mode"] == "kquant"
        got = [GpuW4.quantize(w, awq=a, kquant=kq) for w, a in zip(state["w"], state["awq"])]
        return [(g.nibbles, g.scales, g.awq_scales) for g in got]
    if kind == "decode":
        m = state["model"]
        m.start(state["token"])
        m.generate(1)
        p = case["context"]
        return {"logits": m.logits, "k": [lw["k_cache"][:, p] for lw in m.layers],
                "v": [lw["v_cache"][:, p] for lw in m.layers]}
    w, x = state["w"], state["x"]
    if kind == "prefill":
        return [hk.gemm_w4a16_ws(x[INPUT[nm]], g.nibbles, g.scales, g.n, g.k, state["ws"], awq=g.awq_scales,
                                 out_dtype=x["qkv"].dtype) for nm, g in w.items()]
    if kind == "batch":
        xq = {nm: hk.quantize_q8_rows(v, per_token=case["per_token"]) for nm, v in x.items()}
        return [hk.matvec_w4a8_batched(*xq[INPUT[nm]], g.nibbles, g.scales, g.n, g.k) for nm, g in w.items()]
    if case["precision"] == "w4a16":
        q, k, v = w["q"], w["k"], w["v"]
        out = list(hk.fused_qkv_matvec_w4a16(x["qkv"], q.nibbles, q.scales, None, q.n, k.nibbles, k.scales, None, k.n,
                                             v.nibbles, v.scales, None, v.n, q.k))
        return out + [hk.fused_matvec_w4a16(x[INPUT[nm]], w[nm].nibbles, w[nm].scales, None, w[nm].n, w[nm].k)
                      for nm in ("o", "gate", "up", "down")]
    g3 = [(w[nm].nibbles, w[nm].scales, w[nm].n) for nm in ("q", "k", "v")]
    g2 = [(w[nm].nibbles, w[nm].scales, w[nm].n) for nm in ("gate", "up")]
    out = hk.grouped_matvec_w4a8_x(x["qkv"][0], g3, w["q"].k)
    out.append(hk.matvec_w4a8_x(x["o"][0], w["o"].nibbles, w["o"].scales, w["o"].n, w["o"].k))
    out += hk.grouped_matvec_w4a8_x(x["ffn"][0], g2, w["gate"].k)
    xq, xs = hk.quantize_f16_q8(x["down"])
    out.append(hk.matvec_w4a8(xq, xs, w["down"].nibbles, w["down"].scales, w["down"].n, w["down"].k,
                              out_dtype=torch.float32))
    return out


# ---- what a pass cannot do without -----------------------------------------------------
def work(case):
    kind = case["kind"]
    w4 = 0.625  # bytes per packed weight: a nibble and a 1/32 share of an f32 scale
    if kind in ("gemv", "head"):
        n, k, m = case["n"], case["k"], case.get("m", 1)
        return {"bytes": w4 * n * k + 2 * m * k + (2 if kind == "gemv" else 4) * m * n, "flops": 2 * m * n * k}
    if kind == "decode":
        h, q, kv, f = dims(case)
        per = sum(n * k for _, n, k in mats(case))
        cache = 2 * 2 * kv * (case["context"] + 1)
        params = case["layers"] * per + VOCAB * h
        return {"bytes": w4 * params + case["layers"] * cache + 4 * VOCAB, "flops": 2 * params}
    ms = mats(case)
    params = sum(n * k for _, n, k in ms)
    if kind == "load":
        size = 4 if case["dtype"] == "f32" else 2
        return {"bytes": (size + w4) * params, "flops": 0}
    h, q, kv, f = dims(case)
    m = case.get("m", 1)
    osz = 4 if kind == "batch" or case.get("precision") == "w4a8" else 2
    act = 2 * m * (2 * h + q + f) + osz * m * sum(n for _, n, _ in ms)
    return {"bytes": w4 * params + act, "flops": 2 * m * params}


def tolerance(case):
    kind = case["kind"]
    if kind == "load":
        return "exact"  # nibbles, block scales and inverse scales are defined bit for bit
    if kind == "decode":
        # a rounding may move an int8 activation code, which the later layers carry on (the attention's
        # key split set to 2 instead of 4, over six seeds: up to 0.7% after two layers, 1.3% after four)
        return {"rel": 3e-2, "max": 0.5}
    if kind in ("batch", "head") or (kind == "layer" and case["precision"] == "w4a8"):
        return {"rel": 2e-6, "max": 1e-4}  # fp32 outputs: the order of fp32 sums (1.3e-7 off 64 bits)
    if kind == "gemv" or case["dtype"] == "f16":
        # fp16 outputs (project returns fp16), rounded once: 2.1e-4 off 64 bits
        return {"rel": 8e-4, "max": 2e-2}
    return {"rel": 7e-3, "max": 5e-2}  # bf16 outputs: 1.7e-3 off 64 bits


# ---- the same results in 64 bits -------------------------------------------------------
def _values(nib, sc):
    """(nibble - 8) [n, k/32, 32] and scales [n, k/32, 1], in element order."""
    n, k2 = nib.shape
    b = nib.view(n, k2 // 16, 16)
    return torch.cat((b & 15, b >> 4), -1).to(torch.float64) - 8.0, sc[..., None]


def _matrix(nib, sc, awq=None, dtype=None):
    """The weight matrix in float64; `dtype`: as the prefill product uses it, formed in f32
    and rounded to the activation type."""
    v, s = _values(nib, sc)
    if dtype is None:
        return (v * s.double()).view(nib.shape[0], -1)
    w = (v.float() * s).view(nib.shape[0], -1)
    return (w if awq is None else w * awq).to(dtype).double()


def _q8_group(x):
    """Group-32 int8 codes times their f32 scales, in float64 (x: f32 [..., K])."""
    g = x.float().view(*x.shape[:-1], -1, 32)
    a = g.abs().amax(-1, keepdim=True)
    s = torch.where(a > 0, a / 127.0, torch.ones_like(a))
    q = (g * (1.0 / s)).round().clamp(-127, 127)
    return (q.double() * s.double()).view(x.shape)


def _q8_row(x):
    x = x.float()
    a = x.abs().amax(-1, keepdim=True)
    s = torch.where(a > 0, a / 127.0, torch.ones_like(a)).to(torch.bfloat16).float()
    return (x * (1.0 / s)).round().clamp(-127, 127).double() * s.double()


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        return _exact_decode(case, seed)
    r = _Rand(seed)
    if kind == "load":
        if case["mode"] != "plain":
            return None  # the scale is the result of a search over candidates in f32
        out = []
        for _, n, k in mats(case):
            w = r.dense(n, k).to(DT[case["dtype"]])
            out.append((None, w.double().view(n, k // 32, 32).abs().amax(-1) / 7, None))
        return out
    if kind == "gemv":
        nib, sc = r.w4(case["n"], case["k"])
        x = r.acts(1, case["k"], DT[case["dtype"]])
        xv = _q8_group(x.float()) if case["precision"] == "w4a8" else x.double()
        return xv @ _matrix(nib, sc).T
    if kind == "head":
        nib, sc = r.w4(case["n"], case["k"])
        x = r.acts(case["m"], case["k"], torch.float16)
        xv = _q8_row(x) if case["per_token"] else _q8_group(x.float())
        return torch.cat([xv @ _matrix(nib[i:i + 16384], sc[i:i + 16384]).T for i in range(0, case["n"], 16384)], 1)
    h, q, kv, f = dims(case)
    m = case.get("m", 1)
    if kind == "prefill" and work(case)["flops"] > 5e11:
        return None
    ws = []
    for nm, n, k in mats(case):
        w = r.w4(n, k)
        ws.append((nm, w, r.awq(k) if case.get("awq") else None))
    dt = DT[case.get("dtype", "f16")]
    x = {"qkv": r.acts(m, h, dt), "o": r.acts(m, q, dt), "ffn": r.acts(m, h, dt), "down": r.acts(m, f, dt)}
    out = []
    for nm, (nib, sc), awq in ws:
        xv = x[INPUT[nm]]
        if kind == "prefill":
            y = xv.double() @ _matrix(nib, sc, awq, dt).T
        elif kind == "batch":
            y = (_q8_row(xv) if case["per_token"] else _q8_group(xv.float())) @ _matrix(nib, sc).T
        elif case["precision"] == "w4a16":
            y = xv.double() @ _matrix(nib, sc).T
        else:
            y = (_q8_group(xv.float()) @ _matrix(nib, sc).T)[0]
            if nm == "down":
                y = y[None]
        out.append(y)
    return out


def _exact_decode(case, seed):
    s, w, imp, token = _decode_parts(case, seed)
    g = torch.Generator(device=DEV).manual_seed(seed)
    ctx, d, half = case["context"], s.head_dim, s.head_dim // 2
    f64 = torch.float64

    def norm(x, name):
        return (x * torch.rsqrt((x * x).mean() + s.eps) * w[name].to(f64)).float()

    def mv(x, name, w4a8):
        xv = _q8_group(x) if w4a8 else x.half().to(f64)
        return _matrix(*w[name]) @ xv

    inv = s.rope_theta ** (-2.0 * torch.arange(half, dtype=f64, device=DEV) / d)
    cos, sin = torch.cos(ctx * inv).float().to(f64), torch.sin(ctx * inv).float().to(f64)

    def rope(x, heads):
        y = x.view(heads, d)
        a, b = y[:, :half], y[:, half:]
        return torch.cat((a * cos - b * sin, a * sin + b * cos), -1)

    hid = w["model.embed_tokens.weight"][token].to(f64)
    ks, vs = [], []
    for i in range(s.layers):
        p, w4a8 = f"model.layers.{i}.", imp[i] < 0.7
        kc = torch.randn((s.kv_heads, ctx, d), generator=g, device=DEV).to(torch.bfloat16)
        vc = torch.randn((s.kv_heads, ctx, d), generator=g, device=DEV).to(torch.bfloat16)
        x = norm(hid, p + "input_layernorm.weight")
        q = rope(mv(x, p + "self_attn.q_proj.weight", w4a8), s.heads)
        k = rope(mv(x, p + "self_attn.k_proj.weight", w4a8), s.kv_heads)
        v = mv(x, p + "self_attn.v_proj.weight", w4a8).view(s.kv_heads, d)
        ks.append(k)
        vs.append(v)
        k = torch.cat((kc.to(f64), k.to(torch.bfloat16).to(f64)[:, None]), 1)
        v = torch.cat((vc.to(f64), v.to(torch.bfloat16).to(f64)[:, None]), 1)
        q = q.view(s.kv_heads, s.heads // s.kv_heads, d)
        a = torch.softmax((q @ k.transpose(1, 2).contiguous()) / math.sqrt(d), -1) @ v
        hid = hid + mv(a.reshape(-1).float(), p + "self_attn.o_proj.weight", w4a8)
        x = norm(hid, p + "post_attention_layernorm.weight")
        gate, up = mv(x, p + "mlp.gate_proj.weight", w4a8), mv(x, p + "mlp.up_proj.weight", w4a8)
        act = (gate * torch.sigmoid(gate) * up).half().float()
        hid = hid + mv(act, p + "mlp.down_proj.weight", w4a8)
    x = _q8_group(norm(hid, "model.norm.weight"))
    nib, sc = w["lm_head.weight"]
    logits = torch.cat([_matrix(nib[i:i + 16384], sc[i:i + 16384]) @ x for i in range(0, VOCAB, 16384)])
    return {"logits": logits, "k": ks, "v": vs}
