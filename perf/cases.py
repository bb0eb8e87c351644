"""Performance cases of the DiT hot path: its single layers (quantized linears, fused activation quantizers, the MLP,
the attentions) and two whole blocks, each called as a node pack or an engine calls them, over the sizes a video DiT
meets: from a prompt of 77 tokens to a full-size step of 145,152.

Model widths are the two this repository's benchmark runs: "c2" (hidden 3072, 24 x 128 heads, FFN 8192) and "h3"
(hidden 5376, 56 x 128 heads, FFN 14336).

  listed()             the cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  inputs from the seed, and the quantized weights that a program keeps
  run(state)           one pass through the public entry points
  exact(case, seed)    the same result in float64 by plain torch (the quantization rules kept, everything else in 64 bits)
  work(case)           bytes and operations a pass cannot do without
  tolerance(case)      how far two correct implementations at this precision may be apart
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("rapid-h3_amd"))   # the package folder of the tree this runs in

from rapid_h3 import attention, gemm, kernels, quant  # noqa: E402
from rapid_h3.block import BlockWeights, fused_block, fused_mlp  # noqa: E402
from rapid_h3.linear import QuantLinear  # noqa: E402

D = 128
MODELS = {"c2": (3072, 24, 8192), "h3": (5376, 56, 14336)}   # hidden, heads, FFN width
DEV = "cuda"
BF16 = torch.bfloat16


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call: one prompt's text tokens through a projection patched by the node (its default mode, a bias)
        {"name": "linear_prompt", "kind": "quantlinear", "mode": "int8_rot", "m": 77, "k": 3072, "n": 9216},
        # the K / V projection of the text tokens that the draft block's cross-attention reads
        {"name": "linear_text_kv", "kind": "linear", "mode": "int8_rowwise", "m": 512, "k": 3072, "n": 6144},
        # the plain W8A8 linear that the reference's PyTorch path is checked with
        {"name": "linear_4096", "kind": "linear", "mode": "int8_rowwise", "m": 4096, "k": 3072, "n": 3072},
        # the FP8 QKV projection of a full-size step
        {"name": "linear_fp8_full", "kind": "linear", "mode": "fp8_rowwise", "m": 145152, "k": 3072, "n": 9216},
        # RMSNorm + modulation + rotation + INT8 at the head of every block of a full-size step
        {"name": "quant_norm_mod_rot_full", "kind": "quant", "prologue": "norm_mod", "rot": True, "m": 145152, "k": 3072},
        # the input of out_proj at the draft size of the wider model: head-major attention output, rotated
        {"name": "quant_heads_rot", "kind": "quant", "prologue": "heads", "rot": True, "m": 22332, "k": 7168},
        # the fused MLP that the node installs when only fc1 and fc2 are quantized: a preview-size step, odd length
        {"name": "mlp_preview", "kind": "mlp", "model": "c2", "m": 7001},
        # the shortest self-attention that takes the fused route, RMSNorm + RoPE included: a thumbnail step
        {"name": "attn_short", "kind": "attn", "config": None, "rr": True, "sq": 1560, "sk": 1560, "heads": 24},
        # cross-attention of the draft step's tokens to the text
        {"name": "attn_cross", "kind": "attn", "config": None, "rr": False, "sq": 72216, "sk": 512, "heads": 24},
        # the preset's attention (production numerics) at a preview size of the wider model
        {"name": "attn_preset_preview", "kind": "attn", "config": 94, "rr": True, "sq": 5583, "sk": 5583, "heads": 56},
        # a whole block as the preset runs it at the draft size of the wider model: text tokens, then video tokens
        {"name": "block_preset_draft", "kind": "block", "model": "h3", "recipe": "int8_rot", "config": 94, "s": 22332, "text": 512},
        # a whole block of a full-size step in the benchmark's recipe
        {"name": "block_full", "kind": "block", "model": "c2", "recipe": "int8_rowwise", "config": None, "s": 145152, "text": 0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "quantlinear", "quant", "quant", "mlp", "attn", "attn", "cross", "block"))
    model = rng.choice(("c2", "h3"))
    hid, heads, ffn = MODELS[model]
    top = 145152 if model == "c2" else 44992
    if kind in ("linear", "quantlinear"):
        k, n = rng.choice(((hid, 3 * heads * D), (heads * D, hid), (hid, 2 * ffn), (ffn, hid)))
        mode = rng.choice(("int8_rot", "int8_rowwise", "fp8_rowwise"))
        return {"kind": kind, "mode": mode, "m": _log(rng, 64, top), "k": k, "n": n}
    if kind == "quant":
        pro = rng.choice(("rows", "norm_mod", "heads", "swiglu"))
        k = {"rows": ffn, "norm_mod": hid, "heads": heads * D, "swiglu": ffn}[pro]
        return {"kind": kind, "prologue": pro, "rot": rng.random() < 0.6, "m": _log(rng, 512, top), "k": k}
    if kind == "mlp":
        return {"kind": kind, "model": model, "m": _log(rng, 512, top)}
    if kind == "attn":
        config = rng.choice((None, None, 94, 94, 60, 50))
        s = _log(rng, 1024, 72216 if model == "c2" else 44992)
        return {"kind": kind, "config": config, "rr": config != 60 and rng.random() < 0.75, "sq": s, "sk": s, "heads": heads}
    if kind == "cross":
        return {"kind": "attn", "config": rng.choice((None, 94)), "rr": False, "sq": _log(rng, 1024, 72216),
                "sk": _log(rng, 77, 1024), "heads": heads}
    recipe, config = rng.choice((("int8_rot", 94), ("int8_rowwise", None)))
    return {"kind": kind, "model": model, "recipe": recipe, "config": config, "s": _log(rng, 1024, 44992), "text": rng.choice((0, 226, 512))}


# ---------------------------------------------------------------- inputs
def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV) * std


def _acts(g, m, k):
    """Hidden states: N(0, 1) with 1 % of the channels x20, the outliers that the rotation is for."""
    x = _randn(g, m, k)
    x[:, torch.randperm(k, generator=g, device=DEV)[:max(1, k // 100)]] *= 20
    return x.to(BF16)


def _weight(g, n, k):
    return _randn(g, n, k, std=0.02).to(BF16)


def _norm_w(g, n):
    return (1 + 0.3 * _randn(g, n)).to(BF16)


def _rope(s):
    """Split-half RoPE table [1, S, 1, 48, 2, 2] = (cos, -sin, sin, cos) over (t, h, w) latent positions, 16 frequencies each."""
    i = torch.arange(s, device=DEV)
    pos = torch.stack([i // 4032, (i // 84) % 48, i % 84], 1).float()
    inv = 1.0 / (10000.0 ** (torch.arange(16, dtype=torch.float32, device=DEV) / 16))
    a = torch.cat((pos.unsqueeze(-1) * inv).unbind(1), -1)
    c, n = torch.cos(a), torch.sin(a)
    return torch.stack([c, -n, n, c], -1).reshape(1, s, 1, 48, 2, 2).to(BF16)


def _inputs(case, seed):
    """The raw tensors of a case (bf16 weights, activations, tables), from the seed alone."""
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    kind = case["kind"]
    if kind in ("linear", "quantlinear"):
        r = {"x": _acts(g, case["m"], case["k"]), "w": _weight(g, case["n"], case["k"])}
        if kind == "quantlinear":
            r["bias"] = _randn(g, case["n"], std=0.1).to(BF16)
        return r
    if kind == "quant":
        m, k, pro = case["m"], case["k"], case["prologue"]
        if pro == "heads":   # head-major attention output [H, M, 128]
            return {"x": _randn(g, k // D, m, D).to(BF16)}
        if pro == "swiglu":
            return {"x": _randn(g, m, 2 * k).to(BF16)}
        r = {"x": _acts(g, m, k)}
        if pro == "norm_mod":
            text = min(512, m // 4)   # two modality segments: text tokens, then video tokens
            r["w"] = _norm_w(g, k)
            r["idx"] = (torch.arange(m, device=DEV) >= text).to(torch.int32)
            r["shift"], r["scale"] = _randn(g, 2, k, std=0.1), _randn(g, 2, k, std=0.1)
        return r
    if kind == "mlp":
        hid, _, ffn = MODELS[case["model"]]
        return {"x": _acts(g, case["m"], hid), "fc1": _weight(g, 2 * ffn, hid), "fc2": _weight(g, hid, ffn)}
    if kind == "attn":
        sq, sk, h = case["sq"], case["sk"], case["heads"]
        if sq == sk:   # views of one qkv projection output, as in a block; K carries a per-channel offset
            qkv = _randn(g, sq, 3, h, D)
            qkv[:, 1] += 2 * _randn(g, h, D)
            q, k, v = qkv.to(BF16).unbind(1)
        else:
            q = _randn(g, sq, h, D).to(BF16)
            kv = _randn(g, sk, 2, h, D)
            kv[:, 0] += 2 * _randn(g, h, D)
            k, v = kv.to(BF16).unbind(1)
        r = {"q": q, "k": k, "v": v}
        if case["rr"]:
            r["tab"], r["qw"], r["kw"] = _rope(sq), _norm_w(g, D), _norm_w(g, D)
        return r
    hid, heads, ffn = MODELS[case["model"]]
    r = {"x": _acts(g, case["s"], hid), "tab": _rope(case["s"])}
    for name, n, k in (("qkv", 3 * heads * D, hid), ("out", hid, heads * D), ("fc1", 2 * ffn, hid), ("fc2", hid, ffn)):
        r[name] = _weight(g, n, k)
    for name, n in (("norm1", hid), ("norm2", hid), ("qw", D), ("kw", D)):
        r[name] = _norm_w(g, n)
    r["mod"] = tuple(_randn(g, 2, hid, std=0.1) for _ in range(6))
    return r


def _segments(case):
    s, t = case["s"], case["text"]
    return [(0, t, 0), (t, s, 1)] if t else [(0, s, 1)]


def prepare(case, seed):
    r, kind = _inputs(case, seed), case["kind"]
    st = {"case": case, **r}
    if kind == "linear":
        st["qw"] = kernels.quantize_weight(r["w"], case["mode"])
        del st["w"]
    elif kind == "quantlinear":
        st["layer"] = QuantLinear(r["w"], r["bias"], case["mode"])
        st["layer"].qweight_for()
    elif kind == "mlp":
        st["fc1"], st["fc2"] = (QuantLinear(r[n], None, "int8_rot", n) for n in ("fc1", "fc2"))
        st["fc1"].qweight_for(), st["fc2"].qweight_for()
    elif kind == "block":
        hid, heads, ffn = MODELS[case["model"]]
        qw = {n: kernels.quantize_weight(r[n], case["recipe"]) for n in ("qkv", "out", "fc1", "fc2")}
        perm = gemm.swiglu_perm(2 * ffn, DEV)
        fc1 = kernels.QWeight(qw["fc1"].q[perm].contiguous(), qw["fc1"].scale[:, perm].contiguous())
        st["weights"] = BlockWeights(qkv=qw["qkv"], out=qw["out"], fc1_perm=fc1, fc2=qw["fc2"], norm1_w=r["norm1"],
                                     norm2_w=r["norm2"], q_norm_w=r["qw"], k_norm_w=r["kw"], heads=heads,
                                     recipe=case["recipe"])
        st["segments"] = _segments(case)
        # the modulation row of each token: built once per model call, shared by its blocks
        st["idx"] = (torch.arange(case["s"], device=DEV) >= case["text"]).to(torch.int32)
        for n in ("qkv", "out", "fc1", "fc2"):
            del st[n]
    return st


# ---------------------------------------------------------------- one pass
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "linear":
        return kernels.linear(st["x"], st["qw"], case["mode"])
    if kind == "quantlinear":
        return st["layer"](st["x"])
    if kind == "quant":
        pro, rot = case["prologue"], case["rot"]
        if pro == "norm_mod":
            f = quant.norm_mod_rot_quant_rows_i8 if rot else quant.norm_mod_quant_rows_i8
            return f(st["x"], st["w"], 1e-6, st["idx"], st["shift"], st["scale"])
        if pro == "heads":
            return (quant.rot_quant_heads_i8 if rot else quant.heads_quant_rows_i8)(st["x"])
        if pro == "swiglu":
            return (quant.swiglu_rot_quant_rows_i8 if rot else quant.swiglu_quant_rows_i8)(st["x"])
        return (quant.rot_quant_rows_i8 if rot else quant.quant_rows_i8)(st["x"])
    if kind == "mlp":
        return fused_mlp(st["x"], st["fc1"], st["fc2"])
    if kind == "attn":
        if case["rr"]:
            return attention.attention_rr(st["q"], st["k"], st["v"], st["tab"], st["qw"], st["kw"], 1e-6, config=case["config"])
        return attention.attention(st["q"], st["k"], st["v"], config=case["config"])
    # the block updates its residual stream in place: each pass gets the same stream
    return fused_block(st["x"].clone(), st["weights"], st["mod"], st["segments"], st["tab"], idx=st["idx"], attn_config=case["config"])


# ---------------------------------------------------------------- the same in 64 bits
def _bf(x):
    return x.to(BF16).double()


def _chunks(m, row_bytes, most=4 << 30):
    n = max(1, min(m, most // max(1, row_bytes)))
    return [(a, min(m, a + n)) for a in range(0, m, n)]


def _hadamard(n):
    """Sylvester's matrix, normalized."""
    h = torch.ones(1, 1, dtype=torch.float64, device=DEV)
    while h.shape[0] < n:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(n)


def _convrot(x):
    """x @ blockdiag(H256)^T with the regular Hadamard matrix of order 256."""
    h4 = torch.tensor([[1, 1, 1, -1], [1, 1, -1, 1], [1, -1, 1, 1], [-1, 1, 1, 1]], dtype=torch.float64, device=DEV)
    h = h4
    for _ in range(3):
        h = torch.kron(h, h4)
    return (x.reshape(-1, 256) @ (h / 16).T).reshape(x.shape)


def _rows8(x):
    s = (x.abs().amax(1, keepdim=True) / 127).clamp_min(1e-12)
    return torch.round(x / s), s


def _rows_fp8(x):
    s = (x.abs().amax(1, keepdim=True) / 448).clamp_min(1e-12)
    return (x / s).clamp(-448, 448).float().to(torch.float8_e4m3fn).double(), s


def _codes(x, mode):
    """Codes and row scales of float64 rows (activations or a weight) in a linear's mode."""
    if mode == "fp8_rowwise":
        return _rows_fp8(x)
    return _rows8(_convrot(x) if mode == "int8_rot" else x)


def _silu(g):
    return g * torch.sigmoid(g)


def _linear(x, w, mode, bias=None):
    """bf16 x [M, K] (or float64 values), bf16 w [N, K] -> float64 [M, N], rows in chunks."""
    wq, ws = _codes(w.double(), mode)
    out = torch.empty(x.shape[0], w.shape[0], dtype=torch.float64, device=DEV)
    for a, b in _chunks(x.shape[0], 8 * (4 * x.shape[1] + 2 * w.shape[0])):
        xq, xs = _codes(x[a:b].double(), mode)
        out[a:b] = (xq @ wq.T) * xs * ws.T
    return out if bias is None else _bf(out) + bias.double()


def _norm_mod(x, w, idx, shift, scale, eps=1e-6):
    x = x.double()
    y = x / torch.sqrt((x * x).mean(1, keepdim=True) + eps) * w.double()
    return y * (1 + scale.double()[idx.long()]) + shift.double()[idx.long()]


def _rms_rope(x, tab, w, eps=1e-6):
    """x [S, 128] of one head -> float64, rounded to bf16 where the path holds bf16."""
    x = x.double()
    y = _bf(x / torch.sqrt((x * x).mean(1, keepdim=True) + eps) * w.double())
    t = tab.reshape(x.shape[0], -1, 2, 2).double()
    hr = t.shape[1]
    a, b = y[:, :hr], y[:, hr:2 * hr]
    return torch.cat([_bf(a * t[:, :, 0, 0] + b * t[:, :, 0, 1]), _bf(a * t[:, :, 1, 0] + b * t[:, :, 1, 1]), y[:, 2 * hr:]], 1)


def _block8(x):
    """One scale per 128 rows: the dequantized values."""
    s = x.shape[0]
    p = torch.nn.functional.pad(x, (0, 0, 0, -s % 128)).reshape(-1, 128, D)
    sc = p.abs().amax((1, 2), keepdim=True).clamp_min(1e-8) / 127
    return (torch.round(p / sc) * sc).reshape(-1, D)[:s]


def _token8(x):
    sc = x.abs().amax(1, keepdim=True).clamp_min(1e-8) / 127
    return torch.round(x / sc) * sc


def _attention(q, k, v, config, rr=None):
    """[S, H, 128] -> float64 [Sq, H, 128]: Q, K (and V) quantized by the numerics' rules, the softmax in float64."""
    sq, h = q.shape[:2]
    out = torch.empty(sq, h, D, dtype=torch.float64, device=DEV)
    h128 = _hadamard(D)
    for i in range(h):
        if rr is not None:
            qf, kf = _rms_rope(q[:, i], rr[0], rr[1]), _rms_rope(k[:, i], rr[0], rr[2])
        else:
            qf, kf = q[:, i].double(), k[:, i].double()
        kf = kf - kf.mean(0)
        vf = v[:, i].double()
        if config is None:
            qf, kf = _block8(qf), _block8(kf)
        else:
            qf, kf = _token8(qf @ h128), (_block8 if config == 60 else _token8)(kf @ h128)
            vm = vf.mean(0)
            vs = torch.maximum(vf.amax(0) - vm, vm - vf.amin(0)).clamp_min(1e-6) / 127
            if config == 50:
                vf = (((vf - vm) / vs) * (448 / 127)).float().to(torch.float8_e4m3fn).double() * (127 / 448) * vs + vm
            else:
                vf = torch.round((vf - vm) / vs) * vs + vm
        for a, b in _chunks(sq, 8 * 3 * k.shape[0]):
            out[a:b, i] = torch.softmax((qf[a:b] @ kf.T) * D ** -0.5, -1) @ vf
    return out


def _quant_exact(case, r):
    pro = case["prologue"]
    m, k = case["m"], case["k"]
    scale = torch.empty(m, 1, dtype=torch.float64, device=DEV)
    for a, b in _chunks(m, 8 * 10 * k):
        if pro == "norm_mod":
            x = _norm_mod(r["x"][a:b], r["w"], r["idx"][a:b], r["shift"], r["scale"])
        elif pro == "heads":
            x = r["x"][:, a:b].transpose(0, 1).reshape(b - a, k).double()
        elif pro == "swiglu":
            x = r["x"][a:b].double()
            x = _silu(x[:, :k]) * x[:, k:]
        else:
            x = r["x"][a:b].double()
        scale[a:b] = _rows8(_convrot(_bf(x)) if case["rot"] else x)[1]
    return None, scale   # codes are whole numbers


def exact(case, seed):
    kind = case["kind"]
    h = case.get("heads") or MODELS.get(case.get("model"), (0, 0, 0))[1]
    pairs = {"attn": lambda: case["sq"] * case["sk"], "block": lambda: case["s"] ** 2}.get(kind, lambda: 0)() * h
    if pairs > 1.3e11:   # about 20 seconds of float64 attention
        return None
    r = _inputs(case, seed)
    if kind in ("linear", "quantlinear"):
        return _linear(r["x"], r["w"], case["mode"], r.get("bias"))
    if kind == "quant":
        return _quant_exact(case, r)
    if kind == "mlp":
        ffn = MODELS[case["model"]][2]
        out = torch.empty(case["m"], r["x"].shape[1], dtype=torch.float64, device=DEV)
        for a, b in _chunks(case["m"], 8 * 12 * ffn):
            y = _bf(_linear(r["x"][a:b], r["fc1"], "int8_rot"))
            out[a:b] = _linear(_bf(_silu(y[:, :ffn]) * y[:, ffn:]), r["fc2"], "int8_rot")
        return out
    if kind == "attn":
        return _attention(r["q"], r["k"], r["v"], case["config"], (r["tab"], r["qw"], r["kw"]) if case["rr"] else None)
    hid, heads, ffn = MODELS[case["model"]]
    s, mode, mod = case["s"], case["recipe"], r["mod"]
    idx = (torch.arange(s, device=DEV) >= case["text"]).to(torch.int32)
    pre = (lambda x: _bf(x)) if mode == "int8_rot" else (lambda x: x)   # the rotation takes bf16 values
    x = r["x"].double()
    qkv = torch.cat([_linear(pre(_norm_mod(x[a:b], r["norm1"], idx[a:b], mod[0], mod[1])), r["qkv"], mode).to(BF16)
                     for a, b in _chunks(s, 8 * 12 * hid)]).view(s, 3, heads, D)
    o = _bf(_attention(qkv[:, 0], qkv[:, 1], qkv[:, 2], case["config"], (r["tab"], r["qw"], r["kw"]))).reshape(s, -1)
    del qkv
    gate = [_bf(mod[i])[idx.long()] for i in (2, 5)]
    for a, b in _chunks(s, 8 * 8 * ffn):
        y = _bf(x[a:b] + gate[0][a:b] * _bf(_linear(o[a:b], r["out"], mode)))
        f = _bf(_linear(pre(_norm_mod(y, r["norm2"], idx[a:b], mod[3], mod[4])), r["fc1"], mode))
        f = _bf(_silu(f[:, :ffn]) * f[:, ffn:])
        x[a:b] = y + gate[1][a:b] * _bf(_linear(f, r["fc2"], mode))
    return x


# ---------------------------------------------------------------- work and tolerance
def work(case):
    kind = case["kind"]
    if kind in ("linear", "quantlinear"):
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 2 * m * k + n * k + 4 * n + 2 * m * n, "flops": 2 * m * n * k}
    if kind == "quant":
        m, k = case["m"], case["k"]
        return {"bytes": (5 if case["prologue"] == "swiglu" else 3) * m * k + 4 * m, "flops": 0}
    if kind == "mlp":
        hid, _, ffn = MODELS[case["model"]]
        return {"bytes": 4 * case["m"] * hid + 3 * hid * ffn, "flops": 6 * case["m"] * hid * ffn}
    if kind == "attn":
        sq, sk, h = case["sq"], case["sk"], case["heads"]
        return {"bytes": 4 * (sq + sk) * h * D + (384 * sq if case["rr"] else 0), "flops": 4 * sq * sk * h * D}
    hid, heads, ffn = MODELS[case["model"]]
    s = case["s"]
    weights = 4 * heads * D * hid + 3 * hid * ffn
    return {"bytes": 4 * s * hid + 384 * s + weights, "flops": 2 * s * weights + 4 * s * s * heads * D}


def tolerance(case):
    kind = case["kind"]
    if kind == "quant":      # codes and scales follow a fixed rule to the last bit (SwiGLU: its exponential does not)
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.01} if case["prologue"] == "swiglu" else "exact"
    if kind in ("linear", "quantlinear"):    # one bf16 rounding
        return {"rel": 7e-3, "max": 2e-2}
    if kind == "mlp":        # two linears, bf16 between them
        return {"rel": 1e-2, "max": 0.2}
    if kind == "attn":       # P in 16 bits, 8 bits, or FP8
        return {"rel": {None: 1e-2, 94: 1.6e-2, 60: 1.6e-2}.get(case["config"], 3e-2), "max": 0.3}
    return {"rel": 1e-2, "max": 0.5}
