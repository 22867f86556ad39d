"""The calls that a user of this package has it do, with their sizes, inputs,
tolerances and 64-bit results: what its speed is measured on.

Two models give the widths: the Flash model (hidden 5376, 56 heads of 128, SwiGLU
FFN of inner width 14336) and the benchmark block (hidden 5120, 40 heads of 128,
GELU FFN of 20480). Tokens come as frames of 32 x 64 rows, of which spatial
selection keeps 17 x 33 = 561, and 317 text rows: 6 frames and text are 12605
tokens, 3683 after selection; one selected frame and text are 878.

Kinds of case:
  proj     one W8A8 projection layer, quantizer included (Int8Linear.__call__)
  norm     fused RMSNorm + adaLN modulate + INT8 quantizer
  resnorm  the same behind the gated residual of the attention output
  act      FFN activation fused into the re-quantizer (SwiGLU or GELU-tanh)
  qk       Q/K RMSNorm + RoPE on views of the fused QKV output
  table    the adaLN table of a set of time embeddings
  select   Flash token selection: row gathers, then the residual restore
  chain    every projection of a block, norms, residuals and FFN included
"""
import math
import types

import torch

from lynnreal_omni_amd import flash, fusion, kernels
from lynnreal_omni_amd.int8 import Int8Linear

EPS = 1e-6
GRID = (32, 64)  # rows of one frame

# hidden, attention width, FFN-up columns, FFN-down inputs, FFN activation
MODELS = {
    "flash": (5376, 7168, 28672, 14336, "swiglu"),
    "bench": (5120, 5120, 20480, 20480, "gelu_tanh"),
}


def _projections(model):
    """(N, K) of the block's projections: QKV, out, up, down."""
    hidden, attn, up, down, _ = MODELS[model]
    return {"qkv": (3 * attn, hidden), "out": (hidden, attn), "up": (up, hidden), "down": (hidden, down)}


# ------------------------------------------------------------------ cases ----
def listed():
    return [
        # A projection of a handful of tokens (32 rows, the smallest installation
        # check): latency, launches and the weight stream.
        {"name": "proj_m32", "kind": "proj", "model": "flash", "layer": "out", "rows": 32},
        # The decode-like projection of streaming: 256 rows.
        {"name": "proj_m256", "kind": "proj", "model": "bench", "layer": "out", "rows": 256},
        # One frame through one layer: the single W8A8 linear of the benchmarks.
        {"name": "proj_frame", "kind": "proj", "model": "bench", "layer": "out", "rows": 2048},
        # The attention prologue of one selected frame and its text.
        {"name": "norm_frame", "kind": "norm", "model": "flash", "rows": 878, "groups": 2},
        # The FFN prologue at full resolution: 6 frames with a time step each, and text.
        {"name": "resnorm_full", "kind": "resnorm", "model": "flash", "rows": 12605, "groups": 6},
        # The Flash FFN's activation and re-quantizer on the selected tokens.
        {"name": "act_kept", "kind": "act", "model": "flash", "rows": 3683},
        # Q and K of the selected tokens, full-width rotary embedding.
        {"name": "qk_kept", "kind": "qk", "model": "flash", "rows": 3683, "rotary": 128},
        # The modulation table of 6 frames' time embeddings.
        {"name": "table_6", "kind": "table", "model": "flash", "rows": 6},
        # Selection of 6 frames, before and after the selected blocks.
        {"name": "select_6", "kind": "select", "model": "flash", "frames": 6, "text": 317},
        # A block's projections on one selected frame and text (streaming).
        {"name": "chain_frame", "kind": "chain", "model": "flash", "rows": 878, "groups": 2},
        # The same on the selected tokens of 6 frames: most of Flash's blocks.
        {"name": "chain_kept", "kind": "chain", "model": "flash", "rows": 3683, "groups": 6},
        # The benchmark's block at 12288 tokens.
        {"name": "chain_full", "kind": "chain", "model": "bench", "rows": 12288, "groups": 1},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["proj", "proj", "proj", "norm", "resnorm", "act", "qk", "table", "select",
                       "chain", "chain"])
    model = rng.choice(["flash", "flash", "bench"])
    case = {"kind": kind, "model": model}
    if kind == "proj":
        case.update(layer=rng.choice(["qkv", "out", "up", "down"]), rows=_log_int(rng, 1, 12605))
    elif kind in ("norm", "resnorm"):
        case.update(rows=_log_int(rng, 16, 16385), groups=rng.choice([1, 2, 6]))
    elif kind == "act":
        case.update(rows=_log_int(rng, 16, 12605))
    elif kind == "qk":
        case.update(rows=_log_int(rng, 16, 12605), rotary=rng.choice([128, 128, 64]))
    elif kind == "table":
        # The width of the embedding varies with the model, the rows with the frames.
        case.update(rows=rng.randint(1, 8))
    elif kind == "select":
        case.update(frames=rng.randint(1, 6), text=rng.randint(16, 512))
    else:
        case.update(rows=_log_int(rng, 64, 8192), groups=rng.choice([1, 2, 6]))
    return case


# ----------------------------------------------------------------- inputs ----
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, scale=1.0):
    return torch.randn(*shape, device="cuda", generator=g) * scale


def _activations(g, *shape):
    """N(0, 1) with 1% of the channels 20 times larger (outlier channels)."""
    x = _randn(g, *shape)
    channels = torch.randperm(shape[-1], device="cuda", generator=g)[: max(1, shape[-1] // 100)]
    x[..., channels] *= 20
    return x.bfloat16()


def _layer(g, n, k):
    w = torch.randint(-127, 128, (n, k), device="cuda", dtype=torch.int8, generator=g)
    scale = torch.rand(n, 1, device="cuda", generator=g) * 4e-3 + 1e-3
    layer = Int8Linear.from_packed(w, scale, _randn(g, n, scale=0.02).bfloat16(), gemm="hip")
    layer.fused_ops = True
    return layer


def _norm(g, hidden):
    return types.SimpleNamespace(weight=(1 + _randn(g, hidden, scale=0.05)).bfloat16(), eps=EPS)


def _table(g, groups, hidden):
    return _randn(g, groups, 6 * hidden, scale=0.1).bfloat16()


def _indices(rows, groups):
    """Table row of each token: the frames in order, then text with the first row's."""
    text = min(317, rows // 4) if groups > 1 else 0
    video = rows - text
    frame = torch.arange(video, device="cuda") * groups // max(1, video)
    return torch.cat([frame, torch.zeros(text, device="cuda", dtype=torch.int64)])


def _rotary(g, rows, width):
    phase = _randn(g, rows, width)
    return phase.cos(), phase.sin()


def _layout(frames, text):
    """Positions (time, h, w) and tags of `text` rows and then `frames` frames."""
    height, width = GRID
    time = torch.arange(frames, device="cuda", dtype=torch.float64)
    h = torch.arange(height, device="cuda", dtype=torch.float64)
    w = torch.arange(width, device="cuda", dtype=torch.float64)
    video = torch.cartesian_prod(time, h, w)
    words = torch.zeros(text, 3, device="cuda", dtype=torch.float64)
    words[:, 0] = torch.arange(text, device="cuda")
    tags = torch.zeros(text + video.shape[0], device="cuda", dtype=torch.int64)
    tags[:text] = 1
    return torch.cat([words, video]), tags


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    hidden, attn, up, down, activation = MODELS[case["model"]]
    s = types.SimpleNamespace(kind=kind, activation=activation)
    rows = case.get("rows")
    if kind == "proj":
        n, k = _projections(case["model"])[case["layer"]]
        s.x = _activations(g, 1, rows, k)
        s.layer = _layer(g, n, k)
    elif kind in ("norm", "resnorm"):
        s.x = _activations(g, 1, rows, hidden)
        s.norm = _norm(g, hidden)
        s.table, s.indices = _table(g, case["groups"], hidden), _indices(rows, case["groups"])
        if kind == "resnorm":
            s.update = _activations(g, 1, rows, hidden)
    elif kind == "act":
        s.x = _randn(g, rows, up).bfloat16()
    elif kind == "qk":
        heads = attn // 128
        qkv = _randn(g, 1, rows, 3 * heads, 128).bfloat16()
        s.q, s.k = qkv[:, :, :heads], qkv[:, :, heads:2 * heads]
        s.qw, s.kw = _norm(g, 128).weight, _norm(g, 128).weight
        s.rotary = _rotary(g, rows, case["rotary"])
    elif kind == "table":
        s.temb = _randn(g, rows, hidden)
        s.weight = _randn(g, 6 * hidden, hidden, scale=0.02).bfloat16()
        s.bias = _randn(g, 6 * hidden, scale=0.1).bfloat16()
    elif kind == "select":
        positions, tags = _layout(case["frames"], case["text"])
        s.keep, s.inverse = flash.spatial_layout(positions, tags)
        tokens = tags.numel()
        s.x = _activations(g, 1, tokens, hidden)
        s.current = _activations(g, 1, s.keep.numel(), hidden)
        s.indices = torch.where(tags == 0, positions[:, 0].long(), 0)
        s.rotary = _rotary(g, tokens, 128)
    else:
        s.x = _activations(g, 1, rows, hidden)
        s.attention = _randn(g, 1, rows, attn).bfloat16()
        s.norm1, s.norm2 = _norm(g, hidden), _norm(g, hidden)
        s.table, s.indices = _table(g, case["groups"], hidden), _indices(rows, case["groups"])
        shapes = _projections(case["model"])
        s.layers = fusion.ChainLayers(**{field: _layer(g, *shapes[name]) for field, name in
                                         (("to_qkv", "qkv"), ("to_out", "out"), ("up", "up"), ("down", "down"))})
    return s


# ------------------------------------------------------------------- call ----
@torch.inference_mode()
def run(s):
    if s.kind == "proj":
        return s.layer(s.x)
    if s.kind == "norm":
        return kernels._rms_adaln_quant_int8(s.x, s.norm, s.table, s.indices, 0, 1)
    if s.kind == "resnorm":
        return kernels.residual_rms_quant(s.x, s.update, s.norm, s.table, s.indices)
    if s.kind == "act":
        if s.activation == "swiglu":
            return kernels._swiglu_quant_int8(s.x)
        return kernels._gelu_quant_int8(s.x)
    if s.kind == "qk":
        return kernels.qk_norm_rope(s.q, s.k, s.qw, s.kw, s.rotary, EPS)
    if s.kind == "table":
        return kernels.adaln_table(s.temb, s.weight, s.bias)
    if s.kind == "select":
        entered = flash.gather_rows(s.x, s.keep, 1)
        indices = flash.gather_rows(s.indices, s.keep, 0)
        cos, sin = (flash.gather_rows(t, s.keep, -2) for t in s.rotary)
        return entered, indices, cos, sin, flash.restore(s.x, s.current, entered, s.inverse, 1.0)
    return fusion.projection_chain(s.x, s.layers, s.norm1, s.norm2, s.table, s.indices, s.attention,
                                   ffn=s.activation)


# ------------------------------------------------------------------- work ----
def work(case):
    kind = case["kind"]
    hidden, attn, up, down, activation = MODELS[case["model"]]
    rows = case.get("rows")
    if kind == "proj":
        n, k = _projections(case["model"])[case["layer"]]
        return {"bytes": 2 * rows * k + n * k + 6 * n + 2 * rows * n, "flops": 2 * rows * n * k}
    if kind == "norm":
        return {"bytes": rows * (3 * hidden + 12) + (3 * case["groups"] + 1) * 2 * hidden,
                "flops": 10 * rows * hidden}
    if kind == "resnorm":
        return {"bytes": rows * (7 * hidden + 12) + (4 * case["groups"] + 1) * 2 * hidden,
                "flops": 12 * rows * hidden}
    if kind == "act":
        return {"bytes": rows * (2 * up + down + 4), "flops": 12 * rows * down}
    if kind == "qk":
        return {"bytes": 8 * rows * attn + 8 * rows * case["rotary"], "flops": 12 * rows * attn}
    if kind == "table":
        return {"bytes": 12 * hidden * hidden + 12 * hidden + rows * (4 * hidden + 12 * hidden),
                "flops": 12 * rows * hidden * hidden}
    if kind == "select":
        h, w = GRID
        tokens = case["frames"] * h * w + case["text"]
        kept = case["frames"] * (h // 2 + 1) * (w // 2 + 1) + case["text"]
        return {"bytes": 4 * tokens * hidden + 6 * kept * hidden + 2 * kept * (8 + 2 * 128 * 4) + 8 * tokens,
                "flops": 2 * tokens * hidden}
    macs = 3 * attn * hidden + attn * hidden + up * hidden + down * hidden
    return {"bytes": macs + 2 * rows * (2 * hidden + attn + 3 * attn + hidden) + 12 * case["groups"] * hidden,
            "flops": 2 * rows * macs}


# -------------------------------------------------------------- tolerance ----
def tolerance(case):
    """bf16 outputs: about four times the rounding of a bf16 result against 64
    bits, or of what a change of one rounding upstream does to it. INT8 rows
    follow values that were rounded to bf16 on the way, so another order of the
    norm's sum or another correct exponential moves a few of them by one (below
    one in ten thousand)."""
    kind = case["kind"]
    if kind in ("proj", "qk", "table", "chain"):
        return {"rel": 8e-3, "max": 0.1}
    if kind == "select":
        return {"rel": 5e-3, "max": 0.05}
    return {"rel": 5e-3, "max": 0.05, "differ": 4e-4}


# ------------------------------------------------------------------ exact ----
def _quantized(x):
    scale = x.abs().amax(-1, keepdim=True).clamp_min(1e-8) / 127
    return torch.round(x / scale), scale


def _linear(x, layer):
    q, scale = _quantized(x)
    y = (q @ layer.weight_int8.double()) * scale * layer.weight_scale.double()
    return y if layer.bias is None else y + layer.bias.double()


def _modulated(x, norm, table, indices, shift, scale):
    hidden = x.shape[-1]
    rows = table.double().view(-1, 6, hidden)[indices]
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * norm.weight.double()
    return y * (1 + rows[:, scale]) + rows[:, shift]


def _gate(table, indices, slot, hidden):
    return table.double().view(-1, 6, hidden)[indices, slot]


def _activated(p, activation):
    if activation == "swiglu":
        v, g = p.chunk(2, -1)
        return v * g * torch.sigmoid(g)
    return torch.nn.functional.gelu(p, approximate="tanh")


def exact(case, seed):
    s = prepare(case, seed)
    kind = s.kind
    hidden = MODELS[case["model"]][0]
    if kind == "proj":
        return _linear(s.x.double(), s.layer)
    if kind == "norm":
        y = _modulated(s.x.double().view(-1, hidden), s.norm, s.table, s.indices, 0, 1)
        return None, _quantized(y)[1]
    if kind == "resnorm":
        x = s.x.double() + _gate(s.table, s.indices, 2, hidden) * s.update.double()
        y = _modulated(x.view(-1, hidden), s.norm, s.table, s.indices, 3, 4)
        return x, None, _quantized(y)[1]
    if kind == "act":
        return None, _quantized(_activated(s.x.double(), s.activation))[1]
    if kind == "qk":
        out = []
        for x, w in ((s.q.double(), s.qw.double()), (s.k.double(), s.kw.double())):
            n = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w
            width = case["rotary"]
            cos, sin = (t.bfloat16().double()[None, :, None] for t in s.rotary)
            a, b = n[..., :width].chunk(2, -1)
            turned = n[..., :width] * cos + torch.cat([-b, a], -1) * sin
            out.append(torch.cat([turned, n[..., width:]], -1))
        return tuple(out)
    if kind == "table":
        a = torch.nn.functional.silu(s.temb).bfloat16().double()
        return a @ s.weight.double().t() + s.bias.double()
    if kind == "select":
        entered = s.x.double()[:, s.keep]
        moved = (s.current.double() - entered)[:, s.inverse]
        return (entered, s.indices[s.keep], s.rotary[0].double()[s.keep], s.rotary[1].double()[s.keep],
                s.x.double() + moved)
    x, table, idx = s.x.double().view(-1, hidden), s.table, s.indices
    qkv = _linear(_modulated(x, s.norm1, table, idx, 0, 1), s.layers.to_qkv)
    attended = _linear(s.attention.double().view(x.shape[0], -1), s.layers.to_out)
    x1 = x + _gate(table, idx, 2, hidden) * attended
    projected = _linear(_modulated(x1, s.norm2, table, idx, 3, 4), s.layers.up)
    x2 = x1 + _gate(table, idx, 5, hidden) * _linear(_activated(projected, s.activation), s.layers.down)
    return qkv[None], x1[None], x2[None]
