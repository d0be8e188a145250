"""The work a user of this library has it do, as measurable cases.

Families (``case["kind"]``), each through the entry point a program calls:

  quant        torch.ops.act_lib.quant_pack(_tiles) then dequant_unpack(_tiles): the quantizer's round
               trip on one activation (nearest, noise-tensor and Philox rounding, flat and tile layouts)
  saved_input  modules.module_utils.unified_quantize / unified_dequantize: what every compressed Linear and
               Conv layer does with its input (clamp, tanh squash, nearest codes, bf16 scale / min)
  linear       layers.DOLinear: training forward and backward under bf16 autocast
  activation   DOGELU / DOSiLU / DOReLU_Variance: training forward and backward
  batchnorm    DOBatchNorm2d / DOBatchNormReLU2d: training forward and backward
  fp8          torch.ops.act_lib.fp8_gemm_nt (B as [N, K]) and fp8_linear (B row-major [K, N])
  vit          a ViT with the Controller's compressed layers: forward, cross-entropy, backward

``exact`` restates each in plain torch in 64 bits. It keeps the storage roundings that are part of the
format (bf16 inputs and weights under autocast, bf16 scale / min and restored activations).
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import deep_optimization_amd  # noqa: F401  (registers torch.ops.act_lib)
from deep_optimization_amd.controller import Controller, layer_group_meta
from deep_optimization_amd.fusion import DOBatchNormReLU2d
from deep_optimization_amd.layers import DOLinear
from deep_optimization_amd.modules.activations import DOGELU, DOReLU_Variance, DOSiLU
from deep_optimization_amd.modules.module_utils import unified_dequantize, unified_quantize
from deep_optimization_amd.modules.normalization import DOBatchNorm2d
from deep_optimization_amd.vit import VisionTransformer

DEV = "cuda"
NAME = "layer"  # the layers' key in their meta dict
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2}
ROUNDING = {"nearest": 0, "noise": 1, "philox": 2}
SEED, OFFSET = 1, 0  # Philox key and offset
HALF = 0.5 - 1e-6  # the nearest codes' rounding offset
LARGEST = 256 * 256 * 56 * 56  # elements of the largest activation


def listed():
    return [
        # the smallest call: the CPU-sized case (fp32 [8, 64, 32, 32] in 16 x 16 tiles); launches and host time
        dict(name="quant_small_tiles", kind="quant", layout="tiles", dims="8x64x32x32", group=256, bits=2,
             rounding="nearest", dtype="f32", meta="f32", out="f32", data="normal"),
        # the headline: a ResNet-50 stage-1 activation at batch 256 with a caller's noise tensor; the largest
        dict(name="quant_resnet_noise", kind="quant", layout="flat", dims="256x256x56x56", group=256, bits=2,
             rounding="noise", dtype="bf16", meta="f32", out="bf16", data="relu"),
        # stochastic rounding from the counter-based generator on the ViT MLP activation
        dict(name="quant_vit_philox", kind="quant", layout="flat", dims="256x197x3072", group=128, bits=2,
             rounding="philox", dtype="bf16", meta="f32", out="bf16", data="gelu"),
        # the input that a compressed ViT fc2 layer saves and restores at batch 128
        dict(name="saved_vit_fc2", kind="saved_input", dims="128x197x3072", bits=2, dtype="bf16", data="gelu"),
        # one ViT fc1 layer's training pass at batch 128 (its input is LayerNorm's fp32 output)
        dict(name="linear_fc1_b128", kind="linear", batch=128, tokens=197, fin=768, fout=3072, bits=2, dtype="f32"),
        # a small odd batch: 985 tokens through an attention projection
        dict(name="linear_proj_b5", kind="linear", batch=5, tokens=197, fin=768, fout=768, bits=2, dtype="bf16"),
        # the ViT MLP's GELU at batch 128
        dict(name="gelu_vit_b128", kind="activation", act="gelu", dims="128x197x3072", bits=2, dtype="bf16"),
        # BatchNorm on the ResNet-50 stage-1 activation
        dict(name="bn_resnet_56", kind="batchnorm", relu=False, dims="256x256x56x56", bits=2, dtype="bf16"),
        # the fused BatchNorm + ReLU on ResNet-50's last stage: 49-element rows
        dict(name="bnrelu_resnet_7", kind="batchnorm", relu=True, dims="64x512x7x7", bits=2, dtype="bf16"),
        # the FP8 GEMM's headline size
        dict(name="fp8_8192", kind="fp8", m=8192, n=8192, k=8192, b="nk"),
        # an ordinary FP8 Linear with the weight in its row-major [K, N] layout and an odd token count
        dict(name="fp8_linear_985", kind="fp8", m=985, n=3072, k=768, b="kn"),
        # a whole training call: logits, loss and every gradient of a 2-block ViT, compressed by the Controller
        dict(name="vit_2_blocks", kind="vit", batch=64, depth=2, bits=2),
    ]


# ------------------------------------------------------------------------------------------ draws
def _log(rng, lo, hi):
    """A whole number, uniform over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dims3(rng, most=LARGEST):
    f = 64 * _log(rng, 1, 48)
    b = _log(rng, 1, 128)
    return f"{b}x{max(1, min(_log(rng, 1, 400), most // (b * f)))}x{f}"


def _dims4(rng, side=None, most=LARGEST):
    h = side or rng.choice([7, 14, 28, 56])
    c = 64 * _log(rng, 1, 16)
    return f"{max(1, min(_log(rng, 1, 128), most // (c * h * h)))}x{c}x{h}x{h}"


def _draw_quant(rng):
    case = dict(kind="quant", layout=rng.choice(["flat", "flat", "tiles"]), bits=rng.choice([1, 2, 2, 4, 8]),
                rounding=rng.choice(["nearest", "noise", "philox"]), dtype=rng.choice(["bf16", "bf16", "f32", "f16"]),
                meta=rng.choice(["f32", "bf16"]), out=rng.choice(["bf16", "bf16", "f32"]),
                data=rng.choice(["normal", "relu", "gelu"]))
    e = _log(rng, 1 << 14, LARGEST // (2 if case["dtype"] == "f32" else 1))
    if case["layout"] == "tiles":
        s = rng.choice([8, 16])
        h, w, c = s * rng.randint(1, 7), s * rng.randint(1, 7), _log(rng, 3, 512)
        dims = f"{max(1, min(256, e // (c * h * w)))}x{c}x{h}x{w}"
        return dict(case, group=s * s, dims=dims)
    g, n = rng.choice([64, 128, 256, 512, 1024]), _log(rng, 1, 256)
    return dict(case, group=g, dims=f"{n}x{max(1, e // (n * g)) * g}")


def _draw_saved(rng):
    dims = _dims3(rng) if rng.random() < 0.6 else _dims4(rng)
    return dict(kind="saved_input", dims=dims, bits=rng.choice([1, 2, 2, 2, 4, 8]),
                dtype=rng.choice(["bf16", "bf16", "bf16", "f32"]), data=rng.choice(["normal", "relu", "gelu"]))


def _draw_linear(rng):
    return dict(kind="linear", batch=_log(rng, 1, 128), tokens=_log(rng, 1, 197), fin=64 * _log(rng, 1, 48),
                fout=64 * _log(rng, 1, 48), bits=rng.choice([1, 2, 2, 2, 4, 8]), dtype=rng.choice(["f32", "bf16"]))


def _draw_activation(rng):
    act = rng.choice(["gelu", "silu", "relu", "relu6"])
    relu = act.startswith("relu")
    return dict(kind="activation", act=act, dims=_dims4(rng) if relu else _dims3(rng),
                bits=1 if relu else rng.choice([1, 2, 2, 4, 8]), dtype=rng.choice(["bf16", "bf16", "f32"]))


def _draw_batchnorm(rng):
    h = rng.choice([7, 14, 28, 56, 112, 9, 13, 30])
    c = 16 * _log(rng, 1, 64)
    n = max(1, min(_log(rng, 1, 128), LARGEST // (c * h * h)))
    n = max(16, n // 16 * 16) if rng.random() < 0.6 and 16 * c * h * h <= LARGEST else n
    whole = n * h * h % 64 == 0  # BatchNorm + ReLU takes whole groups only
    return dict(kind="batchnorm", relu=whole and rng.random() < 0.5, dims=f"{n}x{c}x{h}x{h}",
                bits=rng.choice([1, 2, 2, 2, 4, 8]), dtype=rng.choice(["bf16", "bf16", "f32"]))


def _draw_fp8(rng):
    b = rng.choice(["nk", "nk", "kn"])
    k = 16 * _log(rng, 8, 512) if b == "nk" else _log(rng, 128, 8192)
    return dict(kind="fp8", m=_log(rng, 1, 8192), n=_log(rng, 64, 8192), k=k, b=b)


def _draw_vit(rng):
    return dict(kind="vit", batch=rng.randint(8, 96), depth=rng.choice([1, 2]), bits=rng.choice([1, 2, 4, 8]))


def draw(rng):
    return rng.choice([_draw_quant] * 4 + [_draw_saved] * 3 + [_draw_linear] * 4 + [_draw_activation] * 3
                      + [_draw_batchnorm] * 4 + [_draw_fp8] * 4 + [_draw_vit])(rng)


# ----------------------------------------------------------------------------------------- inputs
def _shape(case):
    return tuple(int(v) for v in case["dims"].split("x"))


def _randn(shape, gen, dtype=torch.float32, scale=1.0):
    return torch.randn(shape, generator=gen, device=DEV).mul_(scale).to(dtype)


def _data(case, shape, gen):
    """Activations as layers see them: pre-activations N(0, 1), post-ReLU |N(0, 1)| or GELU(N(0, 1))."""
    x = _randn(shape, gen)
    if case["data"] == "relu":
        x = x.abs_()
    elif case["data"] == "gelu":
        x = F.gelu(x)
    return x.to(DTYPES[case["dtype"]])


def _meta(shape, bits, batchnorm=False, pack_only=False):
    """A layer's meta dict, as the Controller writes it."""
    return {NAME: {"bits": bits, "pack_only": pack_only, "AVG_ALAM": False, "ALAM_BITS": 0, "DIVISION": None,
                   **layer_group_meta(shape, bits, batchnorm=batchnorm)}}


def _linear_inputs(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    x = _randn((case["batch"], case["tokens"], case["fin"]), gen, DTYPES[case["dtype"]])
    dy = _randn((case["batch"], case["tokens"], case["fout"]), gen, torch.bfloat16, 1e-2)
    return x, dy, _randn((case["fout"], case["fin"]), gen, scale=0.02), _randn((case["fout"],), gen, scale=0.02)


def _activation_inputs(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    shape = _shape(case)
    scale = 3.0 if case["act"] == "relu6" else 1.0
    return _randn(shape, gen, DTYPES[case["dtype"]], scale), _randn(shape, gen, torch.bfloat16)


def _batchnorm_inputs(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    shape = _shape(case)
    c = shape[1]
    mean, std = _randn((1, c, 1, 1), gen, scale=0.5), torch.rand((1, c, 1, 1), generator=gen, device=DEV) + 0.5
    x = _randn(shape, gen).mul_(std).add_(mean).to(DTYPES[case["dtype"]])
    dy = _randn(shape, gen, torch.bfloat16)
    return x, dy, torch.rand(c, generator=gen, device=DEV) + 0.5, _randn((c,), gen, scale=0.5)


def _fp8_inputs(case, seed):
    """N(0, 1) operands quantized to e4m3 with per-tensor scales, and the scale of their product."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    kn = case["b"] == "kn"
    a = _randn((case["m"], case["k"]), gen)
    b = _randn((case["k"], case["n"]) if kn else (case["n"], case["k"]), gen)
    scale = 448.0 / 6.5  # covers |N(0, 1)| at these sizes: a calibrated scale, known on the host
    a8, b8 = (t.mul_(scale).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn) for t in (a, b))
    return a8, b8, 1.0 / (scale * scale)


def _vit_weights(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    d, h = 768, 3072

    def w(*shape):
        return _randn(shape, gen, scale=0.02)

    p = {"cls_token": w(1, 1, d), "pos_embed": w(1, 197, d), "patch_embed.proj.weight": w(d, 3, 16, 16),
         "patch_embed.proj.bias": w(d), "norm.weight": 1 + w(d), "norm.bias": w(d), "head.weight": w(1000, d),
         "head.bias": w(1000)}
    for i in range(case["depth"]):
        for name, rows, cols in (("attn.qkv", 3 * d, d), ("attn.proj", d, d), ("mlp.fc1", h, d), ("mlp.fc2", d, h)):
            p[f"blocks.{i}.{name}.weight"], p[f"blocks.{i}.{name}.bias"] = w(rows, cols), w(rows)
        for name in ("norm1", "norm2"):
            p[f"blocks.{i}.{name}.weight"], p[f"blocks.{i}.{name}.bias"] = 1 + w(d), w(d)
    images = _randn((case["batch"], 3, 224, 224), gen)
    return p, images, torch.randint(0, 1000, (case["batch"],), generator=gen, device=DEV)


def _prepare_quant(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    shape, g = _shape(case), case["group"]
    x = _data(case, shape, gen)
    if case["layout"] == "flat":
        x = x.view(shape[0], -1, g)
    noise = None
    if case["rounding"] == "noise":
        noise = torch.rand((shape[0], x.numel() // shape[0] // g, g), generator=gen, device=DEV)
    return {"x": x, "noise": noise}


def _prepare_saved(case, seed):
    x = _data(case, _shape(case), torch.Generator(device=DEV).manual_seed(seed))
    return {"x": x, "meta": _meta(_shape(case), case["bits"])}


def _prepare_linear(case, seed):
    x, dy, w, b = _linear_inputs(case, seed)
    layer = DOLinear(case["fin"], case["fout"], target_name=NAME, meta=_meta(x.shape, case["bits"]), device=DEV).train()
    with torch.no_grad():
        layer.weight.copy_(w)
        layer.bias.copy_(b)
    return {"x": x.requires_grad_(True), "dy": dy, "layer": layer}


def _prepare_activation(case, seed):
    x, dy = _activation_inputs(case, seed)
    act = case["act"]
    kw = dict(target_name=NAME, meta=_meta(x.shape, case["bits"], pack_only=act.startswith("relu")))
    if act in ("gelu", "silu"):
        layer = (DOGELU if act == "gelu" else DOSiLU)(**kw)
    else:
        layer = DOReLU_Variance(relu=act == "relu", relu6=act == "relu6", **kw)
    return {"x": x.requires_grad_(True), "dy": dy, "layer": layer.train()}


def _prepare_batchnorm(case, seed):
    x, dy, w, b = _batchnorm_inputs(case, seed)
    cls = DOBatchNormReLU2d if case["relu"] else DOBatchNorm2d
    layer = cls(x.shape[1], target_name=NAME, meta=_meta(x.shape, case["bits"], batchnorm=True), device=DEV).train()
    with torch.no_grad():
        layer.weight.copy_(w)
        layer.bias.copy_(b)
    return {"x": x.requires_grad_(True), "dy": dy.to(torch.bfloat16), "layer": layer}


def _prepare_fp8(case, seed):
    a, b, scale = _fp8_inputs(case, seed)
    return {"a": a, "b": b, "scale": scale}


def _prepare_vit(case, seed):
    p, images, labels = _vit_weights(case, seed)
    with torch.device(DEV):
        model = VisionTransformer(depth=case["depth"])
    model.load_state_dict(p)
    ctl = Controller(model.train(), {"batch_size": case["batch"], "default_bits": case["bits"]},
                     input_shape=(3, 224, 224))
    return {"model": ctl.warp_model(quantizer=True), "images": images, "labels": labels}


_PREPARE = {"quant": _prepare_quant, "saved_input": _prepare_saved, "linear": _prepare_linear,
            "activation": _prepare_activation, "batchnorm": _prepare_batchnorm, "fp8": _prepare_fp8,
            "vit": _prepare_vit}


def prepare(case, seed):
    return {"case": dict(case), **_PREPARE[case["kind"]](case, seed)}


# -------------------------------------------------------------------------------------- one pass
def _run_quant(s, case):
    ops = torch.ops.act_lib
    x, g, bits, meta, out = s["x"], case["group"], case["bits"], DTYPES[case["meta"]], DTYPES[case["out"]]
    args = (bits, g, False, 0.0, False, ROUNDING[case["rounding"]], s["noise"], SEED, OFFSET, meta)
    if case["layout"] == "tiles":
        packed, scale, xmin = ops.quant_pack_tiles(x, *args)
        restored = ops.dequant_unpack_tiles(packed, scale, xmin, bits, g, *x.shape, out)
    else:
        packed, scale, xmin = ops.quant_pack(x, *args)
        restored = ops.dequant_unpack(packed, scale, xmin, bits, g, out)
    return {"packed": packed, "scale": scale, "min": xmin, "restored": restored}


def _run_saved(s, case):
    q, q_meta, _ = unified_quantize(s["x"], None, NAME, s["meta"], clamp=True, clamp_alpha=3.0)
    return {"packed": q[0], "scale": q[1], "min": q[2], "restored": unified_dequantize(q, q_meta, None)}


def _run_layer(s, case):
    x, layer = s["x"], s["layer"]
    x.grad = None
    for p in layer.parameters():
        p.grad = None
    if case["kind"] == "linear":
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = layer(x)
    else:
        y = layer(x)
    y.backward(s["dy"])
    out = {"y": y, "dx": x.grad, **{f"d{n}": p.grad for n, p in layer.named_parameters()}}
    if case["kind"] == "batchnorm":
        out.update(running_mean=layer.running_mean, running_var=layer.running_var)
    return out


def _run_fp8(s, case):
    op = torch.ops.act_lib.fp8_linear if case["b"] == "kn" else torch.ops.act_lib.fp8_gemm_nt
    return op(s["a"], s["b"], s["scale"])


def _run_vit(s, case):
    model = s["model"]
    for p in model.parameters():
        p.grad = None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        logits = model(s["images"])
        loss = F.cross_entropy(logits, s["labels"])
    loss.backward()
    return {"logits": logits, "loss": loss, "grads": {n: p.grad for n, p in model.named_parameters()}}


_RUN = {"quant": _run_quant, "saved_input": _run_saved, "linear": _run_layer, "activation": _run_layer,
        "batchnorm": _run_layer, "fp8": _run_fp8, "vit": _run_vit}


def run(state):
    return _RUN[state["case"]["kind"]](state, state["case"])


# ------------------------------------------------------------------------ what a pass cannot avoid
def work(case):
    """Bytes: every input read once, every output (saved codes, scale and min among them) written once
    and the saved ones read back once. Flops: those of the contractions, and a few per element."""
    kind, bits = case["kind"], case.get("bits", 0)
    if kind == "fp8":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": m * k + n * k + 2 * m * n, "flops": 2 * m * n * k}
    if kind == "linear":
        rows, fin, fout = case["batch"] * case["tokens"], case["fin"], case["fout"]
        g = layer_group_meta((case["batch"], case["tokens"], fin), bits)["group_size"]
        saved = rows * fin * (bits / 8 + 4 / g)
        return {"bytes": rows * fin * 2 * BYTES[case["dtype"]] + rows * fout * 4 + fin * fout * 12 + 2 * saved,
                "flops": 6 * rows * fin * fout}
    if kind == "vit":
        rows, params = case["batch"] * 197, 12 * 768 * 768 * case["depth"]
        attention = 3.5 * 4 * case["batch"] * 197 * 197 * 768 * case["depth"]
        activations = rows * 768 * case["depth"] * (16 * 2 + 10 * bits / 8)
        return {"bytes": case["batch"] * 3 * 224 * 224 * 4 + 8 * params + 2 * activations,
                "flops": 6 * rows * params + attention + 4 * rows * 768 * 768}
    shape = _shape(case)
    e = math.prod(shape)
    if kind == "quant":
        saved = e * bits / 8 + e / case["group"] * 2 * BYTES[case["meta"]]
        noise = 4 * e if case["rounding"] == "noise" else 0
        return {"bytes": e * (BYTES[case["dtype"]] + BYTES[case["out"]]) + noise + 2 * saved, "flops": 6 * e}
    g = layer_group_meta(shape, bits, batchnorm=kind == "batchnorm")["group_size"]
    if kind == "saved_input":
        return {"bytes": e * (BYTES[case["dtype"]] + 2) + 2 * e * (bits / 8 + 4 / g), "flops": 20 * e}
    saved = e * bits / 8 if case.get("act", "").startswith("relu") else e * (bits / 8 + 4 / g)
    if kind == "batchnorm" and case["relu"]:
        saved += e / 8
    # x in, y out, dy in, dx out (in x's type)
    relu_y = BYTES[case["dtype"]] if case.get("act", "").startswith("relu") else 2
    return {"bytes": e * (2 * BYTES[case["dtype"]] + relu_y + 2) + 2 * saved, "flops": 20 * e}


def tolerance(case):
    """quant: fixed arithmetic, bit for bit. The others: bf16 outputs whose last bit depends on the order
    of 32-bit sums, and codes of squashed values that may fall on either side of a tie (one code is one
    step of the restored value, hence the wide "max" there). FP8: the last bf16 bit of a 32-bit sum."""
    kind = case["kind"]
    if kind == "quant":
        return "exact"
    if kind == "saved_input":
        return {"rel": 2e-3, "max": 0.9, "differ": 1e-3}
    if kind == "activation":
        return {"rel": 2e-3, "max": 0.9}
    if kind == "linear":
        return {"rel": 5e-3, "max": 0.05}
    if kind == "batchnorm":
        return {"rel": 2e-3, "max": 0.05}
    if kind == "fp8":
        return {"rel": 2e-3, "max": 0.02}
    return {"rel": 0.02, "max": 0.5}


# ---------------------------------------------------------------------------------------- 64 bits
def _bf16(t):
    return t.to(torch.bfloat16).double()


def _codes(t, bits, u=None, floor=0.0):
    """Per-group (last axis) min, step and codes of 64-bit values; u: the stochastic rounding's noise."""
    mn, mx = t.amin(-1, keepdim=True), t.amax(-1, keepdim=True)
    rng, qmax = (mx - mn).clamp_min(floor), 2 ** bits - 1
    step = torch.where(rng > 0, rng / qmax, torch.ones_like(rng))
    arg = (t - mn) / step
    q = torch.floor(arg + HALF) if u is None else torch.round(arg + u - 0.5)
    return mn, step, q.clamp_(0, qmax)


def _group(t, case, g, padded=False, tiles=False):
    """t's values as [N, G, g], and the way back."""
    n = t.shape[0]
    if tiles:
        s = int(math.isqrt(g))
        c, h, w = t.shape[1:]
        v = t.view(n, c, h // s, s, w // s, s).permute(0, 1, 2, 4, 3, 5).reshape(n, -1, g)
        return v, lambda r: (r.view(n, c, h // s, w // s, s, s).permute(0, 1, 2, 4, 3, 5).reshape(t.shape))
    flat = t.reshape(n, -1)
    per = flat.shape[1]
    if padded:
        flat = F.pad(flat, (0, -per % g))
    return flat.reshape(n, -1, g), lambda r: r.reshape(n, -1)[:, :per].reshape(t.shape)


def _saved_exact(x, bits):
    """(scale, min, restored) of the layers' saved input: clamp, squash, codes, bf16 scale / min."""
    m = layer_group_meta(x.shape, bits)
    g, s = m["group_size"], int(math.isqrt(m["group_size"]))
    tiles = (not m["act_padding"] and x.dim() == 4 and s * s == g and x.shape[2] % s == 0 and x.shape[3] % s == 0)
    v, back = _group(x.double(), None, g, m["act_padding"], tiles)
    mn, step, q = _codes(torch.tanh(2 * v.clamp_(-3.0, 3.0)) / 2, bits)
    restored = back(q * _bf16(step) + _bf16(mn))
    return step.squeeze(-1), mn.squeeze(-1), restored


def _exact_quant(case, seed):
    s = _prepare_quant(case, seed)
    v, back = _group(s["x"].double(), case, case["group"], tiles=case["layout"] == "tiles")
    u = s["noise"].double() if s["noise"] is not None else None
    mn, step, q = _codes(v, case["bits"], u)
    out = {"packed": None, "scale": step.squeeze(-1), "min": mn.squeeze(-1), "restored": None}
    if case["rounding"] != "philox":
        if case["meta"] == "bf16":
            step, mn = _bf16(step), _bf16(mn)
        out["restored"] = back(q * step + mn)
    return out


def _exact_saved(case, seed):
    scale, mn, restored = _saved_exact(_prepare_saved(case, seed)["x"], case["bits"])
    return {"packed": None, "scale": scale, "min": mn, "restored": restored}


def _exact_linear(case, seed):
    x, dy, w, b = _linear_inputs(case, seed)
    x, w, b, dyd = x.to(torch.bfloat16), _bf16(w), _bf16(b), dy.double().reshape(-1, case["fout"])
    x_hat = _bf16(_saved_exact(x, case["bits"])[2]).reshape(-1, case["fin"])
    return {"y": x.double() @ w.t() + b, "dx": (dyd @ w).view(x.shape), "dweight": dyd.t() @ x_hat, "dbias": dyd.sum(0)}


def _exact_activation(case, seed):
    x, dy = _activation_inputs(case, seed)
    act, v, dyd = case["act"], x.double(), dy.double()
    if act.startswith("relu"):
        on = (v > 0) if act == "relu" else (v > 0) & (v < 6)
        return {"y": torch.where(on, v, 0.0), "dx": dyd * on}
    if act == "gelu":
        a, b = math.sqrt(2 / math.pi), 0.044715
        t = torch.tanh(a * (v + b * v ** 3))
        y, d = v * (1 + t) / 2, (1 + t) / 2 + v * (1 - t * t) * a * (1 + 3 * b * v * v) / 2
    else:
        s = torch.sigmoid(v)
        y, d = v * s, s + v * s * (1 - s)
    g = layer_group_meta(x.shape, case["bits"])["group_size"]
    grouped, back = _group(torch.tanh(2 * d.clamp(-3.0, 3.0)) / 2, case, g)
    mn, step, q = _codes(grouped, case["bits"], floor=1e-4)
    return {"y": y, "dx": dyd * back(q * _bf16(step) + _bf16(mn))}


def _exact_batchnorm(case, seed):
    x, dy, w, b = _batchnorm_inputs(case, seed)
    n, c, h, wd = x.shape
    m = n * h * wd
    meta = layer_group_meta(x.shape, case["bits"], batchnorm=True)
    col = (1, c, 1, 1)
    v, dyd, w, b = x.double(), dy.double(), w.double().view(col), b.double().view(col)
    mean, var = v.mean((0, 2, 3), keepdim=True), v.var((0, 2, 3), unbiased=False, keepdim=True)
    xh = (v - mean) / torch.sqrt(var + (1e-5 if not meta["act_padding"] or case["relu"] else 1e-7))
    del v
    y = xh * w + b
    if case["relu"]:
        on = y > 0
        y, dyd = torch.where(on, y, 0.0), dyd * on
        t = xh
    elif meta["act_padding"]:
        y = torch.where(torch.isnan(y), 0.0, y)
        return {"y": y, "dx": None, "dweight": None, "dbias": dyd.sum((0, 2, 3)),
                "running_mean": 0.1 * mean.flatten(), "running_var": 0.9 + 0.1 * var.flatten()}
    else:
        t = 2 * torch.tanh(xh.clamp(-3.0, 3.0) / 2)
    chan = t.transpose(0, 1).reshape(c, -1, meta["group_size"] // 2)
    mn, step, q = _codes(chan, case["bits"])
    saved = (q * _bf16(step) + _bf16(mn)).reshape(c, n, h, wd).transpose(0, 1)
    db, dw = dyd.sum((0, 2, 3), keepdim=True), (dyd * saved).sum((0, 2, 3), keepdim=True)
    inv = 1 / torch.sqrt(var + (1e-5 if case["relu"] else 1e-7))
    dx = (dyd - db / m - saved * dw / m) * w * inv
    return {"y": y, "dx": dx, "dweight": dw.flatten(), "dbias": db.flatten(), "running_mean": 0.1 * mean.flatten(),
            "running_var": 0.9 + 0.1 * var.flatten()}


def _exact_fp8(case, seed):
    a, b, scale = _fp8_inputs(case, seed)
    a, b = a.float().double(), b.float().double()
    return (a @ (b if case["b"] == "kn" else b.t())) * scale


def _exact_vit(case, seed):
    """The forward (the compression only touches what the backward reads)."""
    p, images, labels = _vit_weights(case, seed)
    p = {k: v.double() for k, v in p.items()}
    x = F.conv2d(images.double(), p["patch_embed.proj.weight"], p["patch_embed.proj.bias"], stride=16)
    x = x.flatten(2).transpose(1, 2)
    x = torch.cat([p["cls_token"].expand(x.shape[0], -1, -1), x], 1) + p["pos_embed"]
    n, t, d = x.shape

    def norm(x, name):
        return F.layer_norm(x, (d,), p[name + ".weight"], p[name + ".bias"], 1e-6)

    def linear(x, name):
        return x @ p[name + ".weight"].t() + p[name + ".bias"]

    for i in range(case["depth"]):
        at = f"blocks.{i}."
        q, k, v = linear(norm(x, at + "norm1"), at + "attn.qkv").view(n, t, 3, 12, 64).permute(2, 0, 3, 1, 4).unbind(0)
        a = torch.softmax(q @ k.transpose(-1, -2).contiguous() / 8.0, -1) @ v
        x = x + linear(a.transpose(1, 2).reshape(n, t, d), at + "attn.proj")
        x = x + linear(F.gelu(linear(norm(x, at + "norm2"), at + "mlp.fc1"), approximate="tanh"), at + "mlp.fc2")
    logits = linear(norm(x, "norm")[:, 0], "head")
    return {"logits": logits, "loss": F.cross_entropy(logits, labels), "grads": None}


_EXACT = {"quant": _exact_quant, "saved_input": _exact_saved, "linear": _exact_linear,
          "activation": _exact_activation, "batchnorm": _exact_batchnorm, "fp8": _exact_fp8, "vit": _exact_vit}


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)
