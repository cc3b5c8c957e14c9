"""Performance cases of the packed ARCQ path: what users of this package have it do, through its public modules and
operators.

A case is a dict of plain values; ``listed()`` names the fixed ones, ``draw(rng)`` takes another one from the same
ranges.  ``prepare`` builds what a user's program holds before a call (model or layer, input tensors), ``run`` is one
pass through the public entry point.  Everything is called eagerly on torch's current stream, the way ``model(images)``
is called by a script; host time per call is therefore part of what a small case measures.

Kinds
-----
model      whole ViT forward with packed block linears (``vit.VisionTransformer``): images in, logits out
layer      one ``ARCQPackedLinearOnTheFly`` call on a batch of tokens
format     one ``ARCQPackedLinear`` call in one of its runtime formats (``packed``, ``u8``, ``dequant_gemm``, ``hip_fused``)
quantize   ``ops.quantize_activation``: activations to packed codes and per-group metadata (the encoding direction)
patch      ``ARCQPackedPatchConv``: quantized patch embedding of a batch of images
"""
import torch

from arcq_vit_amd import ops, synth, vit
from arcq_vit_amd.packed_conv import ARCQPackedPatchConv
from arcq_vit_amd.packed_convert import set_fp8_operands, share_buffers
from arcq_vit_amd.packed_linear import ARCQPackedLinear
from arcq_vit_amd.packed_on_the_fly import ARCQPackedLinearOnTheFly
from arcq_vit_amd.quant_source import QuantConv2dPCARCQ, QuantLinearPCARCQ

GROUP = 64
DEVICE = "cuda"
CLASSES = 1000


def listed():
    return [
        # The single layer of the first baseline configuration (fc1 of the tiny model, one image): the smallest call,
        # what a user's unit test or a latency-bound service of one layer pays.
        {"name": "layer_tiny_b1", "kind": "layer", "m": 197, "k": 192, "n": 768, "bits": 4, "x": "f16", "shared": True},
        # One image through the small model, all fusions on: interactive latency.
        {"name": "small_b1", "kind": "model", "model": "deit_small", "batch": 1, "bits": 4, "image": 224, "fused": True,
         "fp8": False},
        # The headline batch of the small model.
        {"name": "small_b64", "kind": "model", "model": "deit_small", "batch": 64, "bits": 4, "image": 224, "fused": True,
         "fp8": False},
        # The builder's default options (every LayerNorm, GELU, skip connection and the attention as torch runs them; no
        # shared buffers), an odd batch, three-bit codes.
        {"name": "small_b17_defaults", "kind": "model", "model": "deit_small", "batch": 17, "bits": 3, "image": 224,
         "fused": False, "fp8": False},
        # The base model at its configured batch.
        {"name": "base_b64", "kind": "model", "model": "deit_base", "batch": 64, "bits": 4, "image": 224, "fused": True,
         "fp8": False},
        # The large model at its configured batch: the largest case, bound by the matrix units.
        {"name": "large_b256", "kind": "model", "model": "vit_large", "batch": 256, "bits": 3, "image": 224, "fused": True,
         "fp8": False},
        # FP8 operands (the opt-in for throughput on the wide models), a moderate serving batch.
        {"name": "base_b32_fp8", "kind": "model", "model": "deit_base", "batch": 32, "bits": 4, "image": 224, "fused": True,
         "fp8": True},
        # The two formats the converter writes, and the byte-code one, as a converted checkpoint's layers are called: fp32
        # tokens in, fp32 out.
        {"name": "format_packed", "kind": "format", "format": "packed", "m": 1576, "k": 384, "n": 1536, "bits": 4},
        {"name": "format_dequant_gemm", "kind": "format", "format": "dequant_gemm", "m": 12608, "k": 1536, "n": 384,
         "bits": 4},
        {"name": "format_u8", "kind": "format", "format": "u8", "m": 394, "k": 768, "n": 768, "bits": 3},
        # Encoding a batch of activations (the reference extension's own operator).
        {"name": "quantize_b64", "kind": "quantize", "m": 12608, "k": 1536, "bits": 4},
        # Quantized patch embedding, an evaluation batch.
        {"name": "patch_b64", "kind": "patch", "batch": 64, "n": 384, "bits": 4, "image": 224, "x": "f16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One more case.  Batches, rows and widths are spread over their logarithm; odd and ragged sizes are as likely as
    round ones."""
    kind = rng.choices(["model", "layer", "format", "quantize", "patch"], [8, 4, 4, 2, 2])[0]
    bits = rng.choice([2, 3, 4])
    if kind == "model":
        image = rng.choice([224, 224, 224, 160, 192, 256])
        tokens = 1 + (image // 16) ** 2
        fp8 = rng.random() < 0.2
        return {"kind": "model", "model": rng.choice(["deit_tiny", "deit_small", "deit_base", "vit_large"]),
                "batch": _log_int(rng, 1, 50432 // tokens), "bits": bits, "image": image,
                "fused": fp8 or rng.random() < 0.75, "fp8": fp8}
    if kind == "layer":
        return {"kind": "layer", "m": _log_int(rng, 1, 50432), "k": 64 * _log_int(rng, 2, 64),
                "n": rng.choice([32, 32, 32, 8, 1]) * _log_int(rng, 4, 128), "bits": bits, "x": rng.choice(["f16", "f16", "f32"]),
                "shared": rng.random() < 0.75}
    if kind == "format":
        fmt = rng.choice(["packed", "u8", "dequant_gemm", "hip_fused"])
        return {"kind": "format", "format": fmt, "m": _log_int(rng, 1, 12608 if fmt in ("packed", "u8") else 50432),
                "k": 64 * _log_int(rng, 2, 24), "n": rng.choice([32, 32, 8]) * _log_int(rng, 6, 48), "bits": bits}
    if kind == "quantize":
        return {"kind": "quantize", "m": _log_int(rng, 1, 50432), "k": 64 * _log_int(rng, 1, 64), "bits": bits}
    return {"kind": "patch", "batch": _log_int(rng, 1, 256), "n": 32 * _log_int(rng, 6, 32), "bits": bits,
            "image": rng.choice([224, 224, 160, 192, 256]), "x": rng.choice(["f16", "f16", "f32"])}


# ---- making the inputs -------------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _activation(m, k, g, dtype):
    """Post-LayerNorm-like tokens, N(0, 1) with 0.5 % of outliers at +-8; wide inputs (k >= 1536: behind a GELU in the
    models that have them) GELU of N(0, 1.5^2)."""
    x = torch.randn(m, k, generator=g, device=DEVICE)
    if k >= 1536:
        return torch.nn.functional.gelu(1.5 * x).to(dtype)
    u = torch.rand(m, k, generator=g, device=DEVICE)
    return torch.where(u < 0.005, torch.where(u < 0.0025, -8.0, 8.0), x).to(dtype)


def _source(layer, weight, bits, g):
    """A trained fake-quant layer on the device, as the converter finds it: weights N(0, 0.02^2), bias N(0, 0.01^2)."""
    with torch.no_grad():
        weight.copy_(torch.randn(weight.shape, generator=g, device=DEVICE) * 0.02)
        inner = layer.conv if hasattr(layer, "conv") else layer.linear
        inner.bias.copy_(torch.randn(inner.bias.shape, generator=g, device=DEVICE) * 0.01)
    cb = synth.quantile_codebook(bits).to(DEVICE)
    layer.act_quant.set_codebook(cb)
    layer.weight_quant.set_codebook(cb)
    return layer


def _packed(n, k, bits, g, runtime_code_format="packed"):
    with torch.device(DEVICE):
        layer = QuantLinearPCARCQ(k, n, True, bits, bits, GROUP)
    return ARCQPackedLinear(_source(layer, layer.linear.weight, bits, g), runtime_code_format)


def _on_the_fly(n, k, bits, g):
    return ARCQPackedLinearOnTheFly.from_packed(_packed(n, k, bits, g))


def _images(batch, size, g, dtype):
    """U(0, 1) images normalised with the ImageNet mean and deviation."""
    x = torch.rand(batch, 3, size, size, generator=g, device=DEVICE)
    mean = torch.tensor(synth.IMAGENET_MEAN, device=DEVICE).view(1, 3, 1, 1)
    std = torch.tensor(synth.IMAGENET_STD, device=DEVICE).view(1, 3, 1, 1)
    return ((x - mean) / std).to(dtype)


def _model(case, g):
    d = synth.MODEL_DIMS[case["model"]]
    net = vit.VisionTransformer(d["dim"], d["depth"], d["heads"], d["mlp"], CLASSES, img=case["image"],
                                linear=lambda k, n, bias: _on_the_fly(n, k, case["bits"], g))
    net = net.to(DEVICE)
    with torch.no_grad():
        for name, p in net.named_parameters():
            if p.dim() >= 2:
                p.copy_(torch.randn(p.shape, generator=g, device=DEVICE) * 0.02)
            elif name.endswith("bias"):
                p.copy_(torch.randn(p.shape, generator=g, device=DEVICE) * 0.01)
    net = net.half().eval()
    if case["fused"]:
        share_buffers(net, case["batch"] * (1 + (case["image"] // 16) ** 2))
        for block in net.blocks:
            block.fuse_elementwise = True
            block.attn.own_kernel = True
        net.own_patch_embed = True
    if case["fp8"]:
        set_fp8_operands(net)
    return net


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "model":
        return {"call": _model(case, g), "x": _images(case["batch"], case["image"], g, torch.float16)}
    if kind == "layer":
        layer = _on_the_fly(case["n"], case["k"], case["bits"], g)
        if case["shared"]:
            share_buffers(layer, case["m"])
        return {"call": layer, "x": _activation(case["m"], case["k"], g, torch.float16 if case["x"] == "f16" else torch.float32)}
    if kind == "format":
        layer = _packed(case["n"], case["k"], case["bits"], g, case["format"])
        return {"call": layer, "x": _activation(case["m"], case["k"], g, torch.float32)}
    if kind == "quantize":
        bits = case["bits"]
        cb = synth.quantile_codebook(bits)
        thr = synth.midpoint_thresholds(cb).to(DEVICE)
        cb = cb.to(DEVICE)
        return {"call": lambda x: ops.quantize_activation(x, thr, cb, bits, GROUP),
                "x": _activation(case["m"], case["k"], g, torch.float32)}
    with torch.device(DEVICE):
        conv = QuantConv2dPCARCQ(3, case["n"], 16, 16, 0, True, case["bits"], case["bits"], GROUP)
    return {"call": ARCQPackedPatchConv(_source(conv, conv.conv.weight, case["bits"], g)),
            "x": _images(case["batch"], case["image"], g, torch.float16 if case["x"] == "f16" else torch.float32)}


def run(state):
    with torch.no_grad():
        return state["call"](state["x"])


# ---- what a pass cannot do without ---------------------------------------------------------------------------------
def _weight_bytes(n, k, bits):
    return n * k * bits // 8 + 12 * n * (k // GROUP) + 4 * n


def work(case):
    kind, bits = case["kind"], case["bits"]
    if kind == "model":
        d = synth.MODEL_DIMS[case["model"]]
        b, dim, depth = case["batch"], d["dim"], d["depth"]
        tokens = 1 + (case["image"] // 16) ** 2
        m = b * tokens
        linears = [(k, n) for _, k, n in synth.block_linear_shapes(case["model"])]
        weights = depth * sum(_weight_bytes(n, k, bits) for k, n in linears) + 2 * dim * (768 + tokens + CLASSES)
        flops = depth * (sum(2 * m * n * k for k, n in linears) + 4 * b * tokens * tokens * dim)
        flops += 2 * (m - b) * 768 * dim + 2 * b * dim * CLASSES
        return {"bytes": weights + 2 * b * (3 * case["image"] ** 2 + CLASSES), "flops": flops}
    if kind in ("layer", "format"):
        m, n, k = case["m"], case["n"], case["k"]
        size_in = 2 if case.get("x") == "f16" else 4
        size_out = 2 if kind == "layer" else 4
        return {"bytes": _weight_bytes(n, k, bits) + size_in * m * k + size_out * m * n, "flops": 2 * m * n * k}
    if kind == "quantize":
        m, k = case["m"], case["k"]
        return {"bytes": 4 * m * k + m * k * bits // 8 + 12 * m * (k // GROUP), "flops": 0}
    size = 2 if case["x"] == "f16" else 4
    m = case["batch"] * (case["image"] // 16) ** 2
    return {"bytes": _weight_bytes(case["n"], 768, bits) + size * (m * 768 + m * case["n"]), "flops": 2 * m * 768 * case["n"]}


def tolerance(case):
    kind = case["kind"]
    if kind == "model":
        # A value that another order of summation moves across a quantization threshold changes by a whole level in the
        # layers behind it, so whole models differ by more than their fp16 arithmetic does.
        return {"rel": 0.03 if case["fp8"] else 0.02, "max": 0.3}
    if kind == "quantize":
        return "exact"                      # codes and metadata are defined bit for bit
    if kind == "format" and case["format"] in ("packed", "u8"):
        return {"rel": 1.0e-5}              # sums of products in 64 / 32 bits, outputs in 32
    if kind == "format":
        return {"rel": 1.0e-5, "max": 1.0e-3}    # products of fp16 operands summed in 32 bits, outputs in 32
    return {"rel": 1.0e-3, "max": 4.0e-3}        # the same, rounded to fp16
