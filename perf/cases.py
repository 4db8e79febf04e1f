"""The work that programs have this library do, as cases that can be timed and checked.

Whole depth inferences through the public inference entries, and the layers
they are made of through the operator surface (include/dav2_ops.h) and the
launcher layer (include/dav2_hip.h), over image sizes from thumbnails to
1036 pixels, all three encoders and every precision mode:

  model       one call of dav2_infer_tensor_f32 (host buffers), of its batched
              device-resident variant, or of the variant that returns logits
  linear_i8   dav2_ops_linear_int8: row quantization + int8 GEMM (+ GELU)
  attn_i8     dav2_hip_attention_fused: the int8 mode's attention
  conv_i8     dav2_ops_conv2d_int8: 3x3 convolutions of the DPT head
  linear_f32  dav2_ops_linear: the fp32 mode's linears
  conv_f32    dav2_ops_conv2d: the fp32 / fp16 modes' convolutions
  attn_ref    dav2_ops_attention_head64: attention in the reference's own order
  resize      dav2_ops_bilinear_align_true: the DPT's upsampling

Models have random weights of the official shapes; LayerScale, LayerNorm and
biases are spread as in trained networks (the encoder's blocks matter to the
output). The int8 path promises the same bits for the same input, so its
cases are "exact"; the float modes state a relative error.
"""

from __future__ import annotations

import importlib.util
import math
import sys
import tempfile
from pathlib import Path

import numpy as np
import torch
import torch.nn.functional as F

ROOT = Path(__file__).resolve().parents[1]


def _package():
    if "dav2_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location("dav2_amd", ROOT / "depth-anything-v2_amd" / "__init__.py")
        mod = importlib.util.module_from_spec(spec)
        sys.modules["dav2_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["dav2_amd"]


MODES = {"int8": "FORCE_INT8", "fp16": "FORCE_FP16", "fp32": "FORCE_FP32"}
CAPTURE = {"vits": (2, 5, 8, 11), "vitb": (2, 5, 8, 11), "vitl": (4, 11, 17, 23)}


def listed():
    return [
        # a thumbnail through the smallest encoder: the latency of one host call
        dict(name="vits_252x196_host", kind="model", encoder="vits", mode="int8", entry="host", batch=1, width=252,
             height=196),
        # the headline call: one 518x518 image, host buffers
        dict(name="vitl_518_host", kind="model", encoder="vitl", mode="int8", entry="host", batch=1, width=518,
             height=518),
        # a serving loop's batch, device resident
        dict(name="vitl_518_b8_device", kind="model", encoder="vitl", mode="int8", entry="device", batch=8, width=518,
             height=518),
        # the two float modes, logits returned
        dict(name="vitb_518_fp16_logits", kind="model", encoder="vitb", mode="fp16", entry="logits", batch=1, width=518,
             height=518),
        dict(name="vitb_686x518_fp32_logits", kind="model", encoder="vitb", mode="fp32", entry="logits", batch=1,
             width=686, height=518),
        # ViT-L's fc1 on one 518x518 image
        dict(name="linear_i8_1370x1024x4096_gelu", kind="linear_i8", rows=1370, k=1024, n=4096, gelu=True),
        # ViT-L attention on a 16:9 video frame (924x518: 66x37 patches + class token)
        dict(name="attn_i8_2443x16", kind="attn_i8", tokens=2443, heads=16, batch=1),
        # ViT-L refinenet1's 3x3 convolution at 518x518
        dict(name="conv_i8_148_256_256", kind="conv_i8", width=148, height=148, channels=256, out_channels=256,
             kernel=3),
        # ViT-L's fc1 in the fp32 mode
        dict(name="linear_f32_1370x1024x4096_gelu", kind="linear_f32", rows=1370, k=1024, n=4096, gelu=True),
        # ViT-B refinenet1's 3x3 convolution at 518x518 in the float modes
        dict(name="conv_f32_148_128_128", kind="conv_f32", width=148, height=148, channels=128, out_channels=128,
             kernel=3),
        # the reference's binary16 attention, ViT-B at 518x518
        dict(name="attn_ref_fp16_1370x12", kind="attn_ref", tokens=1370, heads=12, precision="fp16"),
        # ViT-L's last upsampling, 296 -> 518
        dict(name="resize_296_518_128", kind="resize", width=296, height=296, out_width=518, out_height=518,
             channels=128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["model", "model", "model", "linear_i8", "attn_i8", "conv_i8", "linear_f32", "conv_f32",
                       "attn_ref", "resize"])
    dim, heads = rng.choice([(384, 6), (768, 12), (1024, 16)])
    while True:
        if kind == "model":
            mode = rng.choice(["int8", "int8", "int8", "fp16", "fp32"])
            entry = rng.choice(["host", "device"]) if mode == "int8" else "logits"
            case = dict(kind=kind, encoder=rng.choice(["vits", "vitb", "vitl"]), mode=mode, entry=entry,
                        batch=rng.randint(1, 8) if entry == "device" else 1, width=14 * _log_int(rng, 6, 74),
                        height=14 * _log_int(rng, 5, 74))
        elif kind in ("linear_i8", "linear_f32"):
            k, n, gelu = rng.choice([(dim, 3 * dim, False), (dim, dim, False), (dim, 4 * dim, True),
                                     (4 * dim, dim, False)])
            case = dict(kind=kind, rows=_log_int(rng, 31, 11000 if kind == "linear_i8" else 5500), k=k, n=n, gelu=gelu)
        elif kind == "attn_i8":
            case = dict(kind=kind, tokens=_log_int(rng, 31, 5477), heads=heads, batch=rng.choice([1, 1, 2, 4, 8]))
        elif kind == "attn_ref":
            case = dict(kind=kind, tokens=_log_int(rng, 31, 2443), heads=heads, precision=rng.choice(["fp16", "fp32"]))
        elif kind in ("conv_i8", "conv_f32"):
            c, oc = rng.choice([(64, 64), (128, 128), (256, 256), (256, 128), (128, 64), (128, 32), (64, 32)])
            case = dict(kind=kind, width=_log_int(rng, 12, 518), height=_log_int(rng, 12, 518), channels=c,
                        out_channels=oc, kernel=rng.choice([3, 3, 3, 1]))
        else:
            w, h = _log_int(rng, 12, 296), _log_int(rng, 12, 296)
            s = rng.choice([2.0, 2.0, 1.75])
            case = dict(kind=kind, width=w, height=h, out_width=int(w * s) - rng.randint(0, 1), out_height=int(h * s),
                        channels=rng.choice([32, 64, 128, 256]))
        if _cost(case) <= _cost(listed()[2]):
            return case


def _cost(case):
    w = work(case)
    rate = {"fp32": 25.0, "fp16": 25.0, "int8": 1.0}
    mode = case.get("mode", case.get("precision", "fp32" if case["kind"].endswith("f32") else "int8"))
    return w["flops"] * rate[mode] + 100.0 * w["bytes"]


# ---- models -------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _weights(encoder):
    """name -> float32 CUDA tensor, the same on every call."""
    specs = _package().dav2_format.tensor_specs(encoder)
    g = _generator(0xDA2 + len(encoder) + ord(encoder[-1]))
    state = {}
    for name, (shape, kind, scale) in sorted(specs.items()):
        n = torch.randn(shape, generator=g, device="cuda")
        if name.endswith("gamma"):
            state[name] = 0.05 + 0.15 * n.abs()
        elif "norm" in name and name.endswith("weight"):
            state[name] = 1.0 + 0.2 * n
        elif name.startswith("pretrained.") and name.endswith("bias"):
            state[name] = 0.05 * n
        elif kind == "uniform":
            state[name] = scale * (2.0 * torch.rand(shape, generator=g, device="cuda") - 1.0)
        else:
            state[name] = (scale if scale else 0.02) * n
    # a depth map that varies, most of it positive, as after training
    state["depth_head.scratch.output_conv2.2.weight"].mul_(8.0)
    state["depth_head.scratch.output_conv2.2.bias"].fill_(0.25)
    return state


_contexts: dict = {}


def _context(encoder, mode):
    """The program's one handle per encoder and precision mode (the weights are loaded once)."""
    if (encoder, mode) not in _contexts:
        pkg = _package()
        with tempfile.TemporaryDirectory(prefix="dav2_cases_") as tmp:
            path = Path(tmp) / f"{encoder}.dav2"
            state = {name: t.cpu().numpy() for name, t in _weights(encoder).items()}
            pkg.dav2_format.write_model(path, encoder, state)
            _contexts[encoder, mode] = pkg.Context(str(path), encoder, getattr(pkg, MODES[mode]))
    return _contexts[encoder, mode]


def _image(case, seed):
    """ImageNet-normalised pixels of smooth shapes with grain, [batch][3][H][W] on the GPU."""
    g = _generator(seed)
    b, h, w = case["batch"], case["height"], case["width"]
    coarse = torch.rand((b, 3, max(2, h // 28), max(2, w // 28)), generator=g, device="cuda")
    x = F.interpolate(coarse, size=(h, w), mode="bilinear", align_corners=False)
    x = (x + 0.05 * torch.randn((b, 3, h, w), generator=g, device="cuda")).clamp_(0, 1)
    mean = torch.tensor([0.485, 0.456, 0.406], device="cuda").view(1, 3, 1, 1)
    std = torch.tensor([0.229, 0.224, 0.225], device="cuda").view(1, 3, 1, 1)
    return ((x - mean) / std).contiguous()


# ---- layers --------------------------------------------------------------------

_ops_handle = None


def _ops():
    """The program's one operator instance."""
    global _ops_handle
    if _ops_handle is None:
        _ops_handle = _package().load().dav2_ops_create(0)
        if not _ops_handle:
            raise RuntimeError("dav2_ops_create failed")
    return _ops_handle


def _buffer(t):
    return _package().DeviceBuffer(t.data_ptr(), t.numel() * t.element_size())


def _int8_rows(w):
    """Per-row symmetric int8 weights and their scales, as a model holds them."""
    s = (w.abs().amax(dim=1) / 127.0).clamp_min(1e-8)
    return torch.round(w / s[:, None]).clamp_(-127, 127).to(torch.int8), s


def _layer_inputs(case, seed):
    g = _generator(seed)

    def normal(*shape, scale=1.0):
        return scale * torch.randn(shape, generator=g, device="cuda")

    kind = case["kind"]
    if kind.startswith("linear"):
        # LayerNorm rows (or GELU activations: mostly small, a heavy positive side) times trained-like weights
        x = normal(case["rows"], case["k"])
        if case["k"] > case["n"]:
            x = F.gelu(1.5 * x)
        return x, normal(case["n"], case["k"], scale=0.03), normal(case["n"], scale=0.05)
    if kind.startswith("attn"):
        return (normal(case.get("batch", 1) * case["tokens"], 3 * 64 * case["heads"], scale=1.2),)
    if kind.startswith("conv"):
        x = normal(case["channels"], case["height"], case["width"])
        inner = case["channels"] * case["kernel"] ** 2
        return x, normal(case["out_channels"], inner, scale=inner ** -0.5), normal(case["out_channels"], scale=0.05)
    return (normal(case["channels"], case["height"], case["width"]),)


def prepare(case, seed):
    pkg = _package()
    lib = pkg.load()
    kind = case["kind"]
    if kind == "model":
        ctx = _context(case["encoder"], case["mode"])
        x = _image(case, seed)
        b, h, w = case["batch"], case["height"], case["width"]
        if case["entry"] == "host":
            host = np.ascontiguousarray(x[0].cpu().numpy())
            return {"call": lambda: ctx.infer(host, w, h)}
        depth = torch.zeros((b, h, w), device="cuda")
        if case["entry"] == "device":
            def call():
                ctx.infer_device(x.data_ptr(), b, w, h, depth.data_ptr(), depth.numel())
                return depth
            return {"call": call}
        logits = torch.zeros((h, w), device="cuda")

        def call_logits():
            pkg.check(lib.dav2_infer_tensor_f32_device_logits(ctx.handle, x.data_ptr(), w, h, depth.data_ptr(),
                                                              logits.data_ptr(), None), lib)
            return {"depth": depth, "logits": logits}
        return {"call": call_logits}

    ops, inputs = _ops(), _layer_inputs(case, seed)
    x = inputs[0]
    if kind.startswith("linear"):
        _, w, bias = inputs
        rows, k, n = case["rows"], case["k"], case["n"]
        out = torch.zeros((rows, n), device="cuda")
        if kind == "linear_i8":
            q, s = _int8_rows(w)
            fn, keep = lib.dav2_ops_linear_int8, (x, q, s, bias)
            args = (ops, _buffer(out), _buffer(x), _buffer(q), _buffer(s), _buffer(bias), rows, k, n,
                    int(case["gelu"]), 0)
        else:
            fn, keep = lib.dav2_ops_linear, (x, w, bias)
            args = (ops, _buffer(out), _buffer(x), _buffer(w), _buffer(bias), rows, k, n, int(case["gelu"]))
    elif kind == "attn_i8":
        t, h, b = case["tokens"], case["heads"], case["batch"]
        out = torch.zeros((b * t, 64 * h), device="cuda")
        size = lib.dav2_hip_attention_fused_scratch_bytes(t, h, b)
        scratch = torch.empty(size, dtype=torch.uint8, device="cuda")
        fn, keep = lib.dav2_hip_attention_fused, (x, scratch)
        args = (out.data_ptr(), x.data_ptr(), t, h, b, scratch.data_ptr(), size, lib.dav2_ops_stream(ops))
    elif kind == "attn_ref":
        t, h = case["tokens"], case["heads"]
        half = int(case["precision"] == "fp16")
        out = torch.zeros((t, 64 * h), device="cuda")
        size = max(lib.dav2_hip_attention_ref_scratch_bytes(t, h, 1, half),
                   lib.dav2_hip_attention_ref16_fused_scratch_bytes(t, h, 1) if half else 0)
        scratch = torch.empty(size, dtype=torch.uint8, device="cuda")
        fn, keep = lib.dav2_ops_attention_head64, (x, scratch)
        args = (ops, _buffer(out), _buffer(x), t, h, _buffer(scratch), half)
    elif kind.startswith("conv"):
        _, w, bias = inputs
        size = (case["width"], case["height"], case["channels"], case["out_channels"], case["kernel"], 1,
                case["kernel"] // 2, 1)
        out = torch.zeros((case["out_channels"], case["height"], case["width"]), device="cuda")
        if kind == "conv_i8":
            q, s = _int8_rows(w)
            fn, keep = lib.dav2_ops_conv2d_int8, (x, q, s, bias)
            args = (ops, _buffer(out), _buffer(x), _buffer(q), _buffer(s), _buffer(bias), *size)
        else:
            fn, keep = lib.dav2_ops_conv2d, (x, w, bias)
            args = (ops, _buffer(out), _buffer(x), _buffer(w), _buffer(bias), *size)
    else:
        out = torch.zeros((case["channels"], case["out_height"], case["out_width"]), device="cuda")
        fn, keep = lib.dav2_ops_bilinear_align_true, (x,)
        args = (ops, _buffer(out), _buffer(x), case["width"], case["height"], case["out_width"], case["out_height"],
                case["channels"])

    def call_layer():
        status = fn(*args)
        if status:
            raise RuntimeError(f"{kind}: status {status}: {(lib.dav2_ops_last_error() or b'').decode()}")
        return out
    return {"call": call_layer, "keep": keep}


def run(state):
    return state["call"]()


# ---- what a pass cannot do without -----------------------------------------------


def _model_flops(case):
    a = _package().dav2_format.ARCH[case["encoder"]]
    d, f, oc = a["dim"], a["features"], a["out_channels"]
    pw, ph = case["width"] // 14, case["height"] // 14
    p, t = pw * ph, pw * ph + 1
    flops = 2.0 * p * d * 588 + a["depth"] * (24.0 * t * d * d + 4.0 * t * t * d)
    flops += sum(2.0 * p * d * c for c in oc) + 2.0 * p * 16 * oc[0] ** 2 + 2.0 * p * 4 * oc[1] ** 2
    quarter = ((pw + 1) // 2) * ((ph + 1) // 2)
    flops += 2.0 * quarter * 9 * oc[3] ** 2
    maps = (16 * p, 4 * p, p, quarter)
    flops += sum(2.0 * m * 9 * c * f for m, c in zip(maps, oc))
    units = (2, 2, 2, 1)  # residual units per level, two 3x3 convolutions each
    flops += sum(u * 2 * 2.0 * m * 9 * f * f for m, u in zip(maps, units))
    flops += sum(2.0 * m * f * f for m in (64 * p, 16 * p, 4 * p, p))
    flops += 2.0 * 64 * p * 9 * f * (f // 2) + 2.0 * 196 * p * (9 * (f // 2) * 32 + 32)
    return flops * case["batch"]


def work(case):
    kind = case["kind"]
    if kind == "model":
        specs = _package().dav2_format.tensor_specs(case["encoder"])
        parameters = sum(math.prod(shape) for shape, _, _ in specs.values())
        pixels = case["batch"] * case["width"] * case["height"]
        each = {"int8": 1, "fp16": 2, "fp32": 4}[case["mode"]]
        outputs = 2 if case["entry"] == "logits" else 1
        return {"bytes": float(parameters * each + pixels * 4 * (3 + outputs)), "flops": _model_flops(case)}
    if kind.startswith("linear"):
        m, k, n = case["rows"], case["k"], case["n"]
        return {"bytes": 4.0 * (m * k + m * n + 2 * n) + n * k * (1.0 if kind == "linear_i8" else 4.0),
                "flops": 2.0 * m * n * k}
    if kind.startswith("attn"):
        t, h, b = case["tokens"], case["heads"], case.get("batch", 1)
        return {"bytes": 4.0 * b * t * h * 64 * 4, "flops": 4.0 * b * h * t * t * 64}
    if kind.startswith("conv"):
        p, inner = case["width"] * case["height"], case["channels"] * case["kernel"] ** 2
        n = case["out_channels"]
        return {"bytes": 4.0 * p * (case["channels"] + n) + n * inner * (1.0 if kind == "conv_i8" else 4.0),
                "flops": 2.0 * p * n * inner}
    pixels = case["width"] * case["height"] + case["out_width"] * case["out_height"]
    return {"bytes": 4.0 * case["channels"] * pixels, "flops": 8.0 * case["channels"] * case["out_width"] *
            case["out_height"]}


def tolerance(case):
    kind = case["kind"]
    if kind in ("linear_f32", "conv_f32"):
        return {"rel": 2.6e-6}  # 32-bit sums of up to 4096 terms: 6.5e-7 from 64 bits
    if kind == "model" and case["mode"] == "fp32":
        return {"rel": 6e-6}  # 1.5e-6 from 64 bits
    if kind == "model" and case["mode"] == "fp16":
        return {"rel": 2e-3}  # binary16 operands (4.8e-4 from 64 bits): a rounding that flips travels through the blocks
    return "exact"  # int8 sums and the reference-order attention: the same bits for the same input


# ---- the same in 64 bits -----------------------------------------------------------


def _conv64(x, w, bias, kernel, stride=1):
    """Convolution of a CHW map in float64, a few rows at a time."""
    c, h, wd = x.shape
    pad = kernel // 2
    oh, ow = (h + 2 * pad - kernel) // stride + 1, (wd + 2 * pad - kernel) // stride + 1
    xp = F.pad(x, (pad, pad, pad, pad))
    out = torch.empty((w.shape[0], oh, ow), dtype=torch.float64, device=x.device)
    step = max(1, int(2 ** 27 // (c * kernel * kernel * ow)))
    for y in range(0, oh, step):
        n = min(step, oh - y)
        cols = F.unfold(xp[None, :, y * stride:(y + n - 1) * stride + kernel], kernel, stride=stride)[0]
        out[:, y:y + n] = (w @ cols).view(-1, n, ow)
    return out if bias is None else out + bias[:, None, None]


def _attention64(qkv, heads):
    """softmax(q k^T / 8) v of one image, [T][3*H*64] -> [T][H*64], float64."""
    t = qkv.shape[0]
    q, k, v = qkv.view(t, 3, heads, 64).permute(1, 2, 0, 3)
    out = [torch.softmax((q[h] * 0.125) @ k[h].T.contiguous(), dim=-1) @ v[h].contiguous() for h in range(heads)]
    return torch.stack(out, dim=1).reshape(t, heads * 64)


def _position64(pos, pw, ph):
    grid = pos[0, 1:]
    if (pw, ph) == (37, 37):
        return torch.cat([pos[0, :1], grid])
    grid = grid.view(1, 37, 37, -1).permute(0, 3, 1, 2)
    grid = F.interpolate(grid, scale_factor=((ph + 0.1) / 37, (pw + 0.1) / 37), mode="bicubic", align_corners=False)
    return torch.cat([pos[0, :1], grid[0].flatten(1).T])


def _model64(case, image):
    """Logits of one image in float64, no quantization."""
    a = _package().dav2_format.ARCH[case["encoder"]]
    w = {k: v.double() for k, v in _weights(case["encoder"]).items()}
    d, heads = a["dim"], a["heads"]
    pw, ph = case["width"] // 14, case["height"] // 14
    patches = F.unfold(image[None], 14, stride=14)[0].T
    p = "pretrained."
    x = patches @ w[p + "patch_embed.proj.weight"].view(d, -1).T + w[p + "patch_embed.proj.bias"]
    x = torch.cat([w[p + "cls_token"][0], x]) + _position64(w[p + "pos_embed"], pw, ph)

    def norm(v, name):
        return F.layer_norm(v, (d,), w[name + ".weight"], w[name + ".bias"], 1e-6)

    features = []
    for i in range(a["depth"]):
        b = f"{p}blocks.{i}."

        def linear(v, name):
            return v @ w[b + name + ".weight"].T + w[b + name + ".bias"]

        attended = _attention64(linear(norm(x, b + "norm1"), "attn.qkv"), heads)
        x = x + w[b + "ls1.gamma"] * linear(attended, "attn.proj")
        x = x + w[b + "ls2.gamma"] * linear(F.gelu(linear(norm(x, b + "norm2"), "mlp.fc1")), "mlp.fc2")
        if i in CAPTURE[case["encoder"]]:
            features.append(norm(x, p + "norm")[1:])

    h = "depth_head."

    def conv(v, name, kernel=3, stride=1, bias=True):
        k = w[h + name + ".weight"]
        return _conv64(v, k.view(k.shape[0], -1), w[h + name + ".bias"] if bias else None, kernel, stride)

    def grow(v, name, k):
        kernel = w[h + name + ".weight"]  # [in][out][k][k]
        y = torch.einsum("cp,cm->mp", v.flatten(1), kernel.flatten(1)).view(-1, k, k, ph, pw)
        return y.permute(0, 3, 1, 4, 2).reshape(-1, ph * k, pw * k) + w[h + name + ".bias"][:, None, None]

    def resize(v, oh, ow):
        return F.interpolate(v[None], size=(oh, ow), mode="bilinear", align_corners=True)[0]

    def unit(v, name):
        return v + conv(conv(v.relu(), name + ".conv1").relu(), name + ".conv2")

    levels = []
    for i, feature in enumerate(features):
        v = conv(feature.T.reshape(d, ph, pw).contiguous(), f"projects.{i}", kernel=1)
        if i == 0:
            v = grow(v, "resize_layers.0", 4)
        elif i == 1:
            v = grow(v, "resize_layers.1", 2)
        elif i == 3:
            v = conv(v, "resize_layers.3", stride=2)
        levels.append(conv(v, f"scratch.layer{i + 1}_rn", bias=False))
    path = levels[3]
    for i in (3, 2, 1, 0):
        r = f"scratch.refinenet{i + 1}"
        if i < 3:
            path = path + unit(levels[i], r + ".resConfUnit1")
        path = unit(path, r + ".resConfUnit2")
        oh, ow = levels[i - 1].shape[1:] if i else (levels[0].shape[1] * 2, levels[0].shape[2] * 2)
        path = conv(resize(path, oh, ow), r + ".out_conv", kernel=1)
    path = resize(conv(path, "scratch.output_conv1"), ph * 14, pw * 14)
    return conv(conv(path, "scratch.output_conv2.0").relu(), "scratch.output_conv2.2", kernel=1)[0]


def exact(case, seed):
    kind = case["kind"]
    if kind == "model":
        image = _image(case, seed).double()
        logits = [_model64(case, image[b]) for b in range(case["batch"])]
        if case["entry"] == "host":
            return logits[0].relu().cpu().numpy()
        depth = torch.stack(logits).relu()
        return depth if case["entry"] == "device" else {"depth": depth, "logits": logits[0]}
    inputs = _layer_inputs(case, seed)
    x = inputs[0]
    if kind.startswith("linear"):
        _, w, bias = inputs
        if kind == "linear_i8":
            q, s = _int8_rows(w)
            xq, xs = _int8_rows(x)
            y = (xq.double() @ q.double().T) * xs.double()[:, None] * s.double() + bias.double()
        else:
            y = x.double() @ w.double().T + bias.double()
        return F.gelu(y) if case["gelu"] else y
    if kind.startswith("attn"):
        return torch.cat([_attention64(part, case["heads"]) for part in x.double().split(case["tokens"])])
    if kind.startswith("conv"):
        _, w, bias = inputs
        if kind == "conv_f32":
            return _conv64(x.double(), w.double(), bias.double(), case["kernel"])
        q, s = _int8_rows(w)
        # the scale of an output pixel is that of its whole im2col row
        window = F.max_pool2d(x.abs().amax(dim=0)[None, None], case["kernel"], stride=1, padding=case["kernel"] // 2)[0]
        scale = (window[0] / 127.0).clamp_min(1e-8)
        out = torch.empty((case["out_channels"], case["height"], case["width"]), dtype=torch.float64, device="cuda")
        pad = case["kernel"] // 2
        xp = F.pad(x, (pad, pad, pad, pad))
        step = max(1, int(2 ** 27 // (w.shape[1] * case["width"])))
        for y in range(0, case["height"], step):
            n = min(step, case["height"] - y)
            cols = F.unfold(xp[None, :, y:y + n - 1 + case["kernel"]], case["kernel"])[0]
            rows = scale[y:y + n].reshape(1, -1)
            acc = q.double() @ torch.round(cols * (1.0 / rows)).clamp_(-127, 127).double()
            out[:, y:y + n] = (acc * rows.double() * s.double()[:, None] + bias.double()[:, None]).view(-1, n,
                                                                                                       case["width"])
        return out
    return F.interpolate(x.double()[None], size=(case["out_height"], case["out_width"]), mode="bilinear",
                         align_corners=True)[0]
