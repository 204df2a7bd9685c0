"""The workloads this repository's speed is measured on, through the public entry points.

Each case is one pass of the work a training program hands to the framework: compressing an
activation and restoring it, a converted layer forward and backward, a training step of a small
converted model.  The convolutions around them are the GPU library's own kernels and are left out;
what the framework adds to a convolution - the compression of its input, before and after - is
`compress`.  Kinds:

  cycle     minimax -> pack_mixed_precision -> unpack_mixed_precision of cpp_extension, given widths
  compress  ops.quantize_activation -> ops.dequantize_activation, as conv and linear layers call it:
            with a scheme (per-sample widths, level L3) or at one width (levels L1 / L2)
  mask      QReLU or QDropout, forward and backward
  pool      QMaxPool2d, forward and backward
  norm      QBatchNorm2d at L3, forward and backward: alone, with the ReLU after it, or as the closing
            relu(bn(x) + identity) of a residual block
  linear    QLinear forward and backward
  mlp       training step (loss and gradients) of a small QModule

Random numbers (inputs, stochastic rounding, dropout) follow from the seed given to `prepare`.
"""
import math

import torch
import torch.nn as nn
import torch.nn.functional as F

from actnn_amd import layers, ops
from actnn_amd.conf import config
from actnn_amd.cpp_extension import minimax as ext_minimax
from actnn_amd.cpp_extension import quantization as ext_quantization
from actnn_amd.module import QModule
from actnn_amd.qbnscheme import QBNScheme
from actnn_amd.qscheme import QScheme, greedy_bits

DEVICE = "cuda"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2}
GROUP = 256


def listed():
    return [
        # ResNet-50's first stage, fp32, the batch of the repository's benchmark: the largest tensor
        dict(name="cycle_f32_stage1", kind="cycle", dtype="f32", n=256, c=256, h=56, w=56),
        # a convolution's input at a small batch (the shape of the repository's CPU baseline), bf16 in the
        # layout a training run on this GPU uses: kernels of a few microseconds
        dict(name="compress_bf16_small", kind="compress", dtype="bf16", n=32, c=64, h=56, w=56, level="L3", bits=2,
             channels_last=True),
        # image crops of an odd size, the input of a network's first convolution: rows that are no whole
        # number of quantisation groups
        dict(name="compress_f32_images", kind="compress", dtype="f32", n=32, c=3, h=321, w=321, level="L3", bits=2,
             channels_last=False),
        # level L2: every activation at 4 bits
        dict(name="compress_bf16_4bit", kind="compress", dtype="bf16", n=256, c=256, h=28, w=28, level="L2", bits=4,
             channels_last=False),
        # ReLU on the shape of the reference's ReLU benchmark, in its dtype
        dict(name="relu_f32", kind="mask", op="relu", p=0.0, dtype="f32", n=256, f=56 * 56 * 32),
        # dropout in front of a classifier: a call of a few microseconds
        dict(name="dropout_bf16_small", kind="mask", op="dropout", p=0.5, dtype="bf16", n=128, f=4096),
        # the stem's max-pool of ResNet-50
        dict(name="pool_f16_stem", kind="pool", dtype="f16", n=256, c=64, h=112, w=112, k=3, s=2, p=1,
             channels_last=False),
        # a pool over odd planes without padding
        dict(name="pool_f32_odd", kind="pool", dtype="f32", n=64, c=96, h=55, w=55, k=3, s=2, p=0,
             channels_last=False),
        # the closing step of ResNet-50's second-stage blocks in mixed precision
        dict(name="norm_bf16_block_end", kind="norm", dtype="bf16", n=256, c=512, h=28, w=28, tail="add_relu",
             channels_last=True),
        # batch norm of fp32 planes whose rows are no whole number of groups
        dict(name="norm_f32_odd", kind="norm", dtype="f32", n=64, c=96, h=27, w=27, tail="none",
             channels_last=False),
        # the repository's fully connected benchmark, at its default level
        dict(name="linear_f16_L3", kind="linear", dtype="f16", rows=8192, fin=4096, fout=4096, level="L3", bits=2),
        # a small model at a small batch: bound by the host
        dict(name="mlp_step_small", kind="mlp", rows=64, fin=512, hidden=1024, classes=100, depth=2, level="L3", bits=2),
    ]


# ------------------------------------------------------------------------------------------
# drawn cases: the same kinds over their ranges
# ------------------------------------------------------------------------------------------
MOST_ELEMENTS = {"f32": 200_000_000, "f16": 200_000_000, "bf16": 200_000_000}


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _image_shape(rng, dtype, most):
    """[N, C, H, W] with `most` elements at most: planes of 4 to 224 pixels a side, odd ones among them."""
    h = _log_int(rng, 4, 224)
    w = h if rng.random() < 0.6 else max(4, min(300, int(h * rng.uniform(0.6, 1.8))))
    c = rng.choice([3, 16, 24, 32, 48, 64, 96, 128, 160, 192, 256, 320, 512, 1024])
    n = _log_int(rng, 2, 512)
    while n * c * h * w > most and n > 1:
        n = max(1, n // 2)
    while n * c * h * w > most:
        c = max(3, c // 2)
    return n, c, h, w


def draw(rng):
    kind = rng.choice(["cycle", "compress", "compress", "mask", "pool", "norm", "norm", "linear", "mlp"])
    dtype = rng.choice(["f32", "f16", "bf16", "bf16"])
    case = dict(kind=kind, dtype=dtype)
    most = MOST_ELEMENTS[dtype]
    if kind == "cycle":
        case.update(zip("nchw", _image_shape(rng, dtype, most)))
        case["c"] = max(16, case["c"] // 16 * 16)
        case["h"], case["w"] = case["h"] // 4 * 4, case["w"] // 4 * 4          # whole groups of 256
        while case["n"] * case["c"] * case["h"] * case["w"] > most:
            case["n"] = max(1, case["n"] // 2)
    elif kind == "compress":
        case.update(zip("nchw", _image_shape(rng, dtype, most // 2)))
        case["level"] = rng.choice(["L3", "L3", "L2"])
        case["bits"] = 2 if case["level"] == "L3" else rng.choice([4, 4, 2, 8])
        case["channels_last"] = rng.random() < 0.5
    elif kind == "mask":
        case["op"] = rng.choice(["relu", "dropout"])
        case["p"] = rng.choice([0.1, 0.25, 0.5]) if case["op"] == "dropout" else 0.0
        case["n"] = _log_int(rng, 8, 512)
        case["f"] = max(1, min(_log_int(rng, 128, 1_000_000), most // case["n"]))
    elif kind == "pool":
        case.update(zip("nchw", _image_shape(rng, dtype, most)))
        case["k"], case["s"], case["p"] = rng.choice([(3, 2, 1), (3, 2, 0), (2, 2, 0), (3, 1, 1), (3, 2, 1)])
        case["channels_last"] = rng.random() < 0.4
    elif kind == "norm":
        case.update(zip("nchw", _image_shape(rng, dtype, most // 2)))
        case["c"] = max(16, case["c"])
        case["n"] = max(2, case["n"])
        while case["n"] * case["c"] * case["h"] * case["w"] > most // 2 and case["n"] > 2:
            case["n"] = max(2, case["n"] // 2)
        case["channels_last"] = rng.random() < 0.6
        case["tail"] = rng.choice(["none", "relu", "add_relu"])
    elif kind == "linear":
        case["dtype"] = dtype = rng.choice(["f16", "bf16"])
        case["rows"] = _log_int(rng, 32, 8192)
        case["fin"] = rng.choice([256, 512, 768, 1000, 1024, 2048, 3072, 4096])
        case["fout"] = rng.choice([10, 100, 256, 512, 768, 1000, 1024, 2048, 3072, 4096])
        case["level"] = rng.choice(["L3", "L3", "L2"])
        case["bits"] = 2 if case["level"] == "L3" else rng.choice([2, 4])
    else:
        del case["dtype"]
        case.update(rows=_log_int(rng, 16, 1024), fin=rng.choice([256, 300, 512, 784]), hidden=rng.choice([256, 512, 1024, 2048]),
                    classes=rng.choice([10, 100, 1000]), depth=rng.choice([1, 2, 3]),
                    level=rng.choice(["L3", "L3", "L2"]))
        case["bits"] = 2 if case["level"] == "L3" else 4
    return case


# ------------------------------------------------------------------------------------------
# configuration: process-wide in a user's program, so it changes only when the level does
# ------------------------------------------------------------------------------------------
_profile = None


def _use(profile):
    """Levels L3 (the defaults: adaptive, 2 bits on average) and L2 (one width for everything)."""
    global _profile
    if profile == _profile:
        return
    level, bits = profile
    config.reset()
    if level == "L3":
        config.activation_compression_bits = [bits, 8, 8]
    else:
        config.activation_compression_bits = [bits]
        config.adaptive_conv_scheme = config.adaptive_bn_scheme = False
    config.training = True
    _profile = profile


def _new_model(profile):
    """A program builds one model: the schemes of the one before are forgotten."""
    _use(profile)
    QScheme.reset()
    QBNScheme.reset()


# ------------------------------------------------------------------------------------------
# prepare
# ------------------------------------------------------------------------------------------
def _activation(gen, shape, dtype, relu=True, channels_last=False):
    """What a convolution sees: N(0, 1) with a scale of its own for every channel and, milder, every
    sample, after a ReLU."""
    x = torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float32)
    channel = torch.exp(0.5 * torch.randn(shape[1], generator=gen, device=DEVICE))
    sample = torch.exp(0.25 * torch.randn(shape[0], generator=gen, device=DEVICE))
    x *= channel.view(1, -1, *[1] * (len(shape) - 2))
    x *= sample.view(-1, *[1] * (len(shape) - 1))
    if relu:
        x.relu_()
    x = x.to(dtype)
    return x.contiguous(memory_format=torch.channels_last) if channels_last else x


def _like(gen, x):
    """A gradient laid out like `x`."""
    g = torch.empty_like(x)
    return g.normal_(generator=gen)


def _level(case):
    return case.get("level", "L3"), case.get("bits", 2)


def prepare(case, seed):
    kind, profile = case["kind"], _level(case)
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    torch.manual_seed(seed)                                   # stochastic rounding, dropout, parameters
    state = dict(kind=kind, profile=profile)
    if kind == "cycle":
        _use(profile)
        n, features = case["n"], case["c"] * case["h"] * case["w"]
        x = _activation(gen, (n, case["c"], case["h"], case["w"]), DTYPES[case["dtype"]])
        state["x"] = x.view(n, features // GROUP, GROUP)
        lo, hi = state["x"].amin(2), state["x"].amax(2)
        sensitivity = (hi.float() - lo.float()).square_().sum(1).cpu()
        state["bits"], _ = greedy_bits(sensitivity, n, 8, 2, x.device)
    elif kind == "compress":
        _new_model(profile)
        shape = (case["n"], case["c"], case["h"], case["w"])
        state["x"] = _activation(gen, shape, DTYPES[case["dtype"]], channels_last=case["channels_last"] and case["c"] > 1)
        state["scheme"] = None
        if case["level"] == "L3":
            state["scheme"] = QScheme(nn.Module(), num_locations=9)
            state["scheme"].set_scale(torch.randn(case["n"], 1024, generator=gen, device=DEVICE))
    elif kind == "mask":
        _use(profile)
        x = torch.randn((case["n"], case["f"]), generator=gen, device=DEVICE, dtype=DTYPES[case["dtype"]])
        state["grad"] = _like(gen, x)
        state["x"] = x.requires_grad_()
        state["layer"] = layers.QReLU() if case["op"] == "relu" else layers.QDropout(case["p"])
    elif kind == "pool":
        _use(profile)
        shape = (case["n"], case["c"], case["h"], case["w"])
        x = _activation(gen, shape, DTYPES[case["dtype"]], channels_last=case["channels_last"])
        out = [(d + 2 * case["p"] - case["k"]) // case["s"] + 1 for d in shape[2:]]
        grad = torch.empty((case["n"], case["c"], *out), dtype=x.dtype, device=DEVICE,
                           memory_format=torch.channels_last if case["channels_last"] else torch.contiguous_format)
        state["grad"] = grad.normal_(generator=gen)
        state["x"] = x.requires_grad_()
        state["layer"] = layers.QMaxPool2d(case["k"], case["s"], case["p"])
    elif kind == "norm":
        _new_model(profile)
        shape = (case["n"], case["c"], case["h"], case["w"])
        x = _activation(gen, shape, DTYPES[case["dtype"]], relu=False, channels_last=case["channels_last"])
        state["grad"] = _like(gen, x)
        state["tail"] = case["tail"]
        state["residual"] = None
        state["relu"] = layers.QReLU() if case["tail"] == "relu" else layers.QAddReLU()
        if case["tail"] == "add_relu":
            state["residual"] = _activation(gen, shape, x.dtype, channels_last=case["channels_last"]).requires_grad_()
        state["x"] = x.requires_grad_()
        layer = layers.QBatchNorm2d(case["c"]).to(DEVICE)
        with torch.no_grad():
            layer.weight.uniform_(0.5, 1.5, generator=gen)
            layer.bias.normal_(generator=gen)
        state["layer"] = layer.train()
    elif kind == "linear":
        _new_model(profile)
        dtype = DTYPES[case["dtype"]]
        # heavy-tailed features, as in front of a fully connected layer
        x = torch.randn((case["rows"], case["fin"]), generator=gen, device=DEVICE)
        x *= torch.exp(torch.randn(case["fin"], generator=gen, device=DEVICE))
        state["x"] = x.to(dtype).requires_grad_()
        state["grad"] = torch.randn((case["rows"], case["fout"]), generator=gen, device=DEVICE).to(dtype)
        state["layer"] = layers.QLinear(case["fin"], case["fout"]).to(DEVICE, dtype)
        if state["layer"].scheme is not None:
            state["layer"].scheme.set_scale(state["grad"])
            state["schemes"] = QScheme.layers
    else:
        _new_model(profile)
        width, parts = case["fin"], []
        for _ in range(case["depth"]):
            parts += [nn.Linear(width, case["hidden"]), nn.BatchNorm1d(case["hidden"]), nn.ReLU(), nn.Dropout(0.1)]
            width = case["hidden"]
        model = QModule(nn.Sequential(*parts, nn.Linear(width, case["classes"]))).to(DEVICE)
        state["model"] = model.train()
        state["params"] = list(model.parameters())
        state["x"] = torch.randn((case["rows"], case["fin"]), generator=gen, device=DEVICE)
        state["target"] = torch.randint(case["classes"], (case["rows"],), generator=gen, device=DEVICE)
        state["schemes"], state["bn_schemes"] = QScheme.layers, QBNScheme.layers
    return state


# ------------------------------------------------------------------------------------------
# run: one pass
# ------------------------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    _use(state["profile"])
    if "schemes" in state:                                    # this state's model is the program's model
        QScheme.layers = state["schemes"]
        QBNScheme.layers = state.get("bn_schemes", [])
    return _RUN[kind](state)


def _run_cycle(state):
    x, bits = state["x"], state["bits"]
    n, groups, size = x.shape
    mn, mx = ext_minimax.minimax(x.view(-1, size))
    mn, mx = mn.view(n, groups, 1), mx.view(n, groups, 1)
    packed, scale = ext_quantization.pack_mixed_precision(x, mn, mx, bits, True)
    return mn, mx, packed, scale, ext_quantization.unpack_mixed_precision(packed, bits, scale, mn, n, groups, size)


def _run_compress(state):
    x = state["x"]
    saved = ops.quantize_saved(x, state["scheme"])
    return tuple(saved) + (ops.dequantize_activation(saved, x.shape),)


def _run_layer(state):
    y = state["layer"](state["x"])
    return y, torch.autograd.grad(y, state["x"], state["grad"])[0]


def _run_norm(state):
    layer, x, residual = state["layer"], state["x"], state["residual"]
    wanted = [x, layer.weight, layer.bias]
    if state["tail"] == "none":
        y = layer(x)
    elif state["tail"] == "relu":
        y = layers.bn_relu(layer, state["relu"], x)
    else:
        y = layers.bn_add_relu(layer, state["relu"], x, residual)
        wanted.append(residual)
    grads = torch.autograd.grad(y, wanted, state["grad"])
    return (y, layer.running_mean, layer.running_var) + tuple(grads)


def _run_linear(state):
    layer, x = state["layer"], state["x"]
    y = layer(x)
    return (y,) + torch.autograd.grad(y, [x, layer.weight, layer.bias], state["grad"])


def _run_mlp(state):
    with torch.autocast("cuda", dtype=torch.bfloat16):
        logits = state["model"](state["x"])
        loss = F.cross_entropy(logits, state["target"])
    return (logits, loss) + torch.autograd.grad(loss, state["params"])


_RUN = {"cycle": _run_cycle, "compress": _run_compress, "mask": _run_layer, "pool": _run_layer, "norm": _run_norm,
        "linear": _run_linear, "mlp": _run_mlp}


# ------------------------------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    size = BYTES.get(case.get("dtype"), 2)
    if kind in ("cycle", "compress"):
        n = case["n"]
        features = case["c"] * case["h"] * case["w"]
        groups = n * -(-features // GROUP)
        stream = groups * GROUP * case.get("bits", 2) / 8
        # input read, stream and (scale, minimum) written and read back, tensor written
        total = 2 * n * features * size + 2 * stream + 4 * groups * size
        if kind == "cycle":
            total += groups * size                            # the maxima are handed out as well
        return {"bytes": total, "flops": 0}
    if kind == "mask":
        n = case["n"] * case["f"]
        return {"bytes": 4 * n * size + 2 * n / 8, "flops": 0}
    if kind == "pool":
        n = case["n"] * case["c"] * case["h"] * case["w"]
        out = case["n"] * case["c"]
        for d in (case["h"], case["w"]):
            out *= (d + 2 * case["p"] - case["k"]) // case["s"] + 1
        return {"bytes": 2 * n * size + 2 * out * size + 2 * out / 2, "flops": 0}
    if kind == "norm":
        n = case["n"] * case["c"] * case["h"] * case["w"]
        stream = n * 2 / 8 + 2 * n / GROUP * size
        total = 2 * n * size + stream                         # input, output, packed copy
        total += 2 * n * size + stream                        # gradient in and out, packed copy back
        if case["tail"] != "none":
            total += 2 * n / 8
        if case["tail"] == "add_relu":
            total += 2 * n * size                             # the identity and its gradient
        return {"bytes": total, "flops": 0}
    if kind == "linear":
        m, i, o = case["rows"], case["fin"], case["fout"]
        stream = m * i * case["bits"] / 8 + 2 * m * -(-i // GROUP) * size
        return {"bytes": size * (2 * m * i + 2 * m * o + 2 * i * o) + 2 * stream, "flops": 6 * m * i * o}
    m, widths = case["rows"], [case["fin"]] + [case["hidden"]] * case["depth"] + [case["classes"]]
    pairs = list(zip(widths, widths[1:]))
    weights = sum(a * b for a, b in pairs)
    acts = sum(a + b for a, b in pairs) * m
    return {"bytes": 8 * weights + 2 * 2 * acts, "flops": 6 * m * weights}


def tolerance(case):
    """Streams, widths, masks, dequantised values and maxima are defined bit for bit.  Sums (batch
    norm, the gradients of overlapping windows, matrix products) are kept in 32 bits and rounded to
    the tensor's type: against the same path in 64 bits the results are off by 1.3e-7 (f32), 2.1e-4 (f16)
    and 1.7e-3 (bf16); with |mean| a few times the deviation the sums of fp32 batch norm reach 3e-6."""
    kind = case["kind"]
    if kind in ("cycle", "compress", "mask"):
        return "exact"
    if kind == "mlp":
        return {"rel": 1e-2, "max": 0.5}
    rel = {"f32": 1e-5, "f16": 1e-3, "bf16": 7e-3}[case["dtype"]]
    if kind == "norm":
        return {"rel": rel, "max": 0.5 if case["tail"] != "none" else 40 * rel}
    return {"rel": rel, "max": 40 * rel}
