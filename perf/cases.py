"""The work that users of this package have it do, as cases that can be timed and compared.

Families (`case["op"]`), all through the public entry points:

  conv      u8 x s8 -> i32 convolution on blocked layouts, weights in the reference's layout or prepared once
  fused     the signed convolution of quantized graphs, with bias and scale
  conv3d    the 3-D signed convolution
  chain     a whole network's convolutions back to back, u8 activations requantised between the layers
  relay     the NCHW -> NCHW graph (conv2d(x, w) + b) * 11 of an operator-by-operator runtime
  conv_f16  fp16 -> fp32 convolution: blocked operands, prepared weights, or plain NCHW / OIHW operands
  gemm      fp16 GEMM, fp32 or fp16 output, b as given, prepared once, or with a workspace
  dense     u8 x s8 -> i32 dense, weights row-major, packed by the reference's rule, or prepared once

listed() names twelve of them, from one image to a training-sized batch; draw(rng) takes further ones from the
same families, sizes spread over their logarithm, most of them ragged.
"""
import math

import torch

import unit_amd as U
from unit_amd.chain import ConvChain, resnet18_layers, resnet50_layers
from unit_amd.relay import Conv2dBiasMultiply

MIN_FLOPS = 1e8      # a launch-sized problem
CONV_MACS = 12e9     # largest drawn convolution; the network chains and the square GEMMs are larger
MAX_BYTES = 250e6    # largest drawn operand + result volume
GEMM_MACS = 4096 ** 3


def listed():
    return [
        # one image, one 3 x 3 layer of a residual network on weights prepared at load time: the smallest call
        dict(name="conv_one_image", op="conv", n=1, c=64, h=56, w=56, k=64, ks=3, stride=1, pad=1, weights="prepared"),
        # the operator as a drop-in: the reference's weight layout, an odd batch, odd image and channel counts
        dict(name="conv_ragged", op="conv", n=7, c=112, h=35, w=27, k=208, ks=3, stride=1, pad=1, weights="blocked"),
        # the widest layer of a 50-layer network at batch 32: result traffic
        dict(name="fused_wide_b32", op="fused", n=32, c=64, h=56, w=56, k=256, ks=1, stride=1, pad=0, weights="prepared"),
        # a video / volume layer, sixteen frames
        dict(name="conv3d_16_frames", op="conv3d", n=1, c=64, d=16, h=56, w=56, k=128, ks=3, stride=1),
        # a 50-layer network at serving batch
        dict(name="network_b32", op="chain", net="resnet50", n=32),
        # the first layer of an image network, three input channels, planar in and out
        dict(name="stem_graph_b16", op="relay", n=16, c=3, h=224, w=224, k=64, ks=7, stride=2, pad=3),
        # half precision at batch 32 on prepared weights, data padded by the caller
        dict(name="conv_f16_b32", op="conv_f16", n=32, c=256, h=16, w=16, k=256, ks=3, stride=1, operands="prepared"),
        # the half-precision operator called on plain NCHW / OIHW operands, one image
        dict(name="conv_f16_nchw", op="conv_f16", n=1, c=256, h=30, w=30, k=256, ks=3, stride=2, operands="nchw"),
        # a large square product
        dict(name="gemm_4096", op="gemm", m=4096, n=4096, k=4096, out="float32", b="plain"),
        # a mid-size product with nothing aligned to a tile, half-precision result
        dict(name="gemm_ragged", op="gemm", m=1000, n=1516, k=1096, out="float16", b="plain"),
        # the reference's own dense layer on its packed weight: few rows, a launch-sized problem
        dict(name="dense_128_rows", op="dense", m=128, n=768, k=3072, weights="packed"),
        # a large int8 product on a weight prepared at load time
        dict(name="dense_4096", op="dense", m=4096, n=4096, k=4096, weights="prepared"),
    ]


# ------------------------------------------------------------------------------------- drawn cases
def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _multiple(rng, lo, hi, step):
    return step * _log_int(rng, lo // step, hi // step)


def _image(rng, lo, hi):
    h = _log_int(rng, lo, hi)
    return h, max(lo, min(hi, int(h * rng.uniform(0.6, 1.6))))


def _conv_sizes(rng, max_batch=64):
    h, w = _image(rng, 7, 112)
    return dict(n=_log_int(rng, 1, max_batch), c=_multiple(rng, 16, 2048, 16), h=h, w=w, k=_multiple(rng, 16, 2048, 16),
                ks=rng.choice([1, 1, 1, 3, 3, 3, 5]), stride=rng.choice([1, 1, 1, 2]))


def _draw_one(rng):
    op = rng.choice(["conv", "conv", "fused", "conv3d", "chain", "relay", "conv_f16", "conv_f16", "gemm", "gemm", "dense",
                     "dense"])
    if op in ("conv", "fused"):
        case = dict(op=op, weights=rng.choice(["prepared", "blocked"]), **_conv_sizes(rng))
        case["pad"] = rng.choice([0, case["ks"] // 2])
    elif op == "conv3d":
        h, w = _image(rng, 7, 112)
        case = dict(op=op, n=1, c=_multiple(rng, 16, 512, 16), d=_log_int(rng, 3, 16), h=h, w=w, k=_multiple(rng, 16, 512, 16), ks=rng.choice([1, 3, 3]), stride=rng.choice([1, 1, 2]))
    elif op == "chain":
        case = dict(op=op, net=rng.choice(["resnet18", "resnet50"]), n=_log_int(rng, 1, 32))
    elif op == "relay":
        case = dict(op=op, **_conv_sizes(rng, 32))
        if rng.random() < 0.4:  # image stems
            case.update(c=3, h=rng.randint(64, 256), w=rng.randint(64, 256), k=rng.choice([32, 64, 96]), ks=rng.choice([3, 7]), stride=2)
        elif rng.random() < 0.5:
            case["k"] = max(1, case["k"] - rng.randint(0, 15))  # any number of output channels
        case["pad"] = rng.choice([0, case["ks"] // 2])
    elif op == "conv_f16":
        case = dict(op=op, operands=rng.choice(["prepared", "prepared", "blocked", "nchw"]), **_conv_sizes(rng, 32))
    elif op == "gemm":
        ragged = rng.random() < 0.6
        case = dict(op=op, m=_log_int(rng, 1, 8192), n=_multiple(rng, 64, 8192, 4 if ragged else 64),
                    k=_multiple(rng, 64, 8192, 8 if ragged else 64), out=rng.choice(["float32", "float16"]),
                    b=rng.choice(["plain", "plain", "prepared", "workspace"]))
    else:
        weights = rng.choice(["row_major", "packed", "prepared"])
        case = dict(op=op, m=_log_int(rng, 1, 8192), n=_multiple(rng, 128, 8192, 128 if weights == "packed" else 4),
                    k=_multiple(rng, 64, 8192, 16), weights=weights)
    return case


def draw(rng):
    while True:
        case = _draw_one(rng)
        if case["op"] == "chain":
            return case
        w = work(case)
        limit = 2 * (GEMM_MACS if case["op"] in ("gemm", "dense") else CONV_MACS)
        if MIN_FLOPS <= w["flops"] <= limit and w["bytes"] <= MAX_BYTES:
            return case


# ------------------------------------------------------------------------------------- inputs and state
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _u8(shape, g):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g)


def _s8(shape, g):
    return torch.randint(-128, 128, shape, dtype=torch.int8, device="cuda", generator=g)


def _f16(shape, g, scale=1.0):
    return (torch.randn(shape, device="cuda", generator=g) * scale).half()


def _bias(k, g):
    return torch.randint(-100000, 100000, (k,), dtype=torch.int32, device="cuda", generator=g)


def _chain_layers(case, g):
    """The network's layers with a scale per layer that spreads the requantised activations over 0..255."""
    make = resnet50_layers if case["net"] == "resnet50" else resnet18_layers
    layers = make(lambda oc, ic, k: _s8((oc, ic, k, k), g), lambda oc: _bias(oc, g) // 10)
    out = []
    for i, ly in enumerate(layers):
        _, ic, kh, kw = ly.weight.shape
        sigma = 74.0 * (147.0 if i == 0 else 70.0) * math.sqrt(ic * kh * kw)  # rms(weight) * rms(activation) * sqrt(terms)
        out.append(ly._replace(scale=int(100.0 / sigma * 2 ** 24), shift=24))
    return out


def prepare(case, seed):
    g, op = _gen(seed), case["op"]
    if op in ("conv", "fused"):
        n, c, k, ks = case["n"], case["c"], case["k"], case["ks"]
        weight = _s8((k // 16, c // 16, ks, ks, 4, 16, 4), g)
        if case["weights"] == "prepared":
            weight = U.prepare_conv2d_weight(weight)
        shape = (n, c // 16, case["h"], case["w"], 16)
        return dict(case=case, x=_u8(shape, g) if op == "conv" else _s8(shape, g), w=weight, b=_bias(k, g))
    if op == "conv3d":
        c, k, ks = case["c"], case["k"], case["ks"]
        return dict(case=case, x=_s8((case["n"], c // 16, case["d"], case["h"], case["w"], 16), g),
                    w=_s8((k // 16, c // 16, ks, ks, ks, 4, 16, 4), g))
    if op == "chain":
        shape = (case["n"], 4, 56, 56, 16)
        return dict(case=case, x=_u8(shape, g), net=ConvChain(_chain_layers(case, g), shape))
    if op == "relay":
        c, k, ks = case["c"], case["k"], case["ks"]
        graph = Conv2dBiasMultiply(_s8((k, c, ks, ks), g), _bias(k, g), 11, case["stride"], case["pad"])
        return dict(case=case, x=_s8((case["n"], c, case["h"], case["w"]), g), net=graph)
    if op == "conv_f16":
        n, c, k, ks, h, w = (case[v] for v in ("n", "c", "k", "ks", "h", "w"))
        scale = 1.0 / math.sqrt(c * ks * ks)
        if case["operands"] == "nchw":
            return dict(case=case, x=_f16((n, c, h, w), g), w=_f16((k, c, ks, ks), g, scale))
        weight = _f16((k // 16, c // 16, ks, ks, 16, 16), g, scale)
        if case["operands"] == "prepared":
            weight = U.prepare_conv2d_weight(weight)
        return dict(case=case, x=_f16((n, c // 16, h, w, 16), g), w=weight)
    m, n, k = case["m"], case["n"], case["k"]
    if op == "gemm":
        b = _f16((k, n), g)
        ws = None
        if case["b"] == "prepared":
            b = U.prepare_gemm_b(b)
        elif case["b"] == "workspace":
            ws = torch.empty((max(16, U.gemm_fp16_workspace_bytes(m, n, k)),), dtype=torch.uint8, device="cuda")
        return dict(case=case, x=_f16((m, k), g, 1.0 / math.sqrt(k)), w=b, ws=ws)
    weight = _s8((n, k), g)
    if case["weights"] == "packed":
        weight = U.prepack_dense_weight(weight)
    elif case["weights"] == "prepared":
        weight = U.prepare_dense_weight(weight)
    return dict(case=case, x=_u8((m, k), g), w=weight)


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "conv":
        return U.conv2d_NCHWc_int8(state["x"], state["w"], case["stride"], case["pad"])
    if op == "fused":
        return U.conv2d_NCHWc_int8_fused(state["x"], state["w"], state["b"], 11, case["stride"], case["pad"])
    if op == "conv3d":
        return U.conv3d_NCDHWc_int8(state["x"], state["w"], case["stride"])
    if op == "chain":
        net = state["net"]
        net.run(state["x"])
        return tuple(net.outputs)
    if op == "relay":
        return state["net"](state["x"])
    if op == "conv_f16":
        return U.conv2d_NCHW16c_OHWI16o(state["x"], state["w"], case["stride"], case["stride"])
    if op == "gemm":
        return U.gemm_fp16(state["x"], state["w"], case["out"], workspace=state["ws"])
    if case["weights"] == "packed":
        return U.dense_dotprod(state["x"], state["w"])
    return U.dense(state["x"], state["w"])


# ------------------------------------------------------------------------------------- what a pass cannot do without
def _out(size, ks, stride, pad=0):
    return (size + 2 * pad - ks) // stride + 1


def work(case):
    op = case["op"]
    if op in ("gemm", "dense"):
        m, n, k = case["m"], case["n"], case["k"]
        es = 2 if op == "gemm" else 1
        out = 2 if case.get("out") == "float16" else 4
        return {"bytes": (m * k + n * k) * es + m * n * out, "flops": 2 * m * n * k}
    if op == "chain":
        # every layer's activations are results of the pass: written once; the input and the weights are read once
        layers = (resnet50_layers if case["net"] == "resnet50" else resnet18_layers)(lambda oc, ic, k: (oc, ic, k))
        n, sizes, macs = case["n"], [], 0
        total = n * 64 * 56 * 56
        for i, ly in enumerate(layers):
            oc, ic, k = ly.weight
            src = i - 1 if ly.source is None else ly.source
            size = _out(56 if src < 0 else sizes[src], k, ly.stride, ly.padding)
            sizes.append(size)
            total += oc * ic * k * k + n * oc * size * size
            macs += n * oc * ic * k * k * size * size
        return {"bytes": total, "flops": 2 * macs}
    n, c, h, w, k, ks, st = (case[v] for v in ("n", "c", "h", "w", "k", "ks", "stride"))
    pad = case.get("pad", 0)
    oh, ow = _out(h, ks, st, pad), _out(w, ks, st, pad)
    if op == "conv3d":
        od = _out(case["d"], ks, st)
        return {"bytes": n * c * case["d"] * h * w + k * c * ks ** 3 + 4 * n * k * od * oh * ow,
                "flops": 2 * n * k * od * oh * ow * c * ks ** 3}
    es = 2 if op == "conv_f16" else 1
    read = n * c * h * w if ks >= st else n * c * oh * ow  # a 1 x 1 window with stride 2 reads a quarter of the pixels
    return {"bytes": (read + k * c * ks * ks) * es + 4 * n * k * oh * ow, "flops": 2 * n * k * oh * ow * c * ks * ks}


def tolerance(case):
    op = case["op"]
    if op == "conv_f16" or (op == "gemm" and case["out"] == "float32"):
        # fp32 sums in another order: against the same products summed in 64 bits, 0.7e-7 .. 4.1e-7 and up to 3.4e-6
        return {"rel": 2e-6, "max": 2e-5}
    if op == "gemm":
        # one rounding to fp16: 2.1e-4 and 4.9e-4 against 64 bits
        return {"rel": 1e-3, "max": 2e-3}
    return "exact"
