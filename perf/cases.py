"""The work that users of this framework have it do, as timed cases: inference and training steps of
the approximate dense, convolution, matmul and attention layers over the sizes, tables and options of
the configurations in ``bench.py`` and ``tests/``, from the smallest layer to the largest product."""
import math

import torch

from approxtrain_amd import ApproxMulLut, lut_gen
from approxtrain_amd.layers import AMConv2D, MultiHeadAttention, denseam
from approxtrain_amd.math_ops import matmulam


def _dense(name, table, width, batch, fan_in, units, train):
    return {"name": name, "op": "dense", "table": table, "width": width, "batch": batch, "fan_in": fan_in,
            "units": units, "train": train}


def _conv(name, table, width, n, h, w, c, oc, k, stride, padding, bias_relu, train):
    return {"name": name, "op": "conv", "table": table, "width": width, "n": n, "h": h, "w": w, "c": c, "oc": oc,
            "k": k, "stride": stride, "padding": padding, "bias_relu": bias_relu, "train": train}


def _matmul(name, table, width, batch, m, k, n, transpose_b, train):
    return {"name": name, "op": "matmul", "table": table, "width": width, "batch": batch, "m": m, "k": k, "n": n,
            "transpose_b": transpose_b, "train": train}


def _attention(name, table, width, batch, seq, d_model, heads, mask, train):
    return {"name": name, "op": "attention", "table": table, "width": width, "batch": batch, "seq": seq,
            "d_model": d_model, "heads": heads, "mask": mask, "train": train}


def listed():
    return [
        # the smallest call: inference of LeNet-300-100's first layer, where launches and latency count
        _dense("dense_lenet300_infer", "MBM", 7, 128, 784, 300, False),
        # a small convolution's training step (LeNet-5's second layer) with Mitchell's multiplier
        _conv("conv_lenet5_train", "MIT", 7, 256, 14, 14, 6, 16, 5, 1, "VALID", True, True),
        # inference of an attention block over a few short sequences, with a padding mask
        _attention("attention_short_infer", "MIT", 7, 4, 50, 128, 4, True, False),
        # inference of one fused layer on an odd feature map with odd channel counts
        _conv("conv_odd_infer", "MIT", 5, 7, 35, 45, 37, 71, 3, 1, "SAME", True, False),
        # the headline layer: ResNet-50's first 3x3 convolution, forward and both gradients
        _conv("conv3x3_resnet_train", "MBM", 7, 32, 56, 56, 64, 64, 3, 1, "SAME", False, True),
        # a strided 3x3 layer, whose input gradient runs by residue classes
        _conv("conv3x3_stride2_train", "MBM", 7, 32, 56, 56, 128, 128, 3, 2, "SAME", False, True),
        # a 1x1 bottleneck layer late in the network: few pixels, many channels
        _conv("conv1x1_resnet_train", "MBM", 7, 32, 14, 14, 1024, 256, 1, 1, "SAME", False, True),
        # a middle layer's inference with the exactly multiplied, truncated product as the multiplier
        _conv("conv3x3_acc_infer", "ACC", 7, 32, 28, 28, 128, 128, 3, 1, "SAME", True, False),
        # the headline layer with a table too wide for the compute units' local memory
        _conv("conv3x3_wide_train", "MBM", 11, 32, 56, 56, 64, 64, 3, 1, "SAME", False, True),
        # a ragged product with a narrow table, the second operand stored transposed
        _matmul("matmul_ragged_train", "MBM", 3, 0, 1000, 2049, 515, True, True),
        # the encoder block's attention at full size, forward and backward
        _attention("attention_block_train", "MBM", 7, 32, 256, 512, 8, False, True),
        # the largest: a square product and both its gradients
        _matmul("matmul_4096_train", "MIT", 7, 0, 4096, 4096, 4096, False, True),
    ]


# tables in use, the full-width ones most often
_TABLES = (("MBM", 7), ("MBM", 7), ("MBM", 7), ("MBM", 7), ("MIT", 7), ("MIT", 7), ("ACC", 7), ("MBM", 5), ("MIT", 5),
           ("MBM", 3), ("MIT", 3), ("MIT", 1), ("MBM", 11), ("MIT", 11))
_MAX_MACS = 60.0e9        # of a drawn case with a table of at most 7 bits
_MAX_MACS_WIDE = 8.0e9    # ... of more than 7 bits


def _log_int(rng, lo, hi):
    """An integer from [lo, hi], spread over the logarithm; about half of them round numbers."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if v >= 16 and rng.random() < 0.5:
        step = 8 if v < 128 else 32
        v = int(round(v / step)) * step
    return min(max(v, lo), hi)


def draw(rng):
    while True:
        table, width = rng.choice(_TABLES)
        train = rng.random() < 0.6
        op = rng.choice(("dense", "conv", "conv", "matmul", "attention"))
        if op == "dense":
            c = _dense("", table, width, _log_int(rng, 16, 8192), _log_int(rng, 32, 4096), _log_int(rng, 10, 4096), train)
        elif op == "conv":
            k = rng.choice((1, 3, 3, 5))
            side = _log_int(rng, 7, 64)
            c = _conv("", table, width, _log_int(rng, 4, 256), side, side + rng.choice((0, 0, 3)), _log_int(rng, 3, 1024),
                      _log_int(rng, 6, 1024), k, rng.choice((1, 1, 2)), rng.choice(("SAME", "SAME", "VALID")),
                      rng.random() < 0.5, train)
        elif op == "matmul":
            c = _matmul("", table, width, rng.choice((0, 0, _log_int(rng, 2, 256))), _log_int(rng, 32, 4096),
                        _log_int(rng, 32, 4096), _log_int(rng, 32, 4096), rng.random() < 0.5, train)
        else:
            heads = rng.choice((2, 4, 8))
            c = _attention("", table, width, _log_int(rng, 2, 32), _log_int(rng, 20, 384), heads * rng.choice((16, 32, 64)),
                           heads, rng.random() < 0.5, train)
        del c["name"]
        if 5.0e6 <= _macs(c) <= (_MAX_MACS if width <= 7 else _MAX_MACS_WIDE) and work(c)["bytes"] <= 4.0e9:
            return c


# ---- what a user's program holds before the call ------------------------------------------------

def _lut(case):
    return ApproxMulLut.from_entries(lut_gen.generate_builtin(case["table"], case["width"], 1 if case["width"] <= 7 else 4),
                                     case["width"])


def _out_extent(size, k, stride, padding):
    return -(-size // stride) if padding == "SAME" else (size - k) // stride + 1


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)

    def normal(shape, scale=1.0):
        return torch.randn(shape, device="cuda", generator=gen) * scale

    def glorot(shape, fan_in, fan_out):
        limit = math.sqrt(6.0 / (fan_in + fan_out))
        return (torch.rand(shape, device="cuda", generator=gen) * 2 - 1) * limit

    lut = _lut(case)
    train = case["train"]
    s = {"case": case, "lut": lut, "train": train}
    if case["op"] == "dense":
        # pixels or post-sigmoid activations in, Glorot-uniform weights
        b, i, u = case["batch"], case["fan_in"], case["units"]
        layer = denseam(u, activation="relu", mant_mul_lut=lut, input_dim=i).cuda()
        with torch.no_grad():
            layer.kernel.copy_(glorot((i, u), i, u))
        s.update(layer=layer, x=torch.rand((b, i), device="cuda", generator=gen).requires_grad_(train),
                 wrt=[layer.kernel, layer.bias])
        if train:
            s["dy"] = normal((b, u), 1e-2)
    elif case["op"] == "conv":
        # post-ReLU activations in, He-normal filters, unit-normal upstream gradients
        n, h, w, c, oc, k = (case[v] for v in ("n", "h", "w", "c", "oc", "k"))
        layer = AMConv2D(oc, k, strides=case["stride"], padding=case["padding"].lower(), use_bias=case["bias_relu"],
                         activation="relu" if case["bias_relu"] else None, mant_mul_lut=lut, in_channels=c).cuda()
        with torch.no_grad():
            layer.kernel.copy_(normal((k, k, c, oc), math.sqrt(2.0 / (k * k * c))))
            if case["bias_relu"]:
                layer.bias.copy_(normal((oc,), 0.1))
        s.update(layer=layer, x=normal((n, h, w, c)).relu_().requires_grad_(train),
                 wrt=[layer.kernel] + ([layer.bias] if case["bias_relu"] else []))
        if train:
            s["dy"] = normal((n, _out_extent(h, k, case["stride"], case["padding"]),
                              _out_extent(w, k, case["stride"], case["padding"]), oc))
    elif case["op"] == "matmul":
        lead = (case["batch"],) if case["batch"] else ()
        m, k, n = case["m"], case["k"], case["n"]
        s["a"] = normal(lead + (m, k)).requires_grad_(train)
        s["b"] = normal(lead + ((n, k) if case["transpose_b"] else (k, n))).requires_grad_(train)
        if train:
            s["dy"] = normal(lead + (m, n))
    else:
        # unit-normal embeddings, Glorot-uniform projections; a mask hides each sequence's padding
        b, t, d = case["batch"], case["seq"], case["d_model"]
        block = MultiHeadAttention(lut, case["heads"], d, d, d, input_dim=d).cuda()
        with torch.no_grad():
            for p in (block.W_q, block.W_k, block.W_v, block.W_o):
                p.kernel.copy_(glorot((d, d), d, d))
        s.update(block=block, x=normal((b, t, d)).requires_grad_(train), mask=None)
        if case["mask"]:
            lengths = torch.randint(max(t // 2, 1), t + 1, (b,), device="cuda", generator=gen)
            s["mask"] = (torch.arange(t, device="cuda")[None, :] >= lengths[:, None]).float().reshape(b, 1, 1, t)
        s["wrt"] = [p.kernel for p in (block.W_q, block.W_k, block.W_v, block.W_o)]
        if train:
            s["dy"] = normal((b, t, d))
    return s


def _forward(s):
    case = s["case"]
    if case["op"] == "matmul":
        return matmulam(s["a"], s["b"], transpose_b=case["transpose_b"], mant_mul_lut=s["lut"])
    if case["op"] == "attention":
        return s["block"](s["x"], s["x"], s["x"], s["mask"])
    return s["layer"](s["x"])


def run(state):
    """One inference pass, or one training step's forward and backward passes."""
    if not state["train"]:
        with torch.no_grad():
            return _forward(state)
    out = _forward(state)
    wrt = [state["a"], state["b"]] if state["case"]["op"] == "matmul" else [state["x"]] + state["wrt"]
    return (out.detach(),) + torch.autograd.grad(out, wrt, state["dy"])


# ---- what a pass cannot do without ----------------------------------------------------------------

def _macs(case):
    """Products of one pass: the forward ones, and as many again for each operand's gradient."""
    if case["op"] == "dense":
        f = case["batch"] * case["fan_in"] * case["units"]
    elif case["op"] == "conv":
        oh = _out_extent(case["h"], case["k"], case["stride"], case["padding"])
        ow = _out_extent(case["w"], case["k"], case["stride"], case["padding"])
        f = case["n"] * oh * ow * case["oc"] * case["k"] ** 2 * case["c"]
    elif case["op"] == "matmul":
        f = max(case["batch"], 1) * case["m"] * case["k"] * case["n"]
    else:
        f = case["batch"] * case["seq"] * case["d_model"] * (4 * case["d_model"] + 2 * case["seq"])
    return f * (3 if case["train"] else 1)


def work(case):
    if case["op"] == "dense":
        x, w, y = case["batch"] * case["fan_in"], case["fan_in"] * case["units"], case["batch"] * case["units"]
        w += case["units"]
    elif case["op"] == "conv":
        oh = _out_extent(case["h"], case["k"], case["stride"], case["padding"])
        ow = _out_extent(case["w"], case["k"], case["stride"], case["padding"])
        x, w = case["n"] * case["h"] * case["w"] * case["c"], case["k"] ** 2 * case["c"] * case["oc"]
        w += case["oc"] if case["bias_relu"] else 0
        y = case["n"] * oh * ow * case["oc"]
    elif case["op"] == "matmul":
        b = max(case["batch"], 1)
        x, w, y = b * case["m"] * case["k"], b * case["k"] * case["n"], b * case["m"] * case["n"]
    else:
        x = y = case["batch"] * case["seq"] * case["d_model"]
        w = 4 * case["d_model"] * (case["d_model"] + 1)
    # a training step reads the upstream gradient as well and writes both operands' gradients
    elements = x + w + y + (x + w + y if case["train"] else 0)
    return {"bytes": 4 * elements, "flops": 2 * _macs(case)}


def tolerance(case):
    # 32-bit sums in another order.  Where one product's result is the next one's operand, a last-bit
    # difference may cross a truncation step of the multiplier's mantissa, and a rectifier may let a
    # sum near zero through or not.
    if case["op"] == "attention":
        return {"rel": 1e-3}
    return {"rel": 1e-5}
