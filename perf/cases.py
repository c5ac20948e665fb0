"""The work that a user of this framework has it do, as cases with their inputs, one pass of each, and what a pass cannot do without.

A case is a dict: `kind` names the path and the other entries its sizes and options.

  forward         StochasticLut<n> on fp32 frames, forward only: evaluating a trained layer, down to a handful of frames
  stochastic      StochasticLut<n> training step of a layer: forward (table clamped first) and backward (dW, dx)
  differentiable  DifferentiableLut<n> training step of a layer (per-node batch-norm): `form` "fp32" binarizes fp32 activations (the class's
                  default), "bits" works on packed activations, "real" keeps real-valued activations (binary mode off)
  classifier      training step of the LUT classifier: three DifferentiableLut6 layers, AverageLut, softmax cross entropy, accuracy, Adam
  conv            forward and backward of the convolutional block: Im2Col 3x3, two DifferentiableLut6 layers per pixel, Col2Im, 2x2 pooling
  binary          BinaryLut<n> inference of one layer on packed frames
  serve           inference of a whole packed network on real inputs: RealToBinary with frame modulation, three layers (`lut`: "differentiable"
                  with running statistics, or "binary" truth tables), BinaryToReal

Inputs are drawn from the seed alone: uniform frames, normal gradients, fair bits, wiring of n distinct inputs per node, tables around one half.
"""
import math

import numpy as np
import torch

from binarybrain_amd import ops, synth

CLASSES, VOTES = 10, 7          # ten classes, seven voting nodes each: the last LUT layer of the classifier has 70 nodes


def listed():
    return [
        # a small trained layer on one wavefront of frames: latency and launches
        {"name": "forward_784x1024x64", "kind": "forward", "n": 6, "inputs": 784, "nodes": 1024, "frames": 64, "binary": False},
        # the headline configuration: one large layer, forward and backward
        {"name": "stochastic_4096x4096x8192", "kind": "stochastic", "n": 6, "inputs": 4096, "nodes": 4096, "frames": 8192, "binary": False},
        # a medium layer of another width, with sizes that divide nothing
        {"name": "stochastic4_1001x1531x1999", "kind": "stochastic", "n": 4, "inputs": 1001, "nodes": 1531, "frames": 1999, "binary": False},
        # a large layer of a binary network on fp32 activations
        {"name": "differentiable_fp32_4096x4096x8192", "kind": "differentiable", "form": "fp32", "n": 6, "inputs": 4096, "nodes": 4096, "frames": 8192},
        # the same layer type on packed activations, with a ragged last word and unequal layer sizes
        {"name": "differentiable_bits_2001x3003x5005", "kind": "differentiable", "form": "bits", "n": 6, "inputs": 2001, "nodes": 3003, "frames": 5005},
        # a layer trained with real-valued activations
        {"name": "differentiable_real_1024x1024x1000", "kind": "differentiable", "form": "real", "n": 6, "inputs": 1024, "nodes": 1024, "frames": 1000},
        # the classifier's training step at its full batch, and at the batch of a notebook with a smaller network
        {"name": "classifier_784_6144_1024_x1024", "kind": "classifier", "hidden1": 6144, "hidden2": 1024, "frames": 1024},
        {"name": "classifier_784_1024_360_x64", "kind": "classifier", "hidden1": 1024, "hidden2": 360, "frames": 64},
        # the convolutional block on colour images, and on the odd last batch of small grey ones
        {"name": "conv_256x3x32x32", "kind": "conv", "images": 256, "channels": 3, "size": 32, "hidden1": 216, "hidden2": 36},
        {"name": "conv_50x1x28x28", "kind": "conv", "images": 50, "channels": 1, "size": 28, "hidden1": 72, "hidden2": 24},
        # packed inference of one very large layer: throughput
        {"name": "binary_8192x16384x262144", "kind": "binary", "n": 6, "inputs": 8192, "nodes": 16384, "frames": 262144},
        # a network evaluated on a ragged batch with seven modulated frames per input frame
        {"name": "serve_784_2048_512_x500x7", "kind": "serve", "lut": "differentiable", "hidden1": 2048, "hidden2": 512, "frames": 500, "modulation": 7},
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["forward", "stochastic", "differentiable", "differentiable", "classifier", "conv", "binary", "serve"])
    width = rng.choice([2, 3, 4, 4, 5, 6, 6, 6])
    if kind in ("forward", "stochastic", "differentiable"):
        form = rng.choice(["fp32", "bits", "real"])
        most = 1 << (24 if form == "real" and kind == "differentiable" else 25)         # elements of the larger of x and y
        while True:
            inputs, nodes, frames = _spread(rng, 32, 4096), _spread(rng, 32, 8192), _spread(rng, 1 if kind == "forward" else 16, 8192)
            if max(inputs, nodes) * frames <= most:
                break
        case = {"kind": kind, "n": width, "inputs": inputs, "nodes": nodes, "frames": frames}
        case.update({"form": form} if kind == "differentiable" else {"binary": rng.random() < 0.25})
        return case
    if kind == "classifier":
        return {"kind": kind, "hidden1": _spread(rng, 256, 6144), "hidden2": _spread(rng, 100, 1024), "frames": _spread(rng, 16, 1024)}
    if kind == "conv":
        while True:
            case = {"kind": kind, "images": _spread(rng, 4, 256), "channels": rng.choice([1, 3]), "size": rng.randint(10, 34),
                    "hidden1": _spread(rng, 24, 216), "hidden2": _spread(rng, 12, 36)}
            if case["images"] * (case["size"] - 2) ** 2 * (case["hidden1"] + case["hidden2"]) <= 256 * 900 * 252:
                return case
    if kind == "binary":
        while True:
            inputs, nodes, frames = _spread(rng, 64, 8192), _spread(rng, 64, 16384), _spread(rng, 32, 262144)
            if inputs * frames <= 1 << 31 and nodes * frames <= 1 << 32:
                return {"kind": kind, "n": width, "inputs": inputs, "nodes": nodes, "frames": frames}
    return {"kind": kind, "lut": rng.choice(["differentiable", "binary"]), "hidden1": _spread(rng, 256, 6144), "hidden2": _spread(rng, 100, 1024),
            "frames": _spread(rng, 1, 1024), "modulation": rng.choice([1, 3, 7, 15, 31])}


# ---- inputs ----------------------------------------------------------------------------------------------------------
def _rows(draw_into, rows, frames):
    """[rows, stride] float32 of the framework's frame layout: values in the frames in use, zero padding"""
    a = torch.zeros((rows, synth.frame_stride_fp32(frames)), device="cuda")
    draw_into(a[:, :frames])
    return a


def _bits(gen, rows, frames):
    """[rows, words] fair bits, zero past the last frame"""
    a = torch.zeros((rows, synth.frame_stride_bit(frames)), dtype=torch.int32, device="cuda")
    words = (frames + 31) // 32
    a[:, :words] = torch.randint(-(1 << 31), 1 << 31, (rows, words), device="cuda", generator=gen).to(torch.int32)
    if frames & 31:
        a[:, words - 1] &= (1 << (frames & 31)) - 1
    return a


def _layer(rng, gen, n, inputs, nodes, frames, spread=None, train=True):
    """A LUT layer as a program keeps it: wiring and reverse wiring, table, gradient, statistics, and the buffers kept from forward to backward"""
    idx = torch.from_numpy(synth.wiring(rng, inputs, nodes, n)).cuda()
    W = torch.rand((nodes, 1 << n), device="cuda", generator=gen) if spread is None else \
        0.5 + spread * torch.randn((nodes, 1 << n), device="cuda", generator=gen)
    layer = {"n": n, "inputs": inputs, "nodes": nodes, "idx": idx, "W": W, "rm": torch.zeros(nodes, device="cuda"), "rv": torch.ones(nodes, device="cuda")}
    if train:
        layer.update(dW=torch.zeros_like(W), rev=ops.reverse_table(idx, inputs), tables=ops.prepared_tables_buffer(n, nodes),
                     packed=ops.packed_input_buffer(inputs, frames))
    return layer


def _truth_tables(rng, n, nodes):
    words = rng.integers(0, 1 << min(32, 1 << n), size=(nodes, 2 if n == 6 else 1), dtype=np.uint64)
    return torch.from_numpy(words.astype(np.uint32).view(np.int32)).cuda()


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    uniform = lambda a: a.copy_(torch.rand(a.shape, device="cuda", generator=gen))          # noqa: E731
    normal = lambda a: a.copy_(torch.randn(a.shape, device="cuda", generator=gen))          # noqa: E731
    s = dict(case)
    kind, F = case["kind"], case.get("frames")
    if kind in ("forward", "stochastic"):
        s["layer"] = _layer(rng, gen, case["n"], case["inputs"], case["nodes"], F, train=kind == "stochastic")
        s["x"] = _rows(uniform, case["inputs"], F)
        if kind == "stochastic":
            s["dy"] = _rows(normal, case["nodes"], F)
    elif kind == "differentiable":
        s["layer"] = _layer(rng, gen, case["n"], case["inputs"], case["nodes"], F)
        s["x"] = _bits(gen, case["inputs"], F) if case["form"] == "bits" else _rows(uniform, case["inputs"], F)
        s["dy"] = _rows(normal, case["nodes"], F)
        s["y_bits"] = torch.zeros((case["nodes"], s["x"].shape[1]), dtype=torch.int32, device="cuda") if case["form"] == "bits" else \
            ops.packed_input_buffer(case["nodes"], F)
    elif kind == "classifier":
        sizes = [784, case["hidden1"], case["hidden2"], CLASSES * VOTES]
        s["layers"] = [_layer(rng, gen, 6, i, o, F, 0.01) for i, o in zip(sizes[:-1], sizes[1:])]
        s["votes"] = torch.arange(sizes[-1], dtype=torch.int32, device="cuda").reshape(CLASSES, VOTES).contiguous()
        s["x"] = _rows(uniform, sizes[0], F)
        s["t"] = torch.zeros((CLASSES, s["x"].shape[1]), device="cuda")
        s["t"][torch.from_numpy(rng.integers(0, CLASSES, F)).cuda(), torch.arange(F, device="cuda")] = 1.0
        s["adam"] = ops.AdamState([l["W"] for l in s["layers"]], [l["dW"] for l in s["layers"]], learning_rate=0.001)
    elif kind == "conv":
        images, channels, size = case["images"], case["channels"], case["size"]
        s["windows"] = images * (size - 2) ** 2
        sizes = [9 * channels, case["hidden1"], case["hidden2"]]
        s["layers"] = [_layer(rng, gen, 6, i, o, s["windows"], 0.1) for i, o in zip(sizes[:-1], sizes[1:])]
        s["x"] = _rows(uniform, channels * size * size, images)
        s["dy"] = _rows(normal, case["hidden2"] * ((size - 1) // 2) ** 2, images)
    elif kind == "binary":
        s["idx"] = torch.from_numpy(synth.wiring(rng, case["inputs"], case["nodes"], case["n"])).cuda()
        s["table"] = _truth_tables(rng, case["n"], case["nodes"])
        s["x"] = _bits(gen, case["inputs"], F)
        s["y"] = torch.zeros((case["nodes"], s["x"].shape[1]), dtype=torch.int32, device="cuda")
    else:
        sizes = [784, case["hidden1"], case["hidden2"], CLASSES * VOTES]
        s["layers"] = [_layer(rng, gen, 6, i, o, F, 0.2, train=False) for i, o in zip(sizes[:-1], sizes[1:])]
        for l in s["layers"]:
            # a trained node: its statistics are near those of its table over fair bits
            l["rm"], l["rv"] = l["W"].mean(dim=1).contiguous(), l["W"].var(dim=1, unbiased=False).mul_(0.25).contiguous()
            l["table"] = _truth_tables(rng, 6, l["nodes"])
        s["x"] = _rows(uniform, sizes[0], F)
    return s


# ---- one pass --------------------------------------------------------------------------------------------------------
def run(s):
    return {"forward": _run_forward, "stochastic": _run_stochastic, "differentiable": _run_differentiable, "classifier": _run_classifier,
            "conv": _run_conv, "binary": _run_binary, "serve": _run_serve}[s["kind"]](s)


def _run_forward(s):
    l, F = s["layer"], s["frames"]
    return ops.stochastic_lut_forward(l["n"], s["x"], l["idx"], l["W"], F, input_binary=s["binary"])[:, :F]


def _run_stochastic(s):
    l, F = s["layer"], s["frames"]
    y = ops.stochastic_lut_forward(l["n"], s["x"], l["idx"], l["W"], F, input_binary=s["binary"], clamp_w=(0.0, 1.0))
    dx = ops.stochastic_lut_backward(l["n"], s["x"], s["dy"], l["idx"], l["W"], l["dW"], F, l["rev"], input_binary=s["binary"])
    return {"y": y[:, :F], "dx": dx[:, :F], "dW": l["dW"], "W": l["W"]}


def _run_differentiable(s):
    l, F, form = s["layer"], s["frames"], s["form"]
    common = (l["idx"], l["W"], F, l["rm"], l["rv"])
    if form == "bits":
        y, mean, rstd = ops.bit_differentiable_lut_forward_training(l["n"], s["x"], *common, clamp_w=(0.0, 1.0), tables=l["tables"], out=s["y_bits"])
        dx = ops.bit_differentiable_lut_backward(l["n"], s["x"], s["dy"], l["idx"], l["W"], l["dW"], F, mean, rstd, l["rev"], tables=l["tables"])
    elif form == "fp32":
        # the layer behind takes the binarized activation as packed bits
        y, mean, rstd = ops.differentiable_lut_forward_training(l["n"], s["x"], *common, clamp_w=(0.0, 1.0), packed=l["packed"], tables=l["tables"],
                                                                packed_out=s["y_bits"])
        dx = ops.differentiable_lut_backward(l["n"], s["x"], s["dy"], l["idx"], l["W"], l["dW"], F, mean, rstd, l["rev"], packed=l["packed"],
                                             tables=l["tables"])
        y = s["y_bits"]
    else:
        y, mean, rstd = ops.differentiable_lut_forward_training(l["n"], s["x"], *common, binary_mode=False, clamp_w=(0.0, 1.0), tables=l["tables"])
        dx = ops.differentiable_lut_backward(l["n"], s["x"], s["dy"], l["idx"], l["W"], l["dW"], F, mean, rstd, l["rev"], binary_mode=False,
                                             tables=l["tables"])
    y = y[:, :F] if form == "real" else y[:, :(F + 31) // 32]
    return {"y": y, "dx": dx[:, :F], "dW": l["dW"], "mean": mean, "rstd": rstd, "running_mean": l["rm"], "running_var": l["rv"]}


def _layers_forward(layers, a, F):
    """The training forward of binary layers on fp32 activations, each handing its packed output to the next; the activations for the backward pass"""
    kept = []
    for k, l in enumerate(layers):
        following = layers[k + 1]["packed"] if k + 1 < len(layers) else None
        y, mean, rstd = ops.differentiable_lut_forward_training(6, a, l["idx"], l["W"], F, l["rm"], l["rv"], clamp_w=(0.0, 1.0), packed=l["packed"],
                                                                packed_holds=k > 0, packed_out=following, tables=l["tables"])
        kept.append((a, mean, rstd))
        a = y
    return a, kept


def _layers_backward(layers, kept, dy, F, overwrite):
    for l, (a, mean, rstd) in zip(reversed(layers), reversed(kept)):
        dy = ops.differentiable_lut_backward(6, a, dy, l["idx"], l["W"], l["dW"], F, mean, rstd, l["rev"], packed=l["packed"], tables=l["tables"],
                                             overwrite_dw=overwrite)
    return dy


def _run_classifier(s):
    layers, F, adam = s["layers"], s["frames"], s["adam"]
    a, kept = _layers_forward(layers, s["x"], F)
    _, dy, loss, hits, _, _ = ops.classifier_tail(a, s["votes"], s["t"], F, t_sum=float(F), mean=False)
    dx = _layers_backward(layers, kept, dy, F, False)
    adam.update()
    return {"loss": loss, "hits": hits, "dx": dx[:, :F], "W": [l["W"] for l in layers], "m": adam.m, "v": adam.v,
            "running_mean": [l["rm"] for l in layers], "running_var": [l["rv"] for l in layers]}


def _run_conv(s):
    layers, images, channels, size, F = s["layers"], s["images"], s["channels"], s["size"], s["windows"]
    out = size - 2
    cols = ops.im2col_forward(s["x"], channels, size, size, images, 3, 3)
    a, kept = _layers_forward(layers, cols, F)
    maps = ops.col2im_forward(a, s["hidden2"], out, out, images)
    pooled = ops.stochastic_maxpool2x2_forward(maps, s["hidden2"], out, out, images)
    dmaps = ops.stochastic_maxpool2x2_backward(maps, s["dy"], s["hidden2"], out, out, images)
    dy = _layers_backward(layers, kept, ops.col2im_backward(dmaps, s["hidden2"], out, out, images), F, True)
    dx = ops.im2col_backward(dy, channels, size, size, images, 3, 3)
    return {"pooled": pooled[:, :images], "dx": dx[:, :images], "dW": [l["dW"] for l in layers], "running_mean": [l["rm"] for l in layers],
            "running_var": [l["rv"] for l in layers]}


def _run_binary(s):
    return ops.binary_lutn_forward(s["n"], s["x"], s["idx"], s["table"], s["frames"], out=s["y"])[:, :(s["frames"] + 31) // 32]


def _run_serve(s):
    F, m = s["frames"], s["modulation"]
    a = ops.real_to_binary_forward(s["x"], 1, 784, F, m, bit=True, y_stride=synth.frame_stride_bit(F * m))
    for l in s["layers"]:
        if s["lut"] == "binary":
            a = ops.binary_lutn_forward(6, a, l["idx"], l["table"], F * m)
        else:
            a = ops.bit_differentiable_lut_forward_inference(6, a, l["idx"], l["W"], F * m, l["rm"], l["rv"])
    return ops.binary_to_real_forward(a, CLASSES, F, m)


# ---- what a pass cannot do without -----------------------------------------------------------------------------------
def _table_bytes(n, nodes):
    return nodes * (4 * n + (4 << n))


def work(case):
    """Every input of the pass read once and every output written once (between the layers of a network: a binary activation at one bit, a
    gradient at four bytes, written once and read once).  Operations: a multilinear polynomial of 2^n coefficients per node and frame, by
    Horner's rule 2^n - 1 multiply-adds forward, 2^n for the table gradient and 2 * 2^n for the input gradients; on two-valued inputs a table
    lookup (n operations), one addition and n multiply-adds."""
    kind, F = case["kind"], case.get("frames")

    def operations(n, nodes, frames, two_valued, train):
        per = (n + (2 + 2 * n) * train) if two_valued else 2 * ((1 << n) - 1) + 6 * (1 << n) * train
        return float(nodes) * frames * per

    if kind in ("forward", "stochastic", "differentiable"):
        n, I, O = case["n"], case["inputs"], case["nodes"]
        train = kind != "forward"
        two = case.get("binary", False) or case.get("form") in ("fp32", "bits")
        bits = case.get("form") == "bits"
        nbytes = (I + O) * F / 8 if bits else 4 * F * I + (F * O / 8 if case.get("form") == "fp32" else 4 * F * O)
        nbytes += _table_bytes(n, O)
        if train:
            nbytes += 4 * F * (I + O) + 8 * O * (1 << n)
        return {"bytes": nbytes, "flops": operations(n, O, F, two, train)}
    if kind == "classifier" or kind == "serve":
        sizes = [784, case["hidden1"], case["hidden2"], CLASSES * VOTES]
        train = kind == "classifier"
        frames = F if train else F * case["modulation"]
        nbytes = 4 * 784 * F
        flops = 0.0
        for k, (i, o) in enumerate(zip(sizes[:-1], sizes[1:])):
            nbytes += (_table_bytes(6, o) if train or case["lut"] == "differentiable" else 32 * o) + frames * o / 8 * 2
            if train:
                nbytes += 4 * F * (i * (1 if k == 0 else 2)) + 6 * 256 * o      # gradients; W written, moments read and written, dW written, cleared
            flops += operations(6, o, frames, True, train)
        return {"bytes": nbytes + 4 * CLASSES * F, "flops": flops}
    if kind == "conv":
        images, channels, size = case["images"], case["channels"], case["size"]
        out = size - 2
        frames = images * out * out
        sizes = [9 * channels, case["hidden1"], case["hidden2"]]
        nbytes = 8 * images * channels * size * size + 8 * images * case["hidden2"] * ((size - 1) // 2) ** 2
        flops = 0.0
        for i, o in zip(sizes[:-1], sizes[1:]):
            nbytes += frames * o / 8 * 2 + 8 * frames * o + _table_bytes(6, o) + 256 * o
            flops += operations(6, o, frames, True, True)
        return {"bytes": nbytes, "flops": flops}
    n, I, O = case["n"], case["inputs"], case["nodes"]
    return {"bytes": F / 8 * (I + O) + O * (4 * n + (8 if n == 6 else 4)), "flops": float(n) * O * F / 32}


def tolerance(case):
    """fp32 sums in another order; where a network binarizes or clips at a threshold a frame within rounding of it may fall on the other side."""
    kind = case["kind"]
    if kind in ("binary", "serve"):
        return {"rel": 1e-4, "max": 0.5, "differ": 1e-4} if case.get("lut") == "differentiable" else "exact"
    if kind == "forward":
        return {"rel": 1e-6, "max": 1e-5} if case["binary"] else {"rel": 2e-6, "max": 2e-5}
    if kind == "stochastic":
        return {"rel": 1e-5, "max": 2e-4}
    return {"rel": 1e-4, "max": 0.5, "differ": 1e-4}
