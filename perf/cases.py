"""The work that users of this framework have it do, as cases that can be timed and checked.

A case is a dict of plain values; ``prepare`` builds what a program holds before its call (the imported model and the
inputs on the GPU, all made from the seed), ``run`` is one call of the model. Six kinds:

``encoder``   a transformer encoder layer given as an ONNX graph to ``ONNXModel`` (the layer of the headline benchmark;
              ``masked`` adds the padding mask of a batch of unequal sentences, ``exported`` writes LayerNormalization and
              Gelu node by node, the way opset-12 exports do, ``replayed`` is ``use_hip_graph=True``)
``convnet``   a residual image classifier in inference form: 7 x 7 stem, pooling, four stages of one residual block each,
              global pooling, a dense layer (convolutions with BatchNormalization, as exporters write them)
``mlp``       a small dense classifier, an ``nn.Sequential`` run through ``DaceModule``
``head``      a dense layer over a vocabulary or class list and its log-probabilities
``quantised`` a quantised dense layer: ``MatMulInteger`` with zero points and constant weights
``scores``    the tail of a classifier or of an attention block on its own: probabilities and the largest value of each row

Everything is fp32 except ``quantised``, as in the framework.
"""
import math

import numpy as np
import torch
import torch.nn as nn
import torch.nn.functional as F

import dace_onnx_amd.onnx as donnx
from dace_onnx_amd.onnx.proto import TensorProto, helper, numpy_helper
from dace_onnx_amd.pytorch.module import DaceModule

F32 = TensorProto.FLOAT


def listed():
    return [
        # one short query, host launches: a search or chat front end that encodes a sentence at a time
        {"name": "encoder_query", "kind": "encoder", "batch": 1, "seq": 16, "hidden": 768, "masked": False, "exported": False, "replayed": False},
        # one sentence of usual length, replayed as a HIP graph: what a latency-bound server switches on
        {"name": "encoder_replayed", "kind": "encoder", "batch": 1, "seq": 128, "hidden": 768, "masked": False, "exported": False, "replayed": True},
        # the layer of the headline benchmark
        {"name": "encoder_batch", "kind": "encoder", "batch": 8, "seq": 128, "hidden": 768, "masked": False, "exported": False, "replayed": False},
        # a batch of unequal sentences padded to an odd length, in the form an opset-12 export has
        {"name": "encoder_padded", "kind": "encoder", "batch": 5, "seq": 173, "hidden": 768, "masked": True, "exported": True, "replayed": False},
        # a full batch of long documents: offline embedding of a corpus
        {"name": "encoder_documents", "kind": "encoder", "batch": 16, "seq": 512, "hidden": 768, "masked": True, "exported": False, "replayed": False},
        # one photograph: interactive image classification
        {"name": "convnet_photo", "kind": "convnet", "batch": 1, "size": 224},
        # a full batch of photographs: offline labelling
        {"name": "convnet_batch", "kind": "convnet", "batch": 32, "size": 224},
        # a small dense classifier on a few samples (digits, tabular rows)
        {"name": "mlp_few", "kind": "mlp", "batch": 5, "inputs": 784, "width": 300, "classes": 10},
        # log-probabilities over a vocabulary for the tokens of a batch; the vocabulary has an even but otherwise awkward size
        {"name": "head_vocabulary", "kind": "head", "rows": 1024, "hidden": 768, "classes": 30522},
        # a quantised projection of the int8 benchmark's size
        {"name": "quantised_batch", "kind": "quantised", "rows": 4096, "inner": 768, "columns": 3072, "unsigned": False, "per_column": False},
        # a quantised layer of odd extents, uint8 activations, one weight zero point per column: dynamically quantised exports
        {"name": "quantised_odd", "kind": "quantised", "rows": 197, "inner": 501, "columns": 1001, "unsigned": True, "per_column": True},
        # attention-like probabilities over rows of odd length
        {"name": "scores_odd", "kind": "scores", "rows": 18912, "columns": 197},
    ]


def _log_int(rng, low, high):
    """An integer of [low, high], spread over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    most = work(listed()[4])["flops"]
    while True:
        kind = rng.choice(["encoder", "encoder", "encoder", "convnet", "convnet", "mlp", "head", "quantised", "quantised", "scores"])
        if kind == "encoder":
            case = {"kind": kind, "batch": _log_int(rng, 1, 32), "seq": _log_int(rng, 8, 512), "hidden": rng.choice([256, 512, 768, 1024]),
                    "masked": rng.random() < 0.5, "exported": rng.random() < 0.5, "replayed": rng.random() < 0.3}
        elif kind == "convnet":
            case = {"kind": kind, "batch": _log_int(rng, 1, 32), "size": rng.randint(96, 256)}
        elif kind == "mlp":
            case = {"kind": kind, "batch": _log_int(rng, 1, 512), "inputs": _log_int(rng, 64, 2048), "width": _log_int(rng, 64, 2048),
                    "classes": _log_int(rng, 2, 1000)}
        elif kind == "head":
            case = {"kind": kind, "rows": _log_int(rng, 1, 2048), "hidden": rng.choice([256, 512, 768, 1024]), "classes": _log_int(rng, 1000, 32000)}
        elif kind == "quantised":
            case = {"kind": kind, "rows": _log_int(rng, 1, 8192), "inner": _log_int(rng, 64, 3072), "columns": _log_int(rng, 64, 4096),
                    "unsigned": rng.random() < 0.5, "per_column": rng.random() < 0.5}
            if rng.random() < 0.5:   # layers of networks have round extents more often than not
                case["inner"], case["columns"] = max(64, case["inner"] // 64 * 64), max(64, case["columns"] // 64 * 64)
        else:
            case = {"kind": kind, "rows": _log_int(rng, 16, 65536), "columns": _log_int(rng, 16, 4096)}
            if case["rows"] * case["columns"] > 1 << 25:
                continue
        if work(case)["flops"] <= most:
            return case


# ------------------------------------------------------------------------------------------------ graphs


class _Graph:
    """Nodes and initializers of an ONNX graph under construction, kept plain: ``exact`` reads them too."""

    def __init__(self, opset):
        self.nodes, self.weights, self.opset = [], {}, opset

    def node(self, op, inputs, **attributes):
        out = f"{op.lower()}_{len(self.nodes)}"
        self.nodes.append((op, inputs, out, attributes))
        return out

    def weight(self, value, dtype=np.float32):
        name = f"w{len(self.weights)}"
        self.weights[name] = np.ascontiguousarray(value, dtype=dtype)
        return name

    def finish(self, name, inputs, outputs):
        self.name, self.inputs, self.outputs = name, inputs, outputs
        return self

    def model(self):
        infos = [helper.make_tensor_value_info(n, t, list(s)) for n, t, s in self.inputs]
        outs = [helper.make_tensor_value_info(n, t, list(s)) for n, t, s in self.outputs]
        nodes = [helper.make_node(op, inputs, [out], name=f"n{i}", **attributes) for i, (op, inputs, out, attributes) in enumerate(self.nodes)]
        weights = [numpy_helper.from_array(value, name) for name, value in self.weights.items()]
        graph = helper.make_graph(nodes, self.name, infos, outs, initializer=weights)
        return helper.make_model(graph, opset_imports=[helper.make_opsetid("", self.opset)])


def _normal(rng, *shape, scale=1.0):
    return rng.standard_normal(shape, dtype=np.float32) * np.float32(scale)


def _encoder_graph(case, rng):
    batch, seq, hidden = case["batch"], case["seq"], case["hidden"]
    size, heads, inner = 64, case["hidden"] // 64, 4 * case["hidden"]
    g = _Graph(12 if case["exported"] else 20)

    def dense(x, n_in, n_out):
        y = g.node("MatMul", [x, g.weight(_normal(rng, n_in, n_out, scale=0.02))])
        return g.node("Add", [y, g.weight(_normal(rng, n_out, scale=0.02))])

    def layer_norm(x):
        gamma, beta = g.weight(1 + _normal(rng, hidden, scale=0.02)), g.weight(_normal(rng, hidden, scale=0.02))
        if not case["exported"]:
            return g.node("LayerNormalization", [x, gamma, beta], axis=-1, epsilon=1e-12)
        centred = g.node("Sub", [x, g.node("ReduceMean", [x], axes=[-1], keepdims=1)])
        variance = g.node("ReduceMean", [g.node("Pow", [centred, g.weight(2.0)])], axes=[-1], keepdims=1)
        std = g.node("Sqrt", [g.node("Add", [variance, g.weight(1e-12)])])
        return g.node("Add", [g.node("Mul", [g.node("Div", [centred, std]), gamma]), beta])

    def gelu(x):
        if not case["exported"]:
            return g.node("Gelu", [x])
        t = g.node("Add", [g.node("Erf", [g.node("Div", [x, g.weight(math.sqrt(2.0))])]), g.weight(1.0)])
        return g.node("Mul", [g.node("Mul", [x, t]), g.weight(0.5)])

    split = g.weight([batch, seq, heads, size], np.int64)
    merge = g.weight([batch, seq, hidden], np.int64)
    heads_of = lambda x: g.node("Transpose", [g.node("Reshape", [x, split])], perm=[0, 2, 1, 3])  # noqa: E731
    q, k, v = (heads_of(dense("x", hidden, hidden)) for _ in range(3))
    scores = g.node("MatMul", [q, g.node("Transpose", [k], perm=[0, 1, 3, 2])])
    scores = g.node("Div", [scores, g.weight(math.sqrt(size))])
    if case["masked"]:
        scores = g.node("Add", [scores, "mask"])
    context = g.node("MatMul", [g.node("Softmax", [scores], axis=3), v])
    context = g.node("Reshape", [g.node("Transpose", [context], perm=[0, 2, 1, 3]), merge])
    attended = layer_norm(g.node("Add", [dense(context, hidden, hidden), "x"]))
    out = dense(gelu(dense(attended, hidden, inner)), inner, hidden)
    out = layer_norm(g.node("Add", [out, attended]))
    inputs = [("x", F32, (batch, seq, hidden))] + ([("mask", F32, (batch, 1, 1, seq))] if case["masked"] else [])
    return g.finish("encoder", inputs, [(out, F32, (batch, seq, hidden))])


def _convolved(extent, kernel, stride, pad):
    return (extent + 2 * pad - kernel) // stride + 1


def _convnet_layers(case):
    """(input channels, output channels, kernel, stride, input extent, output extent) of every convolution."""
    stem = _convolved(case["size"], 7, 2, 3)
    layers, extent, channels = [(3, 64, 7, 2, case["size"], stem)], _convolved(stem, 3, 2, 1), 64
    for stage, width in enumerate((64, 128, 256, 512)):
        stride = 1 if stage == 0 else 2
        out = _convolved(extent, 3, stride, 1)
        layers += [(channels, width, 3, stride, extent, out), (width, width, 3, 1, out, out)]
        if stride != 1:
            layers.append((channels, width, 1, stride, extent, out))
        extent, channels = out, width
    return layers


CONVNET_CLASSES = 1000


def _convnet_graph(case, rng):
    g = _Graph(12)

    def conv(x, c_in, c_out, kernel, stride):
        pad = kernel // 2
        w = g.weight(_normal(rng, c_out, c_in, kernel, kernel, scale=math.sqrt(2.0 / (c_in * kernel * kernel))))
        y = g.node("Conv", [x, w], kernel_shape=[kernel] * 2, pads=[pad] * 4, strides=[stride] * 2)
        stats = [1 + _normal(rng, c_out, scale=0.1), _normal(rng, c_out, scale=0.1), _normal(rng, c_out, scale=0.1), rng.uniform(0.5, 1.5, c_out)]
        return g.node("BatchNormalization", [y] + [g.weight(s) for s in stats], epsilon=1e-5)

    x = g.node("Relu", [conv("x", 3, 64, 7, 2)])
    x, channels = g.node("MaxPool", [x], kernel_shape=[3, 3], pads=[1] * 4, strides=[2, 2]), 64
    for stage, width in enumerate((64, 128, 256, 512)):
        stride = 1 if stage == 0 else 2
        y = conv(g.node("Relu", [conv(x, channels, width, 3, stride)]), width, width, 3, 1)
        skip = x if stride == 1 else conv(x, channels, width, 1, stride)
        x, channels = g.node("Relu", [g.node("Add", [y, skip])]), width
    x = g.node("Flatten", [g.node("GlobalAveragePool", [x])], axis=1)
    x = g.node("Gemm", [x, g.weight(_normal(rng, CONVNET_CLASSES, 512, scale=0.05)), g.weight(_normal(rng, CONVNET_CLASSES, scale=0.05))], transB=1)
    return g.finish("convnet", [("x", F32, (case["batch"], 3, case["size"], case["size"]))], [(x, F32, (case["batch"], CONVNET_CLASSES))])


def _head_graph(case, rng):
    g = _Graph(12)
    y = g.node("MatMul", ["x", g.weight(_normal(rng, case["hidden"], case["classes"], scale=0.05))])
    y = g.node("Add", [y, g.weight(_normal(rng, case["classes"], scale=0.05))])
    y = g.node("LogSoftmax", [y], axis=1)
    return g.finish("head", [("x", F32, (case["rows"], case["hidden"]))], [(y, F32, (case["rows"], case["classes"]))])


def _quantised_graph(case, rng):
    g = _Graph(12)
    a_type = np.uint8 if case["unsigned"] else np.int8
    weights = g.weight(rng.integers(-128, 128, (case["inner"], case["columns"]), dtype=np.int8), np.int8)
    a_zero = g.weight(121 if case["unsigned"] else 3, a_type)
    b_zero = g.weight(rng.integers(-8, 8, case["columns"], dtype=np.int8) if case["per_column"] else -2, np.int8)
    y = g.node("MatMulInteger", ["a", weights, a_zero, b_zero])
    return g.finish("quantised", [("a", TensorProto.UINT8 if case["unsigned"] else TensorProto.INT8, (case["rows"], case["inner"]))],
                   [(y, TensorProto.INT32, (case["rows"], case["columns"]))])


def _scores_graph(case, rng):
    g = _Graph(12)
    shape = (case["rows"], case["columns"])
    probabilities = g.node("Softmax", ["x"], axis=1)
    largest = g.node("ReduceMax", ["x"], axes=[1], keepdims=0)
    return g.finish("scores", [("x", F32, shape)], [(probabilities, F32, shape), (largest, F32, shape[:1])])


# ------------------------------------------------------------------------------------------------ the contract


_GRAPHS = {"encoder": _encoder_graph, "convnet": _convnet_graph, "head": _head_graph, "quantised": _quantised_graph, "scores": _scores_graph}


def _inputs(case, rng):
    """The arrays that a call gets; drawn after the weights."""
    kind = case["kind"]
    if kind == "encoder":
        inputs = [_normal(rng, case["batch"], case["seq"], case["hidden"])]
        if case["masked"]:
            lengths = rng.integers((case["seq"] + 1) // 2, case["seq"] + 1, size=case["batch"])
            padding = np.arange(case["seq"])[None, :] >= lengths[:, None]
            inputs.append((padding * np.float32(-10000.0)).astype(np.float32).reshape(case["batch"], 1, 1, case["seq"]))
        return inputs
    if kind == "convnet":
        return [_normal(rng, case["batch"], 3, case["size"], case["size"])]
    if kind == "mlp":
        return [_normal(rng, case["batch"], case["inputs"])]
    if kind == "head":
        return [_normal(rng, case["rows"], case["hidden"])]
    if kind == "quantised":
        low, high, dtype = (0, 256, np.uint8) if case["unsigned"] else (-128, 128, np.int8)
        return [rng.integers(low, high, (case["rows"], case["inner"]), dtype=dtype)]
    return [_normal(rng, case["rows"], case["columns"], scale=2.0)]


def _mlp_layers(case, rng):
    """(weight, bias) of the three dense layers."""
    sizes = [case["inputs"], case["width"], case["width"], case["classes"]]
    return [(_normal(rng, n_out, n_in, scale=1 / math.sqrt(n_in)), _normal(rng, n_out, scale=0.05)) for n_in, n_out in zip(sizes, sizes[1:])]


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "mlp":
        layers = []
        for weight, bias in _mlp_layers(case, rng):
            linear = nn.utils.skip_init(nn.Linear, weight.shape[1], weight.shape[0])
            with torch.no_grad():
                linear.weight.copy_(torch.from_numpy(weight))
                linear.bias.copy_(torch.from_numpy(bias))
            layers += [linear, nn.ReLU()]
        module = nn.Sequential(*layers[:-1], nn.Softmax(dim=1)).cuda().eval()
        x = torch.from_numpy(_inputs(case, rng)[0]).cuda()
        model = DaceModule(module, dummy_inputs=(x,), sdfg_name="mlp")
        return {"model": model, "inputs": [x]}
    model = donnx.ONNXModel(kind, _GRAPHS[kind](case, rng).model(), use_hip_graph=bool(case.get("replayed", False)))
    return {"model": model, "inputs": [torch.from_numpy(a).cuda() for a in _inputs(case, rng)]}


def run(state):
    with torch.no_grad():
        return state["model"](*state["inputs"])


def work(case):
    kind = case["kind"]
    if kind == "encoder":
        batch, seq, hidden = case["batch"], case["seq"], case["hidden"]
        tokens = batch * seq
        weights = 12 * hidden * hidden + 13 * hidden
        return {"bytes": 4.0 * (2 * tokens * hidden + weights + (tokens if case["masked"] else 0)),
                "flops": 24.0 * tokens * hidden * hidden + 4.0 * batch * seq * seq * hidden}
    if kind == "convnet":
        layers = _convnet_layers(case)
        weights = sum(c_in * c_out * k * k + c_out for c_in, c_out, k, _, _, _ in layers) + 513 * CONVNET_CLASSES
        flops = sum(2.0 * c_in * c_out * k * k * out * out for c_in, c_out, k, _, _, out in layers) + 2.0 * 512 * CONVNET_CLASSES
        return {"bytes": 4.0 * (case["batch"] * (3 * case["size"] ** 2 + CONVNET_CLASSES) + weights), "flops": case["batch"] * flops}
    if kind == "mlp":
        macs = case["inputs"] * case["width"] + case["width"] ** 2 + case["width"] * case["classes"]
        return {"bytes": 4.0 * (macs + 2 * case["width"] + case["classes"] + case["batch"] * (case["inputs"] + case["classes"])),
                "flops": 2.0 * case["batch"] * macs}
    if kind == "head":
        rows, hidden, classes = case["rows"], case["hidden"], case["classes"]
        return {"bytes": 4.0 * (rows * hidden + (hidden + 1) * classes + rows * classes), "flops": 2.0 * rows * hidden * classes}
    if kind == "quantised":
        rows, inner, columns = case["rows"], case["inner"], case["columns"]
        return {"bytes": float(rows * inner + inner * columns + 4 * rows * columns), "flops": 2.0 * rows * inner * columns}
    return {"bytes": 4.0 * case["rows"] * (2 * case["columns"] + 1), "flops": 5.0 * case["rows"] * case["columns"]}


# Sums over a window and the running sums of a matrix product are taken in float64, whole numbers too: below 2**53 they are exact.


def _exact_conv(x, w, kernel_shape, pads, strides):
    columns = F.unfold(x, kernel_shape, padding=pads[0], stride=strides[0])
    rows, cols = (_convolved(x.shape[axis], kernel_shape[0], strides[0], pads[0]) for axis in (2, 3))
    return torch.stack([w.reshape(w.shape[0], -1) @ image for image in columns]).reshape(x.shape[0], w.shape[0], rows, cols)


def _exact_batch_norm(x, scale, shift, mean, variance, epsilon):
    scale, shift, mean, variance = (v.reshape(1, -1, 1, 1) for v in (scale, shift, mean, variance))
    return (x - mean) / torch.sqrt(variance + epsilon) * scale + shift


def _exact_layer_norm(x, gamma, beta, axis, epsilon):
    centred = x - x.mean(dim=axis, keepdim=True)
    return centred / torch.sqrt((centred * centred).mean(dim=axis, keepdim=True) + epsilon) * gamma + beta


_EXACT = {
    "MatMul": torch.matmul, "Add": torch.add, "Sub": torch.sub, "Mul": torch.mul, "Div": torch.div, "Pow": torch.pow, "Sqrt": torch.sqrt,
    "Erf": torch.erf, "Relu": torch.relu, "Gelu": F.gelu, "LayerNormalization": _exact_layer_norm, "BatchNormalization": _exact_batch_norm,
    "Reshape": lambda x, shape: x.reshape([int(n) for n in shape]), "Transpose": lambda x, perm: x.permute(perm).contiguous(),
    "Softmax": lambda x, axis: torch.softmax(x, axis), "LogSoftmax": lambda x, axis: torch.log_softmax(x, axis),
    "ReduceMean": lambda x, axes, keepdims: x.mean(dim=axes, keepdim=bool(keepdims)),
    "ReduceMax": lambda x, axes, keepdims: x.amax(dim=axes, keepdim=bool(keepdims)),
    "Conv": _exact_conv, "MaxPool": lambda x, kernel_shape, pads, strides: F.max_pool2d(x, kernel_shape, strides, pads[0]),
    "GlobalAveragePool": lambda x: x.mean(dim=(2, 3), keepdim=True), "Flatten": lambda x, axis: x.flatten(axis),
    "Gemm": lambda x, w, b, transB: x @ w.t() + b, "MatMulInteger": lambda a, b, a_zero, b_zero: (a - a_zero) @ (b - b_zero),
}


def exact(case, seed):
    rng = np.random.default_rng(seed)
    device = "cuda" if torch.cuda.is_available() else "cpu"
    wide = lambda a: torch.from_numpy(a).to(device, torch.float64)  # noqa: E731
    if case["kind"] == "mlp":
        layers = _mlp_layers(case, rng)
        x = wide(_inputs(case, rng)[0])
        for i, (weight, bias) in enumerate(layers):
            x = x @ wide(weight).t() + wide(bias)
            x = torch.relu(x) if i + 1 < len(layers) else torch.softmax(x, 1)
        return x
    graph = _GRAPHS[case["kind"]](case, rng)
    values = {name: wide(value) for name, value in graph.weights.items()}
    values.update({name: wide(array) for (name, _, _), array in zip(graph.inputs, _inputs(case, rng))})
    for op, inputs, out, attributes in graph.nodes:
        values[out] = _EXACT[op](*(values[name] for name in inputs), **attributes)
    outputs = [values[name] for name, _, _ in graph.outputs]
    if case["kind"] == "quantised":
        outputs = [outputs[0].to(torch.int32)]
    return outputs[0] if len(outputs) == 1 else tuple(outputs)


def tolerance(case):
    # four times what the path shows against the same graph evaluated in float64 (encoder 3.2e-7 / 2.7e-6, convnet 3.1e-7 /
    # 1.3e-6, mlp 2.5e-7 / 0.7e-6, head 0.8e-7 / 1.0e-6, scores 0.6e-7 / 0.3e-6), the largest difference rounded up
    return {"encoder": {"rel": 1.4e-6, "max": 1.2e-5}, "convnet": {"rel": 1.3e-6, "max": 8e-6}, "mlp": {"rel": 1e-6, "max": 6e-6},
            "head": {"rel": 4e-7, "max": 5e-6}, "quantised": "exact", "scores": {"rel": 2.5e-7, "max": 1.5e-6}}[case["kind"]]
