"""Constant operands of contractions, packed for the kernels of ``csrc/gemm_f32_packed.hip`` and ``csrc/conv2d_f32_packed.hip`` when a
graph is compiled.

A packed copy holds three bf16 parts of every value in the order in which the matrix unit takes them (``csrc/split_bf16.h``); it is
made once, on the GPU. The reference has no counterpart: its constants are handed to a BLAS
library as they are.
"""
import numpy as np
import torch

from .. import _lib
from ..sdfg import AccessNode, AliasNode, I64Array, KernelCall, PackedCopy, Ptr, Stream, float32, int32
from .fusion import _in_edge, _out_edge, _single_consumer


class PackedOperand:
    """The packed copy ``array`` of a weight, ``shape`` 32-bit words, written by the library's ``function`` from ``offset`` values on.

    The launches that multiply by it get the weight's address too, and read the weight itself where the copy is left out. It is made at
    once (``now``) of a weight that only the model holds (``onnx/weights.py``), and of others on request.
    """

    def __init__(self, model, weight_name, descriptor, now, array, shape, function, geometry, offset):
        self.weights, self.weight_name, self.descriptor, self.array = model.weights, weight_name, descriptor, array
        self.shape, self.function, self.geometry, self.offset = shape, function, geometry, offset
        self.derived = model.weights.derived(weight_name)
        self.device, self.weight, self.version, self.packed, self.declared = model.device, None, None, None, False
        self.record = None   # what csrc/host_call.cpp decides current() by
        if now and model.weights.private(weight_name):
            self.pack()

    def pack(self, declared=False):
        """``declared``: the caller answers for what is written into the weight from here on."""
        weight = self.weights.peek(self.weight_name)
        if not isinstance(weight, torch.Tensor) or weight.dtype != torch.float32 or tuple(weight.shape) != self.descriptor.shape \
                or not weight.is_contiguous() or weight.device != self.device:
            return
        self.weight, self.declared = weight, declared
        # how often it was written in place, as far as torch counts it; tensors made under torch.inference_mode have no such count
        self.version = None if weight.is_inference() else weight._version
        if self.packed is None:
            self.packed = torch.empty(self.shape, dtype=torch.int32, device=self.device)
        self.record = (self.weight_name, weight, self.version, self.derived or declared, self.packed)
        start = weight.data_ptr() + 4 * self.offset
        _lib.check(getattr(_lib.library(), self.function)(start, self.packed.data_ptr(), *self.geometry, _lib.current_stream()), self.function)

    def current(self):
        """Whether the model's weight is still the tensor that was packed, and not written since as far as can be told."""
        weight = self.weight
        return weight is not None and self.weights.peek(self.weight_name) is weight and (self.version is None or weight._version == self.version) \
            and (self.derived or self.declared or self.weights.private(self.weight_name))


def _packed_gemm(call, desc):
    """(name suffix, shape, function, geometry, offset) of the copy that a GEMM multiplies by, and the call that does; None where it does not pay."""
    lib = _lib.library()
    offset = call.args[1].offset
    if call.function == "mi355x_gemm_parts_f32":
        parts, M, N, K, a_row, sk, sn = call.args[4:11]
        if a_row % 4 or not lib.mi355x_gemm_parts_packed_pays(parts, M, N, K, int(sk == 1)):
            return None
        copy = (f"{N}_{K}_{sn}_{sk}_{offset}", [-(-N // 32), K // 32, 2, 3, 64, 4], "mi355x_pack_f32", (N, K, sn, sk), offset)
        return copy, (call.function, call.args[:2] + [Ptr("_packed")] + call.args[3:])
    batch0, batch1, M, N, K, a_strides, b_strides = call.args[5:12]
    sb0, sb1, sk, sn = b_strides.values
    if sb0 or sb1 or min(sk, sn) < 1 or a_strides.values[3] != 1 or a_strides.values[2] % 4 \
            or not lib.mi355x_gemm_packed_pays(batch0 * batch1, M, N, K, int(sk == 1)):
        return None
    copy = (f"{N}_{K}_{sn}_{sk}_{offset}", [-(-N // 32), K // 32, 2, 3, 64, 4], "mi355x_pack_f32", (N, K, sn, sk), offset)
    return copy, ("mi355x_gemm_packed_f32", [call.args[0], Ptr("_packed")] + call.args[1:])


def _by_packed_filters(call, constant):
    """(shape, geometry) of the copy that a convolution multiplies by, and the call that does; None where it does not pay."""
    residual = [] if call.function == "mi355x_conv2d_res_f32" else [Ptr(None)]
    args = [call.args[0], Ptr("_packed")] + call.args[1:3] + residual + call.args[3:]
    N, C, H, Wd, M, KH, KW, pads, strides, dilations = args[6:16]
    size = _lib.library().mi355x_conv2d_packed_pays(N, C, H, Wd, M, KH, KW, *(_lib.i64_array(a.values) for a in (pads, strides, dilations)), constant)
    if not size or call.args[1].offset:
        return None
    return [size // 3072, 3, 64, 4], (M, C, KH, KW), ("mi355x_conv2d_packed_f32", args)


def _packed_conv(call, desc):
    """As :func:`_packed_gemm`, for a convolution."""
    packed = _by_packed_filters(call, True)
    if packed is None or desc.shape != packed[1] or not desc.is_contiguous():
        return None
    shape, geometry, packed_call = packed
    return ("filters", shape, "mi355x_pack_conv_f32", geometry, 0), packed_call


def _packed_stem(call, desc):
    """As :func:`_packed_gemm`, for a convolution with its pooling."""
    geometry = call.args[6:16] + call.args[17:22]
    N, C, H, Wd, M, KH, KW = geometry[:7]
    size = _lib.library().mi355x_conv2d_pool_packed_pays(*[_lib.i64_array(a.values) if isinstance(a, I64Array) else a for a in geometry])
    if not size or call.args[1].offset or desc.shape != (M, C, KH, KW) or not desc.is_contiguous():
        return None
    return ("stem_filters", [size // 3072, 3, 64, 4], "mi355x_pack_conv_pool_f32", (M, C, KH, KW), 0), (call.function, call.args[:2] + [Ptr("_packed")] + call.args[3:])


def _packed_filters(call, desc, argument, connector, size, geometry):
    """The packed copy of the filters that ``call`` takes as an argument, and the call that multiplies by it."""
    if call.args[argument].offset or desc.shape != geometry or not desc.is_contiguous():
        return None
    args = call.args[:argument + 1] + [Ptr(connector)] + call.args[argument + 2:]
    return ("filters", [size // 3072, 3, 64, 4], "mi355x_pack_conv_f32", geometry, 0), (call.function, args)


def _packed_block(call, desc):
    C, M = call.args[11], call.args[14]
    return _packed_filters(call, desc, 1, "_packed", -(-M // 32) * -(-C // 16) * 9 * 3072, (M, C, 3, 3))


def _packed_skip(call, desc):
    C, M = call.args[20], call.args[14]
    return _packed_filters(call, desc, 5, "_packed_skip", -(-M // 32) * -(-C // 16) * 3072, (M, C, 1, 1))


def _packed_part(call, desc):
    C, M = call.args[9], call.args[12]
    return _packed_filters(call, desc, 1, "_packed", -(-M // 32) * -(-C // 16) * 9 * 3072, (M, C, 3, 3))


def _shared_by_calls(sdfg, state):
    """The arrays of which a compiled graph keeps one for all of its calls: transients, but for views of an array of the caller's."""
    shared = {name for name, desc in sdfg.arrays.items() if desc.transient}
    views = [{_in_edge(state, n, n.in_conn).data.data, _out_edge(state, n, n.out_conn).data.data} for n in state.nodes() if isinstance(n, AliasNode)]
    for _ in views:   # (a chain of them is no longer than that)
        for view in views:
            if not view <= shared:
                shared -= view
    return shared


def convolutions_in_parts(model):
    """A convolution by constant filters of few tiles and many channels is computed in parts of them, where the library says that this pays; with a
    global pooling that is all that reads it, the launch that adds the parts up takes its means.

    The parts are an array that all calls of the compiled graph share, so that calls on two streams or from two threads must not overlap. A convolution
    from one array of the caller's into another, which they may, stays whole."""
    from ..onnx.onnx_importer import clean_onnx_name
    sdfg, weights, lib = model.sdfg, {clean_onnx_name(k): k for k in model.weights}, _lib.library()
    for state in sdfg.nodes():
        shared = _shared_by_calls(sdfg, state)
        for call in state.nodes():
            if not isinstance(call, KernelCall) or call.function not in ("mi355x_conv2d_f32", "mi355x_conv2d_res_f32"):
                continue
            X, W, bias = call.args[:3]
            residual, Y = call.args[3:5] if call.function == "mi355x_conv2d_res_f32" else (Ptr(None), call.args[3])
            geometry, epilogue = call.args[-12:-2], call.args[-2]
            weight = weights.get(_in_edge(state, call, W.connector).data.data)
            if weight is None or not model.weights.private(weight) or geometry[5:7] != [3, 3] or Y.offset or W.offset:
                continue
            out = _out_edge(state, call, Y.connector)
            if not {_in_edge(state, call, X.connector).data.data, out.data.data} & shared:
                continue
            read = _single_consumer(sdfg, state, out.dst) if isinstance(out.dst, AccessNode) else None
            pool = read and read.dst
            rows, positions = geometry[0] * geometry[4], int(np.prod(sdfg.arrays[out.data.data].shape)) // (geometry[0] * geometry[4])
            mean = isinstance(pool, KernelCall) and pool.function == "mi355x_reduce_mean_f32" and list(pool.args[2:5]) == [rows, positions, 1] and not pool.args[0].offset
            arrays = [_lib.i64_array(a.values) if isinstance(a, I64Array) else a for a in geometry]
            parts = lib.mi355x_conv2d_parts(*arrays, int(mean))
            if parts <= 1:
                continue
            result = _out_edge(state, pool, pool.args[1].connector) if mean else out
            sums = sdfg.free_name(f"{out.data.data}_parts")
            sdfg.add_transient(sums, [parts, rows, positions], float32)
            target = Ptr("_summed", pool.args[1].offset if mean else 0)
            summed = KernelCall(call.label, "mi355x_conv2d_parts_f32", [X, W, Ptr(None), bias, residual, Ptr("_parts"), parts, target] + geometry + [epilogue, int(mean), Stream()],
                                call.in_connectors, ["_parts", "_summed"])
            state.remove_edge(out)
            if mean:
                state.remove_node(pool)
                state.remove_node(out.dst)
                del sdfg.arrays[out.data.data]
            state.replace_node(call, summed, sdfg)
            state.add_edge(summed, "_parts", state.add_access(sums), None, sdfg.make_array_memlet(sums))
            state.add_edge(summed, "_summed", result.dst, None, result.data)


def skip_in_convolutions(model):
    """A convolution by constant filters whose residual is a 1 x 1 convolution by constant filters becomes one call with it, where the library says that
    this pays."""
    from ..onnx.onnx_importer import clean_onnx_name
    sdfg, weights = model.sdfg, {clean_onnx_name(k) for k in model.weights}
    constant = lambda state, call: _in_edge(state, call, call.args[1].connector).data.data in weights   # noqa: E731
    for state in sdfg.nodes():
        for call in state.nodes():
            if not isinstance(call, KernelCall) or call.function != "mi355x_conv2d_res_f32":
                continue
            X, W, bias, residual, Y = call.args[:5]
            epilogue = call.args[15]
            source = _in_edge(state, call, residual.connector).src
            made = _in_edge_of(state, source)
            skip = made and made.src
            if epilogue & ~(_lib.EPI_BIAS | _lib.EPI_RESIDUAL | _lib.EPI_RELU_AFTER) or not epilogue & _lib.EPI_RESIDUAL or residual.offset or Y.offset \
                    or not isinstance(skip, KernelCall) or skip.function != "mi355x_conv2d_f32" or _single_consumer(sdfg, state, source) is None:
                continue
            X2, W2, bias2, Y2 = skip.args[:4]
            N2, C2, H2, Wd2, M2, KH2, KW2, pads2, strides2, _, epilogue2 = skip.args[4:15]
            geometry = call.args[5:15]
            if (N2, M2, KH2, KW2) != (geometry[0], geometry[4], 1, 1) or any(pads2.values) or epilogue2 & ~_lib.EPI_BIAS or Y2.offset or X2.offset \
                    or not constant(state, call) or not constant(state, skip):
                continue
            arrays = [_lib.i64_array(a.values) if isinstance(a, I64Array) else a for a in geometry]
            if not _lib.library().mi355x_conv2d_skip_pays(*arrays, C2, H2, Wd2, _lib.i64_array(strides2.values)):
                continue
            moved = {"_skip_X": X2, "_skip_W": W2}
            if epilogue2 & _lib.EPI_BIAS:
                moved["_skip_B"] = bias2
            edges = {new: _in_edge(state, skip, old.connector) for new, old in moved.items()}
            both = KernelCall(call.label, "mi355x_conv2d_skip_f32",
                              [X, W, Ptr(None), bias, Ptr("_skip_X"), Ptr("_skip_W", W2.offset), Ptr(None), Ptr("_skip_B", bias2.offset) if "_skip_B" in moved else Ptr(None),
                               Ptr("_scratch"), Y] + geometry + [C2, H2, Wd2, strides2, epilogue & ~_lib.EPI_RESIDUAL, Stream()],
                              [c for c in call.in_connectors if c != residual.connector] + list(moved), list(call.out_connectors) + ["_scratch"])
            state.remove_edge(_in_edge(state, call, residual.connector))
            state.remove_node(skip)
            state.replace_node(call, both, sdfg)
            for new, edge in edges.items():
                state.add_edge(edge.src, None, both, new, edge.data)
            state.add_edge(both, "_scratch", source, None, made.data)


def _in_edge_of(state, access):
    edges = state.in_edges(access) if isinstance(access, AccessNode) else []
    return edges[0] if len(edges) == 1 else None


def pool_in_convolutions(model):
    """A convolution by constant filters whose result only a MaxPool reads becomes one call with it, where the library has a kernel for both."""
    from ..onnx.onnx_importer import clean_onnx_name
    sdfg, weights = model.sdfg, {clean_onnx_name(k) for k in model.weights}
    for state in sdfg.nodes():
        for call in state.nodes():
            if not isinstance(call, KernelCall) or call.function != "mi355x_conv2d_f32" or call.args[14] & ~(_lib.EPI_BIAS | _lib.EPI_RELU):
                continue
            X, W, bias, Y = call.args[:4]
            out = _out_edge(state, call, Y.connector)
            read = out and isinstance(out.dst, AccessNode) and _single_consumer(sdfg, state, out.dst)
            pool = read and read.dst
            filters = sdfg.arrays[_in_edge(state, call, W.connector).data.data] if read else None
            if not isinstance(pool, KernelCall) or pool.function != "mi355x_maxpool2d_f32" or pool.args[0].connector != read.dst_conn \
                    or pool.args[0].offset or Y.offset or _in_edge(state, call, W.connector).data.data not in weights:
                continue
            both = KernelCall(call.label, "mi355x_conv2d_pool_packed_f32", [X, W, Ptr(None), bias, Ptr("_scratch"), Ptr("_pooled", pool.args[1].offset)] + call.args[4:15]
                              + pool.args[6:11] + [Stream()], call.in_connectors, ["_scratch", "_pooled"])
            if _packed_stem(both, filters) is None:
                continue
            result = _out_edge(state, pool, pool.args[1].connector)
            state.remove_edge(out)
            state.remove_node(pool)
            state.replace_node(call, both, sdfg)
            state.add_edge(both, "_scratch", out.dst, None, out.data)
            state.add_edge(both, "_pooled", result.dst, None, result.data)


def pack_variable_filters(sdfg):
    """Pack the filters of the remaining convolutions on every call, where the library says that this pays too."""
    for state in sdfg.nodes():
        for call in state.nodes():
            packed = _by_packed_filters(call, False) if isinstance(call, KernelCall) and call.function in ("mi355x_conv2d_f32", "mi355x_conv2d_res_f32") else None
            if packed is None:
                continue
            shape, geometry, (function, args) = packed
            filters = next(e for e in state.in_edges(call) if e.dst_conn == args[2].connector).src
            clean = f"{filters.data}_packed_for_{state.node_id(call)}"
            sdfg.add_transient(clean, shape, int32)
            packed_call = KernelCall(call.label, function, args, list(call.in_connectors) + ["_packed"], list(call.out_connectors))
            state.replace_node(call, packed_call, sdfg)
            pack = KernelCall(f"{call.label}_pack", "mi355x_pack_conv_f32", [Ptr("W"), Ptr("_packed"), *geometry, Stream()], ["W"], ["_packed"])
            access = state.add_access(clean)
            state.add_edge(filters, None, pack, "W", sdfg.make_array_memlet(filters.data))
            state.add_edge(pack, "_packed", access, None, sdfg.make_array_memlet(clean))
            state.add_edge(access, None, packed_call, "_packed", sdfg.make_array_memlet(clean))


# function -> of each operand that may be packed: the argument that is the weight, the name of the packed copy's connector, the function above
_PACKED = {"mi355x_gemm_f32": [(1, "_packed", _packed_gemm)], "mi355x_gemm_parts_f32": [(1, "_packed", _packed_gemm)], "mi355x_conv2d_f32": [(1, "_packed", _packed_conv)],
           "mi355x_conv2d_res_f32": [(1, "_packed", _packed_conv)], "mi355x_conv2d_pool_packed_f32": [(1, "_packed", _packed_stem)],
           "mi355x_conv2d_parts_f32": [(1, "_packed", _packed_part)],
           "mi355x_conv2d_skip_f32": [(1, "_packed", _packed_block), (5, "_packed_skip", _packed_skip)]}


def pack_constant_operands(model):
    """Give every GEMM and convolution of ``model``'s expanded graph that multiplies by a constant, and for which the library says that
    it pays, a packed copy of it. Returns the copies.

    Under a caller's stream capture none is made: its launches are recorded, not run, and the weights that fusion derives hold nothing yet.
    """
    from ..onnx.onnx_importer import clean_onnx_name
    sdfg = model.sdfg
    by_clean = {clean_onnx_name(k): k for k in model.weights}
    copies, now = [], not model._capturing()
    for state in sdfg.nodes():
        written = {e.dst.data for e in state.edges() if isinstance(e.dst, AccessNode)}
        for call in state.nodes():
            if not isinstance(call, KernelCall):
                continue
            for argument, connector, packed_operand in _PACKED.get(call.function, ()):
                call = _pack_operand(model, state, call, by_clean, written, argument, connector, packed_operand, now, copies)
    if copies and now:
        torch.cuda.current_stream().synchronize()   # later calls may come on other streams
    return copies


def _pack_operand(model, state, call, by_clean, written, argument, connector, packed_operand, now, copies):
    """``call``, or what stands in its place and multiplies by a packed copy of its operand; a copy that there was none of yet is added to ``copies``."""
    from ..onnx.onnx_importer import clean_onnx_name
    sdfg = model.sdfg
    edge = next(e for e in state.in_edges(call) if e.dst_conn == call.args[argument].connector)
    if edge.src.data not in by_clean or edge.src.data in written:
        return call
    weight_name = by_clean[edge.src.data]
    desc = sdfg.arrays[edge.src.data]
    if desc.dtype.name != "float32":
        return call
    packed = packed_operand(call, desc)
    if packed is None:
        return call
    (suffix, *copy), (function, args) = packed
    name = f"{weight_name}_packed_{suffix}"
    clean = clean_onnx_name(name)
    if clean not in sdfg.arrays:
        copies.append(PackedOperand(model, weight_name, desc, now, clean, *copy))
        sdfg.add_datadesc(clean, PackedCopy(int32, copies[-1].shape, copies[-1].derived))
        if copies[-1].derived and copies[-1].packed is not None:
            model.weights.make(name, copies[-1].packed, derived=True)
    packed_call = KernelCall(call.label, function, args, list(call.in_connectors) + [connector], list(call.out_connectors))
    state.replace_node(call, packed_call, sdfg)
    state.add_edge(state.add_access(clean), None, packed_call, connector, sdfg.make_array_memlet(clean))
    return packed_call
