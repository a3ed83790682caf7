"""Constant operands of contractions, packed for the kernels of ``csrc/gemm_f32_packed.hip`` when a graph is compiled.

A packed copy holds three bf16 parts of every value in the order in which the matrix unit takes them (``csrc/split_bf16.h``); it is
made once, on the GPU, and is a further weight of the model. The reference has no counterpart: its constants are handed to a BLAS
library as they are.
"""
import torch

from .. import _lib
from ..sdfg import AccessNode, KernelCall, Ptr, int32


class PackedOperand:
    """A packed copy of ``rows`` x ``k`` values of a weight, at element strides ``row_stride`` and ``k_stride`` from ``offset``."""

    def __init__(self, model, weight_name, rows, k, row_stride, k_stride, offset):
        self.model, self.weight_name = model, weight_name
        self.geometry = (rows, k, row_stride, k_stride)
        self.offset = offset
        self.packed = torch.empty([-(-rows // 32), k // 32, 2, 3, 64, 4], dtype=torch.int32, device=model.weights[weight_name].device)
        self.pack()

    def pack(self):
        self.weight = self.model.weights[self.weight_name]
        self.version = self.weight._version
        start = self.weight.data_ptr() + 4 * self.offset
        _lib.check(_lib.library().mi355x_pack_f32(start, self.packed.data_ptr(), *self.geometry, _lib.current_stream()), "mi355x_pack_f32")

    def refresh(self):
        """Pack again if the weight was replaced or written in place since (a wrapped module whose parameters were updated)."""
        weight = self.model.weights[self.weight_name]
        if weight is not self.weight or weight._version != self.version:
            self.pack()


def pack_constant_operands(model):
    """Give every GEMM of ``model``'s expanded graph that multiplies by a constant, and for which the library says that it pays, a
    packed copy of it. Returns the copies."""
    from ..onnx.onnx_importer import clean_onnx_name
    sdfg, lib = model.sdfg, _lib.library()
    by_clean = {clean_onnx_name(k): k for k in model.weights}
    copies = []
    for state in sdfg.nodes():
        written = {e.dst.data for e in state.edges() if isinstance(e.dst, AccessNode)}
        for call in state.nodes():
            if not isinstance(call, KernelCall) or call.function != "mi355x_gemm_f32":
                continue
            b = call.args[1]
            edge = next(e for e in state.in_edges(call) if e.dst_conn == b.connector)
            batch0, batch1, M, N, K, a_strides, b_strides = call.args[5:12]
            sb0, sb1, sk, sn = b_strides.values
            if edge.src.data not in by_clean or edge.src.data in written or sb0 or sb1 or min(sk, sn) < 1:
                continue
            weight_name = by_clean[edge.src.data]
            if model.weights[weight_name].dtype != torch.float32 or a_strides.values[3] != 1 or a_strides.values[2] % 4 \
                    or not lib.mi355x_gemm_packed_pays(batch0 * batch1, M, N, K, int(sk == 1)):
                continue
            name = f"{weight_name}_packed_{N}_{K}_{sn}_{sk}_{b.offset}"
            clean = clean_onnx_name(name)
            if name not in model.weights:
                copies.append(PackedOperand(model, weight_name, N, K, sn, sk, b.offset))
                model.weights[name] = copies[-1].packed
                sdfg.add_array(clean, list(copies[-1].packed.shape), int32, transient=False)
            args = [call.args[0], Ptr("_packed")] + call.args[1:]
            packed_call = KernelCall(call.label, "mi355x_gemm_packed_f32", args, list(call.in_connectors) + ["_packed"], list(call.out_connectors))
            state.replace_node(call, packed_call, sdfg)
            state.add_edge(state.add_access(clean), None, packed_call, "_packed", sdfg.make_array_memlet(clean))
    if copies:
        torch.cuda.current_stream().synchronize()   # later calls may come on other streams
    return copies
