"""Products of few output tiles in parts of K, added up by the LayerNormalization that follows.

A projection back to the hidden size has few outputs and a long K (16 x 768 x 3072: 48 tiles for 256 CUs). Its product is computed as several
sums over shares of K, by as many times the workgroups, and the normalization, which reads every value anyway, adds them, the bias and the
residual up: no launch, synchronisation or atomic more. The library says for which sizes this pays. The reference has no counterpart.
"""
from .. import _lib
from ..sdfg import AccessNode, KernelCall, Ptr, Stream, float32
from .fusion import _in_edge, _out_edge, _single_consumer


def _normalization_of(sdfg, state, call):
    """The normalization of the rows that ``call``, a GEMM with at most a bias and a residual, computes, if nobody else reads them."""
    batch0, batch1, M, N, _, a_strides, b_strides, c_strides = call.args[5:13]
    epilogue = call.args[15]
    out = _out_edge(state, call, call.args[2].connector)
    if batch0 * batch1 != 1 or epilogue & ~(_lib.EPI_BIAS | _lib.EPI_RESIDUAL) or a_strides.values[3] != 1 or min(b_strides.values[2:4]) < 1 \
            or c_strides.values[2] != N or call.args[2].offset or out is None or not isinstance(out.dst, AccessNode):
        return None
    read = _single_consumer(sdfg, state, out.dst)
    norm = read and read.dst
    if not isinstance(norm, KernelCall) or norm.function != "mi355x_layernorm_f32" or norm.args[0].connector != read.dst_conn \
            or norm.args[0].offset or list(norm.args[4:6]) != [M, N]:
        return None
    return norm


def split_products(model):
    """Replace every such pair of launches of ``model``'s expanded graph where the library says that parts pay; returns how many."""
    from ..onnx.onnx_importer import clean_onnx_name
    sdfg, lib, count = model.sdfg, _lib.library(), 0
    weights = {clean_onnx_name(k): k for k in model.weights}
    for state in sdfg.nodes():
        for call in state.nodes():
            norm = _normalization_of(sdfg, state, call) if isinstance(call, KernelCall) and call.function == "mi355x_gemm_f32" else None
            if norm is None:
                continue
            A, B, C, bias, residual = call.args[:5]
            M, N, K, a_strides, b_strides = call.args[7:12]
            b_k, b_column = b_strides.values[2:4]
            weight = weights.get(_in_edge(state, call, B.connector).data.data)
            parts = lib.mi355x_gemm_parts(M, N, K, int(b_k == 1), int(weight is not None and model.weights.private(weight)))
            if parts <= 1:
                continue
            sums = sdfg.free_name(f"{_out_edge(state, call, C.connector).data.data}_parts")
            sdfg.add_transient(sums, [parts, M, N], float32)
            product = KernelCall(call.label, "mi355x_gemm_parts_f32", [A, B, Ptr(None), Ptr("_parts", C.offset), parts, M, N, K, a_strides.values[2], b_k, b_column,
                                                                       call.args[14], Stream()], [A.connector, B.connector], ["_parts"])
            epilogue = call.args[15]
            # (connectors of the two calls may have the same names)
            moved = {"_bias": bias if epilogue & _lib.EPI_BIAS else Ptr(None), "_residual": residual if epilogue & _lib.EPI_RESIDUAL else Ptr(None)}
            moved = {new: old for new, old in moved.items() if old.connector is not None}
            gamma, beta, Y = norm.args[1:4]
            add = lambda name: Ptr(name, moved[name].offset) if name in moved else Ptr(None)   # noqa: E731
            inputs = ["_parts", gamma.connector] + ([beta.connector] if beta.connector is not None else []) + list(moved)
            result = KernelCall(norm.label, "mi355x_layernorm_parts_f32", [Ptr("_parts"), parts, add("_bias"), add("_residual"), call.args[13].values[2] if "_residual" in moved
                                                                           else N, gamma, beta, Y, M, N, norm.args[6], Stream()], inputs, [Y.connector])
            sources = {new: _in_edge(state, call, old.connector) for new, old in moved.items()}
            intermediate = _out_edge(state, call, C.connector).dst
            state.remove_node(intermediate)
            state.replace_node(norm, result, sdfg)
            for new, edge in sources.items():
                state.add_edge(edge.src, None, result, new, edge.data)
            state.replace_node(call, product, sdfg)
            access = state.add_access(sums)
            state.add_edge(product, "_parts", access, None, sdfg.make_array_memlet(sums))
            state.add_edge(access, None, result, "_parts", sdfg.make_array_memlet(sums))
            del sdfg.arrays[intermediate.data]
            count += 1
    return count
