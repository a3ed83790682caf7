"""What goes into one launch with a Softmax along the last axis: a ReduceMax of the same input, which it knows anyway, and the product whose
rows it normalizes, where these are a few values each.

The reference has no counterpart: each is a map of its own there (pure_implementations.py:130-267, 316-366).
"""
from .. import _lib
from ..sdfg import KernelCall, Ptr, Stream
from .fusion import _in_edge, _out_edge, _single_consumer


def softmax_of_products(model):
    """A product of few columns whose rows a Softmax normalizes, and nobody else reads, becomes one call with it; returns how many."""
    from ..onnx.onnx_importer import clean_onnx_name
    sdfg, lib, count = model.sdfg, _lib.library(), 0
    for state in sdfg.nodes():
        for softmax in state.nodes():
            if not isinstance(softmax, KernelCall) or softmax.function != "mi355x_softmax_f32" or softmax.args[4] != 1 or softmax.args[0].offset:
                continue
            M, N = softmax.args[2:4]
            source = _in_edge(state, softmax, softmax.args[0].connector).src
            made = state.in_edges(source)
            call = made[0].src if len(made) == 1 else None
            if not isinstance(call, KernelCall) or call.function != "mi355x_gemm_f32" or _single_consumer(sdfg, state, source) is None:
                continue
            A, B, C, bias, _, batch0, batch1, rows, columns, K, a_strides, b_strides, c_strides, _, alpha, epilogue = call.args[:16]
            b_k, b_column = b_strides.values[2:4]
            if batch0 * batch1 != 1 or (rows, columns) != (M, N) or epilogue & _lib.EPI_RESIDUAL or a_strides.values[3] != 1 or c_strides.values[2] != N or C.offset \
                    or not lib.mi355x_gemm_softmax_pays(M, N, K, int(b_k == 1)):
                continue
            weight = {clean_onnx_name(k): k for k in model.weights}.get(_in_edge(state, call, B.connector).data.data)
            if weight is not None and model.weights.private(weight) and lib.mi355x_gemm_packed_pays(1, M, N, K, 1):
                continue   # (the packed kernel's sums have half the error)
            result = _out_edge(state, softmax, softmax.args[1].connector)
            both = KernelCall(call.label, "mi355x_gemm_softmax_f32", [A, B, bias if epilogue & _lib.EPI_BIAS else Ptr(None), Ptr("_scratch"),
                                                                      Ptr("_probabilities", softmax.args[1].offset), M, N, K, a_strides.values[2], b_k, b_column, alpha, epilogue,
                                                                      Stream()], call.in_connectors, ["_scratch", "_probabilities"])
            state.remove_edge(made[0])
            state.remove_node(softmax)
            state.replace_node(call, both, sdfg)
            state.add_edge(both, "_scratch", source, None, made[0].data)
            state.add_edge(both, "_probabilities", result.dst, None, result.data)
            count += 1
    return count


def softmax_with_maxima(sdfg):
    """Replace every such pair of launches of an expanded graph; returns how many.

    All of them: over 103 sizes of 16 to 400000 rows of 1 to 30522 values the launch takes 0.07 to 0.75 of the time of the two ([65536, 33] 17.7 -> 10.8 us, [4096, 2048]
    13.3 -> 10.0), and beyond 32768 the function makes two launches itself.
    """
    count = 0
    for state in sdfg.nodes():
        calls = [n for n in state.nodes() if isinstance(n, KernelCall)]
        maxima = [c for c in calls if c.function == "mi355x_reduce_f32" and c.args[0] == _lib.REDUCE_MAX and c.args[5] == 1]
        for softmax in calls:
            if softmax.function != "mi355x_softmax_f32" or softmax.args[4] != 1:
                continue
            X, Y, rows, cols = softmax.args[:4]
            read = _in_edge(state, softmax, X.connector)
            reduce = next((c for c in maxima if list(c.args[3:5]) == [rows, cols] and _in_edge(state, c, c.args[1].connector).src is read.src
                           and c.args[1].offset == X.offset), None)
            if reduce is None:
                continue
            maxima.remove(reduce)
            largest = _out_edge(state, reduce, reduce.args[2].connector)
            both = KernelCall(softmax.label, "mi355x_softmax_max_f32", [X, Y, Ptr("_largest", reduce.args[2].offset), rows, cols, Stream()], softmax.in_connectors,
                              list(softmax.out_connectors) + ["_largest"])
            state.remove_node(reduce)
            state.replace_node(softmax, both, sdfg)
            state.add_edge(both, "_largest", largest.dst, None, largest.data)
            count += 1
    return count
