"""A Softmax and a ReduceMax along the last axis of the same input in one launch: the first knows the largest value of every row anyway.

The reference has no counterpart: each is a map of its own there (pure_implementations.py:316-366).
"""
from .. import _lib
from ..sdfg import KernelCall, Ptr, Stream
from .fusion import _in_edge, _out_edge


def softmax_with_maxima(sdfg):
    """Replace every such pair of launches of an expanded graph; returns how many."""
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
