"""Several launches as one call into the library: what of it runs without a GPU (calls over no data, refusals)."""
import array

import pytest
import torch

from dace_onnx_amd import _lib
from dace_onnx_amd import sdfg as dace


def run(calls, patches=(), addresses=(), words=None, behind=()):
    """``calls``: (function, arguments but the stream)."""
    lib = _lib.library()
    program = array.array("q", [w for name, *args in calls for w in [lib.mi355x_program_function(name.encode()), *args]] + list(behind))
    moved, sources = array.array("q", [v for p in patches for v in p]), array.array("q", addresses)
    pointer = lambda a: a.buffer_info()[0]  # noqa: E731
    return lib.mi355x_program_run(pointer(program), len(program) if words is None else words, len(calls), pointer(moved), len(patches), pointer(sources), None)


EMPTY = ("mi355x_softmax_f32", 0, 0, 0, 5, 1)        # no rows
BAD = ("mi355x_softmax_f32", 0, 0, -1, 5, 1)


def test_every_function_that_takes_a_stream_last_has_a_number():
    lib = _lib.library()
    callable_ = [n for n, (_, types) in _lib.SIGNATURES.items() if len(types) > 4 and types[-1] is _lib._vp and not n.startswith(("mi355x_pack_f32", "mi355x_program"))]
    assert len(callable_) > 15 and sorted({lib.mi355x_program_function(n.encode()) for n in callable_}) == list(range(len(callable_)))
    assert lib.mi355x_program_function(b"mi355x_version") == lib.mi355x_program_function(b"") == -1


def test_calls_run_in_order_and_the_first_that_fails_ends_the_program():
    assert run([]) == run([EMPTY]) == run([EMPTY, EMPTY]) == 0
    assert run([EMPTY, BAD, BAD]) == 1 << 8 | 1 and b"softmax" in _lib.library().mi355x_last_error()
    assert run([EMPTY] * 700) == 0 and run([EMPTY] * 700 + [BAD]) == 700 << 8 | 1   # (a program of more words than the stack holds)


def test_addresses_take_their_place():
    # the number of rows (word 3) is written by a patch: none, and -1
    assert run([BAD], [(3, 0, 1)], [-1]) == 0 and run([EMPTY], [(3, 1, -9)], [0, 8]) == 1
    # strides of a pointer array behind the calls
    lib = _lib.library()
    shape = ("mi355x_permute_b32", 0, 0, 2, 0, 0)
    assert run([shape], [(4, -1, 6), (5, -1, 8)], (), None, [0, 3, 1, 1]) == lib.mi355x_permute_b32(None, None, 2, _lib.i64_array([0, 3]), _lib.i64_array([1, 1]), None) == 0


@pytest.mark.parametrize("arguments", [dict(calls=[EMPTY], words=5), dict(calls=[EMPTY, EMPTY], words=6), dict(calls=[("no_such_function", 0)]),
                                       dict(calls=[EMPTY], patches=[(6, 0, 0)], addresses=[0]), dict(calls=[EMPTY], patches=[(-1, 0, 0)], addresses=[0]),
                                       dict(calls=[EMPTY], patches=[(1, -1, 6)]), dict(calls=[EMPTY], words=-1)])
def test_what_is_no_program_is_refused(arguments):
    assert run(**arguments) & 0xff == 1


def packing_sdfg(rows=40, k=64):
    """A launch that cannot be part of a program, and one that can."""
    sdfg = dace.SDFG("packing")
    state = sdfg.add_state()
    sdfg.add_array("w", [rows, k], dace.float32)
    sdfg.add_array("largest", [rows], dace.float32)
    sdfg.add_array("packed", [-(-rows // 32), k // 32, 2, 3, 64, 4], dace.int32)
    pack = dace.KernelCall("pack", "mi355x_pack_f32", [dace.Ptr("w"), dace.Ptr("p"), rows, k, k, 1, dace.Stream()], ["w"], ["p"])
    top = dace.KernelCall("largest", "mi355x_reduce_f32", [2, dace.Ptr("w"), dace.Ptr("y"), rows, k, 1, dace.Stream()], ["w"], ["y"])
    empty = dace.KernelCall("empty", "mi355x_launch_empty_kernel", [dace.Stream()], [], [])
    w = state.add_read("w")
    for call, conn, name in ((pack, "p", "packed"), (top, "y", "largest")):
        state.add_edge(w, None, call, "w", sdfg.make_array_memlet("w"))
        state.add_edge(call, conn, state.add_write(name), None, sdfg.make_array_memlet(name))
    state.add_node(empty)
    return sdfg


def test_functions_that_are_no_part_of_a_program_are_called_one_at_a_time(monkeypatch):
    compiled = packing_sdfg().compile()
    compiled.device = torch.device("cpu")
    runs = []
    monkeypatch.setattr(compiled, "_run", runs.append)
    buffers = lambda: {k: torch.zeros(compiled.sdfg.arrays[k].shape, dtype=compiled._torch_types[k]) for k in compiled._external}  # noqa: E731
    first, second = buffers(), buffers()
    for arguments in (first, first, second):
        compiled(**arguments)
    assert compiled._program is None and len(runs) == 3 and runs[0] is runs[1]
    for launches, arguments in zip(runs[1:], (first, second)):
        args = {item[2]: item[3] for item in launches}
        assert sorted(args) == ["mi355x_launch_empty_kernel", "mi355x_pack_f32", "mi355x_reduce_f32"]
        w, packed, largest = (arguments[k].data_ptr() for k in ("w", "packed", "largest"))
        assert args["mi355x_pack_f32"][:2] == [w, packed] and args["mi355x_reduce_f32"][1:3] == [w, largest]


@pytest.mark.gpu
def test_functions_that_are_no_part_of_a_program_run():
    compiled = packing_sdfg().compile()
    for _ in range(2):
        w = torch.randn(40, 64, device="cuda")
        packed, largest = torch.zeros(2, 2, 2, 3, 64, 4, dtype=torch.int32, device="cuda"), torch.zeros(40, device="cuda")
        compiled(w=w, packed=packed, largest=largest)
        parts = packed.cpu().view(torch.bfloat16).reshape(2, 2, 2, 3, 2, 32, 2, 4).double().sum(3)   # block, step, s, h, row, a, e
        assert torch.equal(parts.permute(0, 4, 1, 5, 2, 3, 6).reshape(64, 64)[:40] / 65536, w.cpu().double())
        assert torch.equal(largest.cpu(), w.cpu().amax(1))
