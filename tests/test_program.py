"""Several launches as one call into the library: what of it runs without a GPU (calls over no data, refusals)."""
import array

import pytest

from dace_onnx_amd import _lib


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
