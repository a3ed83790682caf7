"""Calls that go through csrc/host_call.cpp, and those that it leaves to the general way: both give what a fresh model gives."""
import threading

import numpy as np
import pytest
import torch

import dace_onnx_amd.onnx as donnx
from dace_onnx_amd.onnx.proto import TensorProto, helper, numpy_helper

pytestmark = pytest.mark.gpu
ROWS, K, N = 64, 96, 127   # (an odd width: fusion derives no copy of the weight)


def _model():
    rng = np.random.default_rng(3)
    info = lambda n, *s: helper.make_tensor_value_info(n, TensorProto.FLOAT, list(s))   # noqa: E731
    nodes = [helper.make_node("MatMul", ["x", "w"], ["y"]), helper.make_node("Softmax", ["y"], ["p"], axis=1), helper.make_node("ReduceMax", ["y"], ["m"], axes=[1], keepdims=0)]
    weights = [numpy_helper.from_array(rng.standard_normal((K, N), dtype=np.float32), "w")]
    graph = helper.make_graph(nodes, "g", [info("x", ROWS, K)], [info("p", ROWS, N), info("m", ROWS)], initializer=weights)
    return donnx.ONNXModel("host_call", helper.make_model(graph, opset_imports=[helper.make_opsetid("", 12)]))


@pytest.fixture
def x():
    return torch.from_numpy(np.random.default_rng(4).standard_normal((ROWS, K), dtype=np.float32)).cuda()


@pytest.fixture
def by_plan(monkeypatch):
    """Whether each call that looked at its plan went by it."""
    seen, call = [], donnx.ONNXModel._call_by_plan

    def recorded(model, args):
        results = call(model, args)
        seen.append(results is not None)
        return results
    monkeypatch.setattr(donnx.ONNXModel, "_call_by_plan", recorded)
    return seen


def same(got, expected):
    return all(torch.equal(g, e) for g, e in zip(got, expected)) and len(got) == len(expected)


def test_plain_calls_go_by_the_plan(x, by_plan):
    model, expected = _model(), _model()(x)
    first = model(x)
    second = model(x)
    assert by_plan == [True] and same(first, expected) and same(second, expected)
    assert second[0].data_ptr() != first[0].data_ptr() and not second[0].requires_grad
    with torch.inference_mode():
        assert same(model(x.clone()), expected)
    assert same(model(torch.nn.Parameter(x)), expected) and by_plan == [True] * 3
    for _, relaunch in model.compile_and_init().bound_launches():   # of the last call, whose tensors are held
        relaunch()
    torch.cuda.synchronize()


class _Sub(torch.Tensor):
    pass


@pytest.mark.parametrize("make, taken", [(lambda x: x.t().contiguous().t(), False), (lambda x: x.cpu(), False), (lambda x: x.cpu().numpy(), False),
                                         (lambda x: x.as_subclass(_Sub), False), (lambda x: torch.stack([x, -x])[0], True)])
def test_arguments_of_other_kinds(x, by_plan, make, taken):
    model, expected = _model(), _model()(x)
    model(x)
    got = model(make(x))
    assert same([torch.as_tensor(g).cuda() for g in got], expected) and by_plan == [taken]
    assert same(model(x=x), expected) and same(model(x), expected) and by_plan == [taken, True]


@pytest.mark.parametrize("make", [lambda x: x.double(), lambda x: x[:32], lambda x: x.reshape(K, ROWS)])
def test_what_was_refused_stays_refused(x, by_plan, make):
    model = _model()
    model(x)
    with pytest.raises(TypeError):
        model(make(x))
    with pytest.raises(TypeError):
        model()
    with pytest.raises(TypeError):
        model(x, x)
    model.weights["unknown"] = x
    with pytest.raises(TypeError):
        model(x)
    assert not any(by_plan)


def test_weights_that_are_written_replaced_or_taken_out(x, by_plan):
    model = _model()
    model(x)
    expected = x.double() @ model.weights["w"].double()
    largest = lambda: model(x)[1].double()   # noqa: E731
    bound = (x.double().abs() @ model.weights["w"].double().abs()).amax(1) * (K + 8) * 2.0**-23
    assert bool(((largest() - expected.amax(1)).abs() <= bound).all())
    with torch.no_grad():
        model.weights["w"].mul_(-2)
    assert bool(((largest() - (-2 * expected).amax(1)).abs() <= 2 * bound).all())
    model.weights["w"].data.mul_(-1)
    assert bool(((largest() - (2 * expected).amax(1)).abs() <= 2 * bound).all())
    model.weights["w"] = model.weights["w"] * 0.5
    assert bool(((largest() - expected.amax(1)).abs() <= bound).all()) and all(by_plan)
    model.weights["w"] = model.weights["w"].double()
    with pytest.raises(TypeError):
        model(x)
    assert not by_plan[-1]


def test_streams_threads_and_recordings(x, by_plan):
    model, expected = _model(), _model()(x)
    model(x)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        got = model(x)
    stream.synchronize()
    assert same(got, expected)
    results = {}

    def work(i):
        for _ in range(20):   # (with one input: calls that overlap write the same into the intermediate array that they share)
            results[i] = model(x)

    threads = [threading.Thread(target=work, args=(i, )) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert all(same(r, expected) for r in results.values()) and all(by_plan)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        recorded = model(x)
    assert not by_plan[-1]
    for _ in range(3):
        for r in recorded:
            r.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.allclose(r, e, rtol=1e-5, atol=1e-6) for r, e in zip(recorded, expected))


def _tail():
    return [helper.make_node("Softmax", ["y"], ["p"], axis=1), helper.make_node("ReduceMax", ["y"], ["m"], axes=[1], keepdims=0)], {"y": [4096, N]}, {"p": [4096, N], "m": [4096]}, []


def _convolution():
    w = numpy_helper.from_array(np.random.default_rng(2).standard_normal((512, 512, 3, 3), dtype=np.float32), "w")
    nodes = [helper.make_node("Conv", ["y", "w"], ["c"], kernel_shape=[3, 3], pads=[1] * 4), helper.make_node("Relu", ["c"], ["p"])]
    return nodes, {"y": [1, 512, 7, 7]}, {"p": [1, 512, 7, 7]}, [w]


@pytest.mark.parametrize("make", [_tail, _convolution])
@pytest.mark.parametrize("shared_stream", [True, False])
def test_calls_of_a_model_without_intermediate_arrays_may_overlap(by_plan, make, shared_stream):
    """From four threads, each with its inputs: on one stream, where their launches come in any order, and on a stream each."""
    nodes, inputs, outputs, weights = make()
    infos = lambda of: [helper.make_tensor_value_info(n, TensorProto.FLOAT, s) for n, s in of.items()]   # noqa: E731
    graph = helper.make_graph(nodes, "g", infos(inputs), infos(outputs), initializer=weights)
    model = donnx.ONNXModel("overlap", helper.make_model(graph, opset_imports=[helper.make_opsetid("", 12)]))
    xs = [torch.from_numpy(np.random.default_rng(i).standard_normal(inputs["y"], dtype=np.float32)).cuda() for i in range(4)]
    call = lambda x: r if isinstance(r := model(x), tuple) else (r, )   # noqa: E731
    expected, results = [call(x) for x in xs], {}
    assert not any(d.transient for d in model.sdfg.arrays.values())
    torch.cuda.synchronize()

    def work(i):
        stream = torch.cuda.current_stream() if shared_stream else torch.cuda.Stream()
        with torch.cuda.stream(stream):
            results[i] = [call(xs[i]) for _ in range(20)]
        stream.synchronize()

    threads = [threading.Thread(target=work, args=(i, )) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(results) == 4 and all(same(r, expected[i]) for i in range(4) for r in results[i])
    assert by_plan == [True] * 83


def test_nothing_outlives_a_dropped_model(x):
    import gc
    gc.collect()
    before = torch.cuda.memory_allocated()
    for _ in range(3):
        model = _model()
        for _ in range(3):
            model(x)
        model.compile_and_init().bound_launches()
        del model
        gc.collect()
    assert torch.cuda.memory_allocated() <= before + 4096   # (the two tensors of _example, once)
