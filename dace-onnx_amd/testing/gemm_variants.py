"""The fp32 GEMM (activations x weights, bias epilogue) through the library's own choice and through each forced form of its
kernels, over a set of shapes.

    python -m dace_onnx_amd.testing.gemm_variants            # the four launches of the BERT-base layer and shapes around them
    python -m dace_onnx_amd.testing.gemm_variants rounds     # 3072-wide outputs of 512 to 3328 tiles of 128 x 48, K = 768 .. 4096
    python -m dace_onnx_amd.testing.gemm_variants few        # outputs of few tiles, and 160 random products and stacks
    python -m dace_onnx_amd.testing.gemm_variants split      # outputs of many tiles, and 160 random products and stacks
    python -m dace_onnx_amd.testing.gemm_variants packed     # by packed weights: the layer's products at 16 to 8192 rows, and 160 random ones

Prints microseconds per launch (HIP events around graph-recorded launches after a warm-up by time, as bench.py measures
its rows), the best of the forced forms and the ratio of the library's choice to it. The forms (``MI355X_GEMM_NT_*``):

* ``48 deep`` / ``48 lean``: 64 x 48 tiles by eight waves, 64-k tiles three deep / 32-k tiles three deep (three workgroups per CU);
* ``48 w16``: 64 x 48 tiles by 16 waves in four k-split groups (where K is a multiple of 64);
* ``64`` / ``96`` / ``144``: 64 x 64, 128 x 96 (16 waves) and 64 x 144 tiles;
* ``128 deep`` / ``128 lean``: 128 x 48 tiles with the six-deep ring (two workgroups per CU) / the three-deep one (three).

``few`` and ``split`` take weights [N, K] (``kc``) and [K, N] (``nc``), ``few`` and ``packed`` weights that are not in the L2 (they rotate through
64 MB of them). Their forms: ``lds``, never the few-tile kernel (``MI355X_GEMM_DIRECT=0``), and its tiles (``=11`` ...); ``fp32``, neither
that nor the bf16 kernel (``MI355X_GEMM_SPLIT=0``), and the latter's tiles (``=64`` ...). ``packed``: ``before``, without the packed copy
(``MI355X_GEMM_PACKED=0``), and the forms of the packed kernel by number, as in its table (``=1`` ...).

Every form is checked against float64 in tests/test_configs_gpu.py::test_k_contiguous_gemm_tiles_and_epilogues and
tests/test_kernel_edges_gpu.py.
"""
import itertools
import math
import os
import random
import sys

from .. import _lib
from .profiling import graph_time_us

VARIABLES = ("MI355X_GEMM_NT_BM", "MI355X_GEMM_NT_BN", "MI355X_GEMM_NT_PER_CU", "MI355X_GEMM_NT_WAVES", "MI355X_GEMM_NT_BK", "MI355X_GEMM_DIRECT",
             "MI355X_GEMM_SPLIT", "MI355X_GEMM_PACKED")
FORMS = (("library", {}),
         ("48 deep", {"MI355X_GEMM_NT_BN": "48", "MI355X_GEMM_NT_PER_CU": "2", "MI355X_GEMM_NT_WAVES": "8"}),
         ("48 lean", {"MI355X_GEMM_NT_BN": "48", "MI355X_GEMM_NT_PER_CU": "3", "MI355X_GEMM_NT_WAVES": "8"}),
         ("48 w16", {"MI355X_GEMM_NT_BN": "48", "MI355X_GEMM_NT_WAVES": "16"}),
         ("64", {"MI355X_GEMM_NT_BN": "64"}), ("96", {"MI355X_GEMM_NT_BN": "96"}), ("144", {"MI355X_GEMM_NT_BN": "144"}),
         ("128 deep", {"MI355X_GEMM_NT_BM": "128", "MI355X_GEMM_NT_BN": "48", "MI355X_GEMM_NT_PER_CU": "2"}),
         ("128 lean", {"MI355X_GEMM_NT_BM": "128", "MI355X_GEMM_NT_BN": "48", "MI355X_GEMM_NT_PER_CU": "3"}))


FEW = (("library", {}), ("lds", {"MI355X_GEMM_DIRECT": "0"}))
FEW_TILES = {True: (("16x16", "11"), ("16x32", "12"), ("32x32", "22")), False: (("16x64", "14"), ("32x64", "24"))}
SPLIT = (("library", {}), ("fp32", {"MI355X_GEMM_DIRECT": "0", "MI355X_GEMM_SPLIT": "0"})) + tuple(
    (name, {"MI355X_GEMM_DIRECT": "0", "MI355X_GEMM_SPLIT": rows}) for name, rows in (("64x64", "64"), ("128x64", "128"), ("256x128", "256")))


def shapes(which: str):
    if which == "rounds":
        return [(128 * m, 3072, K) for K in (768, 1536, 2048, 3072, 4096) for m in (8, 12, 14, 16, 18, 20, 24, 28, 32, 36, 40, 52)]
    out = []
    for K in (256, 768, 1536, 3072):
        for M, N in ((128, 768), (512, 768), (1024, 768), (1024, 1024), (512, 3072), (1024, 1536), (384, 4096), (2048, 768),
                     (1536, 1152), (1024, 2304), (1024, 3072), (2048, 2304), (4096, 1024), (4096, 4096)):
            out.append((M, N, K))
    return out


def random_shapes(which: str, count: int):
    """(batch, M, N, K, kc), extents spread over their logarithm."""
    rng = random.Random(which)
    log_int = lambda low, high: min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))   # noqa: E731
    while count:
        batch, kc = rng.choice((1, 1, 1, 8, 48, 200)), rng.random() < 0.5
        if which == "few":
            M, N, K, step = log_int(1, 4096), log_int(4, 8192), log_int(4, 4096), 32
            work = batch * -(-M // 16) * -(-N // 32) * (1 + K / 512) / 256
        else:
            M, N, K, step = log_int(16, 8192), log_int(16, 8192), 32 * log_int(4, 100), 64
            work = batch * -(-M // 64) * -(-N // 64) / 10 / 256
        if rng.random() < 0.5:
            N, K = max(step, N // step * step), max(32, K // 32 * 32)
        if work <= (300 if which == "few" else 4) and batch * max(M * N, M * K, N * K) < 2e8:
            count -= 1
            yield batch, M, N, K, kc


def few_and_split(which: str):
    import torch
    lib = _lib.library()
    if which == "few":
        fixed = [(1, M, N, K, True) for M in (1, 16, 40, 128, 256, 512) for N, K in ((768, 768), (2304, 768), (3072, 768), (768, 3072))]
        fixed += [(1, M, 30522, 768, False) for M in (1, 16, 64)] + [(1, 5, 300, 784, True), (1, 5, 10, 300, True), (1, 33, 1000, 1503, True)]
    else:
        fixed = [(1, M, N, K, kc) for kc in (True, False) for M in (512, 1024, 2048, 4096, 8192) for N, K in ((768, 768), (2304, 768), (3072, 768), (768, 3072))]
        fixed += [(1, 1024, 30522, 768, False), (1, 4096, 4096, 4096, True)]
    behind = []
    for batch, M, N, K, kc in itertools.chain(fixed, random_shapes(which, 160)):
        forms = SPLIT if which == "split" else FEW + tuple((name, {"MI355X_GEMM_DIRECT": form}) for name, form in FEW_TILES[kc])
        copies = max(1, min(20, int(64e6 / (4 * batch * N * K)))) if which == "few" else 1
        a, w = torch.randn(batch, M, K, device="cuda"), [torch.randn(batch * N * K, device="cuda") * 0.05 for _ in range(copies)]
        bias, out = torch.randn(N, device="cuda"), torch.empty(batch, M, N, device="cuda")
        i64, weights = _lib.i64_array, itertools.cycle(w)
        launch = lambda: lib.mi355x_gemm_f32(a.data_ptr(), next(weights).data_ptr(), out.data_ptr(), bias.data_ptr(), None, 1, batch, M, N, K,   # noqa: E731
                                             i64([0, M * K, K, 1]), i64([0, N * K, 1, K] if kc else [0, N * K, N, 1]), i64([0, M * N, N]),
                                             None, 1.0, _lib.EPI_BIAS, _lib.current_stream())
        times = []
        for _, variables in forms:
            for name in VARIABLES:
                os.environ.pop(name, None)
            os.environ.update(variables)
            lib.mi355x_reload_tuning()
            times.append(min(graph_time_us(launch, reps=20, warm_ms=20.0) for _ in range(2)))
        behind.append((times[0] / times[1], times[0] / min(times[1:])))
        print(f"{batch:4d} x {M:5d} x {N:5d} x {K:5d} {'kc' if kc else 'nc'} " + " ".join(f"{name} {t:9.2f}" for (name, _), t in zip(forms, times)) +
              f"   library / {forms[1][0]} {behind[-1][0]:.3f}, / best {behind[-1][1]:.3f}", flush=True)
    print(f"{len(behind)} shapes: library / {forms[1][0]} at most {max(b for b, _ in behind):.3f}, above 1.03 in {sum(b > 1.03 for b, _ in behind)}; "
          f"library / best form {sum(b for _, b in behind) / len(behind):.3f} on average, at most {max(b for _, b in behind):.3f}")


def set_variables(variables):
    for name in VARIABLES:
        os.environ.pop(name, None)
    os.environ.update(variables)
    _lib.library().mi355x_reload_tuning()


def packed():
    import torch
    lib, i64, rng = _lib.library(), _lib.i64_array, random.Random("packed")
    log_int = lambda low, high: min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))   # noqa: E731
    shapes = [(M, N, K, True) for M in (16, 128, 865, 1024, 2048, 8192) for N, K in ((768, 768), (2304, 768), (3072, 768), (768, 3072))]
    shapes += [(1024, 30522, 768, False), (1500, 1024, 4096, True), (373, 1024, 256, True)]
    while len(shapes) < 27 + 160:
        M, N, K = log_int(8, 16384), log_int(64, 32000), 32 * log_int(2, 128)
        if M * N * K < 2e11:
            shapes.append((M, N // 32 * 32 if rng.random() < 0.5 else N, K, rng.random() < 0.5))
    forms = (("library", {}), ("before", {"MI355X_GEMM_PACKED": "0"})) + tuple((str(f), {"MI355X_GEMM_PACKED": str(f)}) for f in range(1, 11))
    ratios = []
    for M, N, K, kc in shapes:
        a, bias, out = (torch.randn(s, device="cuda") for s in ((M, K), (N, ), (M, N)))
        operands = []
        for _ in range(max(1, min(20, int(64e6 / (4 * N * K))))):
            w, copy = torch.randn((N, K) if kc else (K, N), device="cuda"), torch.empty(-(-N // 32) * (K // 32) * 1536, dtype=torch.int32, device="cuda")
            _lib.check(lib.mi355x_pack_f32(w.data_ptr(), copy.data_ptr(), N, K, *((K, 1) if kc else (1, N)), _lib.current_stream()), "pack")
            operands.append((w, copy))
        turns = itertools.cycle(operands)

        def launch():
            w, copy = next(turns)
            return lib.mi355x_gemm_packed_f32(a.data_ptr(), copy.data_ptr(), w.data_ptr(), out.data_ptr(), bias.data_ptr(), None, 1, 1, M, N, K,
                                              i64([0, M * K, K, 1]), i64([0, 0, 1, K] if kc else [0, 0, N, 1]), i64([0, M * N, N]), None, 1.0,
                                              _lib.EPI_BIAS, _lib.current_stream())

        times = []
        for _, variables in forms:
            set_variables(variables)
            times.append(min(graph_time_us(launch, reps=20, replays=3, warm_ms=10.0) for _ in range(2)))
        set_variables({})
        ratios.append((times[0] / times[1], times[0] / min(times[1:])))
        print(f"{M:5d} x {N:5d} x {K:4d} {'kc' if kc else 'nc'} {'packed' if lib.mi355x_gemm_packed_pays(1, M, N, K, int(kc)) else 'before':6s} " +
              " ".join(f"{name} {t:.1f}" for (name, _), t in zip(forms, times)) +
              f"   library / before {ratios[-1][0]:.3f}, / best {ratios[-1][1]:.3f}", flush=True)
    for name, column in (("before", 0), ("best form", 1)):
        r = [x[column] for x in ratios]
        print(f"{len(r)} products: library / {name} {math.exp(sum(map(math.log, r)) / len(r)):.3f} on (geometric) average, at most {max(r):.3f}, above 1.03 in {sum(x > 1.03 for x in r)}")


def main():
    which = sys.argv[1] if len(sys.argv) > 1 else "layer"
    try:
        packed() if which == "packed" else few_and_split(which) if which in ("few", "split") else tiles(which)
    finally:
        set_variables({})


def tiles(which: str):
    import torch
    lib = _lib.library()
    st = _lib.current_stream

    def run(M, N, K, variables):
        for name in VARIABLES:
            os.environ.pop(name, None)
        os.environ.update(variables)
        lib.mi355x_reload_tuning()
        a, w = torch.randn(M, K, device="cuda"), torch.randn(N, K, device="cuda") * 0.05
        bias, out = torch.randn(N, device="cuda"), torch.empty(M, N, device="cuda")
        launch = lambda: lib.mi355x_gemm_f32(a.data_ptr(), w.data_ptr(), out.data_ptr(), bias.data_ptr(), None, 1, 1, M, N, K,
                                             _lib.i64_array([0, 0, K, 1]), _lib.i64_array([0, 0, 1, K]), _lib.i64_array([0, 0, N]),
                                             None, 1.0, _lib.EPI_BIAS, st())
        return min(graph_time_us(launch, reps=20) for _ in range(2))

    print(f"{'M x N x K':>18s} {'tiles 128x48':>12s} " + " ".join(f"{name:>9s}" for name, _ in FORMS) + "   library / best forced form")
    for M, N, K in shapes(which):
        times = [run(M, N, K, variables) for _, variables in FORMS]
        best = min(times[1:])
        tiles = ((M + 127) // 128) * ((N + 47) // 48)
        print(f"{M:6d}x{N:5d}x{K:5d} {tiles:12d} " + " ".join(f"{t:9.2f}" for t in times) +
              f"   {times[0] / best:5.3f} ({FORMS[1 + times[1:].index(best)][0]}; {2.0 * M * N * K / times[0] / 1e6:5.1f} TFLOP/s)", flush=True)


if __name__ == "__main__":
    main()
