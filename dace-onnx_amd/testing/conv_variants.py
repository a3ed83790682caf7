"""Conv + bias + Relu through the library's own choice and through the other forms of the gather kernel, over the 3 x 3 and
1 x 1 layers of a ResNet-50 at 8 and 32 images.

    python -m dace_onnx_amd.testing.conv_variants
    python -m dace_onnx_amd.testing.conv_variants few     # layers of few tiles: 1 to 16 images, and 160 random ones
    python -m dace_onnx_amd.testing.conv_variants packed  # by packed filters: a residual network's layers of 1 to 32 images, and 100 random ones

Prints microseconds per launch (HIP events around graph-recorded launches after a warm-up by time, as bench.py measures
its rows) for

* ``library``: 64-position tiles through the lean kernel (three-deep register ring, three workgroups per CU);
* ``six-deep``: the same tiles through the six-deep ring, two workgroups per CU (``MI355X_CONV_PER_CU=2``);
* ``wide``: 128-position tiles, one workgroup per CU (``MI355X_CONV_GATHER_BN=128``).

The three add up the same products in the same order: the results are compared bit for bit here as well. ``few`` has the library's
choice, ``lds``, never the few-tile kernel (``MI355X_CONV_DIRECT=0``), and its tiles (``=11`` ...), with weights that are not in the L2. ``packed``, with
such weights too, has the library's choice, ``before``, without the packed filters (``MI355X_CONV_PACKED=0``), and the forms of the packed kernel that take the
layer by number, as in its table (``=1`` ...).
"""
import itertools
import math
import os
import random
import sys

from .. import _lib
from .profiling import graph_time_us

VARIABLES = ("MI355X_CONV_PER_CU", "MI355X_CONV_GATHER_BN", "MI355X_CONV_DIRECT", "MI355X_CONV_PACKED")
FORMS = (("library", {}), ("six-deep", {"MI355X_CONV_PER_CU": "2"}), ("wide", {"MI355X_CONV_GATHER_BN": "128"}))
LAYERS = ((64, 56, 64, 3), (128, 28, 128, 3), (256, 14, 256, 3), (512, 7, 512, 3), (64, 56, 256, 1), (256, 56, 64, 1), (256, 56, 128, 1),
          (512, 28, 128, 1), (1024, 14, 256, 1), (2048, 7, 512, 1), (512, 7, 2048, 1), (128, 28, 512, 1))   # C, H = W, M, k


FEW = (("library", None), ("lds", "0"), ("16x16", "11"), ("32x16", "21"), ("32x32", "22"))


def few_layers():
    """images, C, H = W, M, k, stride"""
    for N in (1, 2, 4, 8, 16):
        for C, H, M in ((64, 56, 64), (128, 28, 128), (256, 14, 256), (512, 7, 512)):
            yield N, C, H, M, 3, 1
        for C, H, M, k in ((64, 56, 128, 3), (64, 56, 128, 1), (128, 28, 256, 3), (128, 28, 256, 1), (256, 14, 512, 3), (256, 14, 512, 1)):
            yield N, C, H, M, k, 2
    rng = random.Random("few")
    for _ in range(160):
        yield (rng.choice((1, 1, 2, 3, 5, 8)), rng.choice((32, 64, 96, 128, 192, 256, 512, 1024)), rng.choice((4, 7, 10, 14, 20, 28, 33, 56)),
               rng.choice((16, 32, 48, 64, 96, 100, 128, 200, 256, 512)), rng.choice((1, 3, 3)), rng.choice((1, 1, 2)))


def few():
    import torch
    lib, i64, behind = _lib.library(), _lib.i64_array, []
    for N, C, H, M, k, stride in few_layers():
        size = (H - 1) // stride + 1
        x, b, y = torch.randn(N, C, H, H, device="cuda"), torch.randn(M, device="cuda"), torch.empty(N, M, size, size, device="cuda")
        w = itertools.cycle([torch.randn(M, C, k, k, device="cuda") * 0.05 for _ in range(max(1, min(20, int(64e6 / (4 * M * C * k * k)))))])
        launch = lambda: lib.mi355x_conv2d_f32(x.data_ptr(), next(w).data_ptr(), b.data_ptr(), y.data_ptr(), N, C, H, H, M, k, k, i64([k // 2] * 4),   # noqa: E731
                                               i64([stride] * 2), i64([1, 1]), _lib.EPI_BIAS | _lib.EPI_RELU, _lib.current_stream())
        times = []
        for _, form in FEW:
            os.environ.pop("MI355X_CONV_DIRECT", None)
            if form is not None:
                os.environ["MI355X_CONV_DIRECT"] = form
            lib.mi355x_reload_tuning()
            times.append(min(graph_time_us(launch, reps=20, warm_ms=20.0) for _ in range(2)))
        behind.append((times[0] / times[1], times[0] / min(times[1:])))
        print(f"{N:3d} x {C:4d} x {H:2d} x {H:2d} -> {M:4d}, {k} x {k}, stride {stride}   " + " ".join(f"{name} {t:7.2f}" for (name, _), t in zip(FEW, times)) +
              f"   library / lds {behind[-1][0]:.3f}, / best {behind[-1][1]:.3f}", flush=True)
    print(f"{len(behind)} layers: library / lds at most {max(b for b, _ in behind):.3f}, above 1.03 in {sum(b > 1.03 for b, _ in behind)}; "
          f"library / best form {sum(b for _, b in behind) / len(behind):.3f} on average, at most {max(b for _, b in behind):.3f}")


def packed_layers():
    """images, C, H = W, M, k, stride"""
    for N in (1, 4, 8, 32):
        for C, H, M, k, stride in ((3, 224, 64, 7, 2), (64, 56, 64, 3, 1), (64, 56, 128, 3, 2), (64, 56, 128, 1, 2), (128, 28, 128, 3, 1), (128, 28, 256, 3, 2),
                                   (128, 28, 256, 1, 2), (256, 14, 256, 3, 1), (256, 14, 512, 3, 2), (256, 14, 512, 1, 2), (512, 7, 512, 3, 1)):
            yield N, C, H, M, k, stride
    rng = random.Random("packed")
    for _ in range(100):
        k = rng.choice((3, 3, 3, 1, 1, 7))
        C = rng.randint(1, 4) if k == 7 else 8 * rng.randint(1, 64)
        H = rng.randint(48, 256) if k == 7 else rng.choice((5, 7, 10, 14, 20, 28, 33, 48, 56, 64, 80))
        yield rng.choice((1, 2, 4, 8, 16, 32)) if H < 64 else rng.choice((1, 2, 4)), C, H, rng.choice((16, 32, 64, 100, 128, 256, 512, 768)), k, rng.choice((1, 1, 2))


def packed():
    import torch
    lib, i64, ratios = _lib.library(), _lib.i64_array, []
    forms = (("library", None), ("before", "0")) + tuple((str(f), str(f)) for f in range(1, 10))
    for N, C, H, M, k, stride in packed_layers():
        size = (H - 1) // stride + 1
        x, b = torch.randn(N, C, H, H, device="cuda"), torch.randn(M, device="cuda")
        y = torch.empty(N, M, size, size, device="cuda")
        geometry = [N, C, H, H, M, k, k, i64([k // 2] * 4), i64([stride] * 2), i64([1, 1])]
        filters = []
        for _ in range(max(1, min(20, int(64e6 / (4 * M * C * k * k))))):
            w, copy = torch.randn(M, C, k, k, device="cuda") * 0.05, torch.empty(-(-M // 32) * -(-C // 16) * (14 if C <= 4 else k * k) * 768, dtype=torch.int32, device="cuda")
            _lib.check(lib.mi355x_pack_conv_f32(w.data_ptr(), copy.data_ptr(), M, C, k, k, _lib.current_stream()), "pack")
            filters.append((w, copy))
        turns = itertools.cycle(filters)

        def launch():
            w, copy = next(turns)
            return lib.mi355x_conv2d_packed_f32(x.data_ptr(), copy.data_ptr(), w.data_ptr(), b.data_ptr(), None, y.data_ptr(), *geometry,
                                                _lib.EPI_BIAS | _lib.EPI_RELU, _lib.current_stream())

        times, names = [], []
        for name, form in forms:
            os.environ.pop("MI355X_CONV_PACKED", None)
            if form is not None:
                os.environ["MI355X_CONV_PACKED"] = form
            lib.mi355x_reload_tuning()
            takes = bool(lib.mi355x_conv2d_packed_pays(*geometry, 1))
            if name == "library":
                choice = "packed" if takes else "before"
            if takes or len(times) < 2:
                names.append(name)
                times.append(min(graph_time_us(launch, reps=20, replays=3, warm_ms=10.0) for _ in range(2)))
        ratios.append((times[0] / times[1], times[0] / min(times[1:])))
        print(f"{N:3d} x {C:4d} x {H:2d} x {H:2d} -> {M:4d}, {k} x {k}, stride {stride}  {choice} " + " ".join(f"{name} {t:.1f}" for name, t in zip(names, times)) +
              f"   library / before {ratios[-1][0]:.3f}, / best {ratios[-1][1]:.3f}", flush=True)
    for name, column in (("before", 0), ("best form", 1)):
        r = [x[column] for x in ratios]
        print(f"{len(r)} layers: library / {name} {math.exp(sum(map(math.log, r)) / len(r)):.3f} on (geometric) average, at most {max(r):.3f}, above 1.03 in {sum(x > 1.03 for x in r)}")


def main():
    try:
        packed() if sys.argv[1:] == ["packed"] else few() if sys.argv[1:] == ["few"] else layers()
    finally:
        for name in VARIABLES:
            os.environ.pop(name, None)
        _lib.library().mi355x_reload_tuning()


def layers():
    import torch
    lib = _lib.library()
    st = _lib.current_stream
    ones = _lib.i64_array([1, 1])

    def run(N, C, H, M, k, variables):
        for name in VARIABLES:
            os.environ.pop(name, None)
        os.environ.update(variables)
        lib.mi355x_reload_tuning()
        g = torch.Generator(device="cuda").manual_seed(1)
        x = torch.randn(N, C, H, H, device="cuda", generator=g)
        w = torch.randn(M, C, k, k, device="cuda", generator=g) * (2.0 / (C * k * k)) ** 0.5
        b = torch.randn(M, device="cuda", generator=g)
        y = torch.full((N, M, H, H), float("nan"), device="cuda")
        pads = _lib.i64_array([k // 2] * 4)
        launch = lambda: lib.mi355x_conv2d_f32(x.data_ptr(), w.data_ptr(), b.data_ptr(), y.data_ptr(), N, C, H, H, M, k, k, pads, ones, ones,
                                               _lib.EPI_BIAS | _lib.EPI_RELU, st())
        _lib.check(launch(), "conv2d")
        torch.cuda.synchronize()
        return min(graph_time_us(launch, reps=20) for _ in range(2)), y.clone()

    print(f"{'images x C x H x W -> M, filter':>34s} {'tiles':>6s} " + " ".join(f"{name:>9s}" for name, _ in FORMS) + "   TFLOP/s  library / best  same bits")
    for N in (8, 32):
        for C, H, M, k in LAYERS:
            results = [run(N, C, H, M, k, variables) for _, variables in FORMS]
            times = [t for t, _ in results]
            same = all(bool(torch.equal(results[0][1], y)) for _, y in results[1:])
            tiles = ((M + 63) // 64) * ((N * H * H + 63) // 64)
            flop = 2.0 * N * M * H * H * C * k * k
            print(f"{N:3d} x {C:4d} x {H:2d} x {H:2d} -> {M:4d}, {k} x {k}    {tiles:6d} " + " ".join(f"{t:9.2f}" for t in times) +
                  f"   {flop / times[0] / 1e6:7.1f}  {times[0] / min(times):14.3f}  {same}", flush=True)


if __name__ == "__main__":
    main()
