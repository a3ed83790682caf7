"""Fused attention through the library's own choice, the fp32 kernels (``MI355X_ATTN_SPLIT=0``) and the split bf16 form (``=1``).

    python -m dace_onnx_amd.testing.attention_variants

Prints microseconds per launch (HIP events around graph-recorded launches after a warm-up by time) for batches of 12 heads over one to 512
keys, without a mask and with one of the keys.
"""
import math
import os

from .. import _lib
from .profiling import graph_time_us

VARIABLE = "MI355X_ATTN_SPLIT"
SHAPES = [(b, s, s) for s, batches in ((16, (1, 8, 64)), (33, (1, 32)), (64, (1, 8, 32, 64)), (100, (1, 8, 32)), (128, (1, 4, 8, 16, 32)), (173, (1, 5, 20)),
                                       (200, (4, 20)), (256, (1, 8, 32)), (384, (2, 8)), (512, (1, 4, 16))) for b in batches] + [(8, 16, 512), (8, 512, 33)]


def main():
    import torch
    lib, i64, ratios = _lib.library(), _lib.i64_array, []

    def force(form):
        os.environ.pop(VARIABLE, None)
        if form is not None:
            os.environ[VARIABLE] = form
        lib.mi355x_reload_tuning()

    try:
        for masked in (False, True):
            for b, sq, sk in SHAPES:
                q, k, v, out = (torch.randn(b, 12, s, 64, device="cuda") for s in (sq, sk, sk, sq))
                mask = torch.zeros(b, 1, 1, sk, device="cuda")
                strides = [i64(t.stride()[:3]) for t in (q, k, v, out)]
                pointers = [t.data_ptr() for t in (q, k, v, out)]
                if masked:
                    launch = lambda: lib.mi355x_attention_masked_f32(*pointers, mask.data_ptr(), b, 12, sq, sk, 64, *strides, i64([sk, 0, 0]), 0.125,   # noqa: E731
                                                                     _lib.current_stream())
                else:
                    launch = lambda: lib.mi355x_attention_f32(*pointers, b, 12, sq, sk, 64, *strides, 0.125, _lib.current_stream())   # noqa: E731
                times = []
                for form in (None, "0", "1"):
                    force(form)
                    times.append(min(graph_time_us(launch, reps=20, warm_ms=20.0) for _ in range(2)))
                ratios.append((times[0] / times[1], times[0] / min(times[1:])))
                print(f"{b:3d} x 12 x {sq:3d} x {sk:3d} {'masked' if masked else '      '} library {times[0]:7.2f} fp32 {times[1]:7.2f} split {times[2]:7.2f}"
                      f"   library / fp32 {ratios[-1][0]:.3f}, / best {ratios[-1][1]:.3f}", flush=True)
        for name, column in (("fp32", 0), ("best form", 1)):
            r = [x[column] for x in ratios]
            print(f"{len(r)} shapes: library / {name} {math.exp(sum(map(math.log, r)) / len(r)):.3f} on (geometric) average, at most {max(r):.3f}, above 1.03 in {sum(x > 1.03 for x in r)}")
    finally:
        force(None)


if __name__ == "__main__":
    main()
