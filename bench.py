#!/usr/bin/env python3
"""Benchmark of the ONNX library-node hot path on one MI355X.

A step is one BERT-base encoder layer (B=8, S=128, hidden 768, 12 heads, FFN
3072, fp32) run through ``ONNXModel`` with the "mi355x" expansions: the
configuration the headline metric is quoted on. Inputs and weights are
synthetic (seeded) and resident in HBM before the timed region. A step is
issued as one HIP-graph replay or as host-issued launches, whichever was
faster during warm-up (--replay).

Prints one JSON line:
  value / ms_per_step   milliseconds per encoder layer (lower is better)
  roofline              the dominant kernel (the fp32 MFMA GEMM): algorithmic FLOP
                        of all GEMM launches of a layer / their measured durations
  cpu_baseline          the CPU restatement of the reference's expansion of the
                        same layer (oracle), timed on the host cores of this box
  kernels               per-kernel roofline rows (every launch of the layer, plus
                        the stand-alone Softmax / LayerNorm / Conv / MatMulInteger
                        configurations), each measured live with HIP events
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

WARM_MS = 40.0   # untimed repetitions before every measurement, see dace_onnx_amd/testing/profiling.py
# published MI355X peaks (dense)
PEAK_FP32_MFMA_TFLOPS = 157.3
PEAK_SPLIT_MFMA_TFLOPS = 2516.6 / 6   # six bf16 products for one of fp32
PEAK_INT8_MFMA_TOPS = 5000.0
PEAK_HBM_GBS = 8000.0
# L2 <-> fabric bytes of the four GEMM launches of one layer, from rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE runs of
# this script scaled by a copy kernel of known size (profiles/bert_layer_gemm_traffic.txt); counters cannot be
# read from inside the process, so the figure is carried here and re-measured whenever the GEMM kernels change
GEMM_TRAFFIC_BYTES_PER_LAYER = 212352205
GEMM_TRAFFIC_SOURCE = "profiles/bert_layer_gemm_traffic.txt (rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE runs of this script; not re-measured by this run)"


def algorithmic_work(name, args):
    """(flops, bytes) of one launch from its C-ABI arguments (fp32 unless stated)."""
    if name == "mi355x_gemm_packed_f32":   # the same arguments with the packed copy of B after A
        return algorithmic_work("mi355x_gemm_f32", args[:1] + args[2:])
    if name == "mi355x_gemm_parts_f32":
        parts, M, N, K = args[4:8]
        return 2.0 * M * N * K, 4.0 * (M * K + K * N + parts * M * N)
    if name == "mi355x_layernorm_parts_f32":   # sums, residual and result
        parts, rows, cols = args[1], args[8], args[9]
        return 0.0, 4.0 * (parts + 2) * rows * cols + 12.0 * cols
    if name == "mi355x_gemm_f32":
        b0, b1, M, N, K = args[5:10]
        epi = args[15]
        flops = 2.0 * b0 * b1 * M * N * K
        nbytes = 4.0 * b0 * b1 * (M * K + K * N + M * N * (2 if epi & 8 else 1))
        return flops, nbytes
    if name == "mi355x_attention_f32":
        b0, b1, sq, sk, d = args[4:9]
        return 4.0 * b0 * b1 * sq * sk * d, 4.0 * b0 * b1 * (2 * sq * d + 2 * sk * d)
    if name == "mi355x_softmax_f32":
        outer, n, inner = args[2:5]
        return 0.0, 8.0 * outer * n * inner
    if name == "mi355x_layernorm_f32":
        rows, cols = args[4:6]
        return 0.0, 8.0 * rows * cols + 8.0 * cols
    if name == "mi355x_eltwise_f32":
        shape = args[5]
        n = 1
        for v in shape:
            n *= v
        reads = 2 if args[0] < 16 else 1
        return 0.0, 4.0 * n * (reads + 1)
    if name == "mi355x_permute_b32":
        n = 1
        for v in args[3]:
            n *= v
        return 0.0, 8.0 * n
    return 0.0, 0.0


def kernel_row(label, us, flops=0.0, nbytes=0.0, bound=None, peak=None):
    row = {"kernel": label, "us": round(us, 3)}
    if flops:
        row["tflops"] = round(flops / us / 1e6, 2)
    if nbytes:
        row["gbs"] = round(nbytes / us / 1e3, 1)
    if bound == "mfma":
        row.update(bound="mfma", frac=round(flops / us / 1e6 / (peak or PEAK_FP32_MFMA_TFLOPS), 4))
    elif bound == "hbm":
        row.update(bound="hbm", frac=round(nbytes / us / 1e3 / PEAK_HBM_GBS, 4))
    return row


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--no-cpu-baseline", action="store_true", help="skip the host-side oracle timing")
    ap.add_argument("--no-kernels", action="store_true", help="skip the per-kernel roofline rows")
    ap.add_argument("--replay", choices=("auto", "graph", "eager"), default="auto",
                    help="how a step is issued: one HIP-graph replay, host-issued launches, or (auto) whichever of the "
                         "two was faster over the warm-up steps")
    ap.add_argument("--eager", action="store_true", help="same as --replay eager")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="also run a plain 256 MiB -> 256 MiB elementwise copy three times, so that a counter run of this "
                         "command holds a kernel of known HBM traffic to scale FETCH_SIZE / WRITE_SIZE by")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU: this path has no multi-GPU part (got --gpus {args.gpus}); "
              f"run with --gpus 1", file=sys.stderr)
        sys.exit(2)

    import numpy as np
    import torch
    import dace_onnx_amd.onnx as donnx
    from dace_onnx_amd import _lib
    from dace_onnx_amd.testing.graphs import bert_encoder_layer_model
    from dace_onnx_amd.testing.profiling import graph_time_us, warm_up
    from oracle import pure_ops  # checker / CPU baseline only

    if not torch.cuda.is_available():
        print("bench.py needs the MI355X (no HIP device visible)", file=sys.stderr)
        sys.exit(1)
    lib = _lib.library()
    torch.cuda.set_device(0)

    # ---- workload: benchmark config 3 -------------------------------------------------
    B, S, H, HEADS, FFN = 8, 128, 768, 12, 3072
    rng = np.random.default_rng(3)
    weights = pure_ops.bert_layer_weights(rng, hidden=H, ffn=FFN)
    x_host = rng.normal(size=(B, S, H)).astype(np.float32)
    model = donnx.ONNXModel("bert_base_encoder_layer", bert_encoder_layer_model(weights, B, S, HEADS))
    x = torch.from_numpy(x_host).cuda()
    y = model(x)  # compiles, binds
    compiled = model.compile_and_init()
    # parity gate inside the benchmark: a fast wrong layer is not a result
    expected = pure_ops.bert_layer(x_host, weights, heads=HEADS)
    err = float(np.abs(y.cpu().numpy().astype(np.float64) - expected).max() / np.abs(expected).max())
    if not err < 1e-4:
        print(f"parity check failed: max rel err {err:.3e}", file=sys.stderr)
        sys.exit(1)

    out = torch.empty_like(y)
    call_kwargs = {"x": x, "y": out, **model.clean_weights}
    compiled(**call_kwargs)
    def eager_step():
        compiled(**call_kwargs)

    def timed(fn, n):
        torch.cuda.synchronize()
        t = time.perf_counter()
        for _ in range(n):
            fn()
        torch.cuda.synchronize()
        return (time.perf_counter() - t) / max(n, 1)

    mode = "eager" if args.eager else args.replay
    if mode == "eager":
        step = eager_step
    else:
        compiled.capture_graph()
        step = compiled.replay
    if mode == "auto":
        # a graph replay has one launch but a few microseconds between replays; host-issued
        # launches have none of that but need the host to stay ahead of the GPU
        # (compared once the core clock is up, over enough steps for the difference of a few per cent to show)
        warm_up(compiled.replay, WARM_MS)
        n_compare = max(args.warmup, 200)
        t_eager, t_graph = timed(eager_step, n_compare), timed(compiled.replay, n_compare)
        t_eager, t_graph = min(t_eager, timed(eager_step, n_compare)), min(t_graph, timed(compiled.replay, n_compare))
        mode, step = ("eager", eager_step) if t_eager < t_graph else ("graph", compiled.replay)
    else:
        timed(step, args.warmup)
    # besides the --warmup steps: steps for at least 40 ms, the time the core clock needs to come back up after
    # idling (every per-kernel row below is warmed the same way, so the headline and the rows are comparable)
    warm_steps = warm_up(step, WARM_MS)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    ms_per_step = elapsed / args.steps * 1e3
    torch.cuda.synchronize()
    final_err = float(np.abs(out.cpu().numpy().astype(np.float64) - expected).max() / np.abs(expected).max())
    assert final_err < 1e-4, final_err

    if args.calibrate_copy:
        src = torch.randn(64 * 1024 * 1024, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(3):
            torch.mul(src, 1.0, out=dst)
        torch.cuda.synchronize()
        del src, dst

    # ---- per-kernel durations, HIP events on the launch stream -----------------------------
    kernels = []
    gemm_flops = gemm_us = gemm_floor_us = gemm_bytes = layer_us = 0.0
    if not args.no_kernels:
        for node, relaunch in compiled.bound_launches():
            name = node.function
            plain = [a.values if hasattr(a, "values") else a for a in node.args]
            flops, nbytes = algorithmic_work(name, plain)
            us = graph_time_us(relaunch)
            layer_us += us   # sum of the layer's kernel durations, to hold against ms_per_step
            if name in ("mi355x_gemm_f32", "mi355x_gemm_packed_f32"):
                packed = name == "mi355x_gemm_packed_f32"
                if packed:
                    plain = plain[:1] + plain[2:]
                gemm_flops += flops
                gemm_bytes += nbytes
                gemm_us += us
                gemm_floor_us += flops / 1e6 / (PEAK_SPLIT_MFMA_TFLOPS if packed else PEAK_FP32_MFMA_TFLOPS)
                label = "gemm_f32{} b{}x{} {}x{}x{} epi={}".format("_packed" if packed else "", *plain[5:10], plain[15])
                kernels.append(kernel_row(label, us, flops, nbytes, "mfma", PEAK_SPLIT_MFMA_TFLOPS if packed else None))
            elif name == "mi355x_gemm_parts_f32":
                packed = node.args[2].connector is not None
                gemm_flops += flops
                gemm_bytes += nbytes
                gemm_us += us
                gemm_floor_us += flops / 1e6 / (PEAK_SPLIT_MFMA_TFLOPS if packed else PEAK_FP32_MFMA_TFLOPS)
                kernels.append(kernel_row("gemm_parts_f32{} {} parts {}x{}x{}".format("_packed" if packed else "", *plain[4:8]), us, flops, nbytes, "mfma",
                                          PEAK_SPLIT_MFMA_TFLOPS if packed else None))
            elif name == "mi355x_attention_f32":
                label = "attention_f32 b{}x{} q{} k{} d{}".format(*plain[4:9])
                kernels.append(kernel_row(label, us, flops, nbytes, "mfma"))
            else:
                label = name.replace("mi355x_", "") + " " + "x".join(str(v) for v in (plain[5] if name == "mi355x_eltwise_f32"
                                                                                     else plain[3] if name == "mi355x_permute_b32"
                                                                                     else plain[2:5] if name == "mi355x_softmax_f32"
                                                                                     else [plain[1], *plain[8:10]] if name == "mi355x_layernorm_parts_f32"
                                                                                     else plain[4:6]))
                kernels.append(kernel_row(label, us, 0.0, nbytes, "hbm"))

        # stand-alone configurations of the metric (benchmark configs 1, 2, 4, 5), seeded as the parity tests seed them;
        # each row also carries the CPU restatement of the reference's expansion of the same operator on the same inputs
        # (oracle/pure_ops.c, OpenMP over the outer map dimensions like the code the reference generates), timed on
        # this box's host cores after the GPU figure is taken: never inside a timed GPU region
        from oracle import c_oracle   # checker / CPU baseline only
        cpu_threads = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))

        def cpu_ms_of(fn, budget_s=6.0, max_runs=20):
            if args.no_cpu_baseline:
                return None
            fn()  # warm-up: thread pool, page faults of the output
            n, t0 = 0, time.perf_counter()
            while n < max_runs and (n == 0 or time.perf_counter() - t0 < budget_s):
                fn()
                n += 1
            return round((time.perf_counter() - t0) / n * 1e3, 4)

        def with_cpu(row, fn, **kw):
            ms = cpu_ms_of(fn, **kw)
            if ms is not None:
                row.update(cpu_ms=ms, cpu_threads=cpu_threads, cpu_kind="port (C restatement of the pure expansion)",
                           cpu_over_gpu_time=round(ms * 1e3 / row["us"], 1))
            kernels.append(row)

        st = _lib.current_stream
        dev = lambda a: torch.from_numpy(a).cuda()
        # what a launch costs when the kernel does nothing: the floor under the small rows below
        launch_floor_us = graph_time_us(lambda: lib.mi355x_launch_empty_kernel(st()), reps=200)

        # config 1: Conv X[5,3,10,10] * W[16,3,3,3], strides 2, no padding, no bias (a latency case: 69 120 FLOP)
        rng1 = np.random.default_rng(1)
        x1, w1 = rng1.random((5, 3, 10, 10), dtype=np.float32), rng1.random((16, 3, 3, 3), dtype=np.float32)
        xc1, wc1, yc1 = dev(x1), dev(w1), torch.empty(5, 16, 4, 4, device="cuda")
        nopad, twos, ones = _lib.i64_array([0, 0, 0, 0]), _lib.i64_array([2, 2]), _lib.i64_array([1, 1])
        us = graph_time_us(lambda: lib.mi355x_conv2d_f32(xc1.data_ptr(), wc1.data_ptr(), None, yc1.data_ptr(), 5, 3, 10, 10, 16,
                                                         3, 3, nopad, twos, ones, 0, st()), reps=200)
        row = kernel_row("cfg1 conv 5x3x10x10 k3 s2", us, 69120.0, 12848.0)
        row.update(bound="latency", launch_floor_us=round(launch_floor_us, 3))
        assert np.allclose(c_oracle.conv2d(x1, w1, None, (2, 2)), yc1.cpu().numpy(), rtol=1e-4, atol=1e-5)
        with_cpu(row, lambda: c_oracle.conv2d(x1, w1, None, (2, 2)), budget_s=1.0, max_runs=2000)

        # config 2
        rng2 = np.random.default_rng(2)
        x2s = rng2.normal(size=(12288, 128)).astype(np.float32)
        x2l = rng2.normal(size=(1024, 768)).astype(np.float32)
        g2, b2 = rng2.normal(1.0, 0.02, size=768).astype(np.float32), rng2.normal(0.0, 0.02, size=768).astype(np.float32)
        xs, xl, g_, b_ = dev(x2s), dev(x2l), dev(g2), dev(b2)
        ys, yl = torch.empty_like(xs), torch.empty_like(xl)

        def small_hbm_row(label, us, nbytes):
            # a launch of its own cannot beat floor + bytes / peak: the fraction of the roofline that bound allows
            row = kernel_row(label, us, 0.0, nbytes, "hbm")
            data_us = nbytes / PEAK_HBM_GBS / 1e3
            row.update(launch_floor_us=round(launch_floor_us, 3), ceiling_frac=round(data_us / (launch_floor_us + data_us), 4))
            return row

        us = graph_time_us(lambda: lib.mi355x_softmax_f32(xs.data_ptr(), ys.data_ptr(), 12288, 128, 1, st()))
        with_cpu(small_hbm_row("cfg2 softmax 8x12x128x128", us, 12582912.0), lambda: c_oracle.softmax(x2s), budget_s=2.0)
        us = graph_time_us(lambda: lib.mi355x_layernorm_f32(xl.data_ptr(), g_.data_ptr(), b_.data_ptr(), yl.data_ptr(),
                                                            1024, 768, 1e-12, st()))
        with_cpu(small_hbm_row("cfg2 layernorm 8x128x768", us, 6297600.0),
                 lambda: c_oracle.layer_normalization(x2l, g2, b2, 1e-12), budget_s=2.0)
        # the same two kernels on inputs large enough that the launch floor no longer matters (805 MB each)
        xs = torch.randn(1572864, 128, device="cuda")
        ys = torch.empty_like(xs)
        us = graph_time_us(lambda: lib.mi355x_softmax_f32(xs.data_ptr(), ys.data_ptr(), 1572864, 128, 1, st()), reps=5)
        kernels.append(kernel_row("softmax 1572864x128 (1.6 GB moved)", us, 0.0, 8.0 * 1572864 * 128, "hbm"))
        del xs, ys
        xl = torch.randn(131072, 768, device="cuda")
        yl = torch.empty_like(xl)
        us = graph_time_us(lambda: lib.mi355x_layernorm_f32(xl.data_ptr(), g_.data_ptr(), b_.data_ptr(), yl.data_ptr(),
                                                            131072, 768, 1e-12, st()), reps=5)
        kernels.append(kernel_row("layernorm 131072x768 (0.8 GB moved)", us, 0.0, 8.0 * 131072 * 768, "hbm"))
        del xl, yl

        # config 4
        rng4 = np.random.default_rng(4)
        x4 = rng4.normal(size=(32, 64, 56, 56)).astype(np.float32)
        w4 = (rng4.normal(size=(64, 64, 3, 3)) * np.sqrt(2.0 / 576)).astype(np.float32)
        b4 = np.zeros(64, np.float32)
        xc, wc, bc = dev(x4), dev(w4), dev(b4)
        yc = torch.empty(32, 64, 56, 56, device="cuda")
        pads = _lib.i64_array([1, 1, 1, 1])
        us = graph_time_us(lambda: lib.mi355x_conv2d_f32(xc.data_ptr(), wc.data_ptr(), bc.data_ptr(), yc.data_ptr(), 32, 64,
                                                         56, 56, 64, 3, 3, pads, ones, ones, 3, st()), reps=20)
        with_cpu(kernel_row("cfg4 conv+relu 32x64x56x56 k3 p1", us, 7398752256.0, 51527680.0, "mfma"),
                 lambda: np.maximum(c_oracle.conv2d(x4, w4, b4, (1, 1), (1, 1, 1, 1), (1, 1)), 0.0), max_runs=3)

        # config 5
        rng5 = np.random.default_rng(5)
        a5 = rng5.integers(-128, 128, size=(4096, 768), dtype=np.int8)
        b5 = rng5.integers(-128, 128, size=(768, 3072), dtype=np.int8)
        ai, bi = dev(a5), dev(b5)
        za, zb = torch.tensor([3], dtype=torch.int8, device="cuda"), torch.tensor([-2], dtype=torch.int8, device="cuda")
        yi = torch.empty(4096, 3072, dtype=torch.int32, device="cuda")
        us = graph_time_us(lambda: lib.mi355x_matmul_integer_i8(ai.data_ptr(), bi.data_ptr(), za.data_ptr(), zb.data_ptr(),
                                                                yi.data_ptr(), 4096, 3072, 768, st()), reps=20)
        row = kernel_row("cfg5 matmul_integer 4096x3072x768", us, 19327352832.0, 55836672.0, "hbm")
        row["mfma_frac"] = round(19327352832.0 / us / 1e6 / PEAK_INT8_MFMA_TOPS, 4)
        with_cpu(row, lambda: c_oracle.matmul_integer(a5, b5, 3, -2), max_runs=5)

    roofline = None
    if gemm_us > 0:
        achieved = gemm_flops / gemm_us / 1e6
        peak = gemm_flops / gemm_floor_us / 1e6   # of the matrix units the launches run on
        roofline = {"bound": "mfma", "achieved": round(achieved, 2), "peak": round(peak, 1), "unit": "TFLOP/s",
                    "frac": round(achieved / peak, 4), "traffic": GEMM_TRAFFIC_BYTES_PER_LAYER,
                    "traffic_source": GEMM_TRAFFIC_SOURCE,
                    "algorithmic_bytes_per_layer": gemm_bytes,
                    "kernel": "gemm_f32_packed_kernel / gemm_f32_nt_kernel (all GEMM launches of one layer: QKV, output projection, FFN1, "
                              "FFN2; fp32 products as six bf16 ones where the weights are packed; the attention core runs in its own fused kernel, listed under kernels)",
                    "flop_per_layer": gemm_flops, "us_per_layer": round(gemm_us, 2)}

    # ---- CPU baseline: the oracle's layer on this box's host cores ---------------------------
    cpu_baseline = None
    if not args.no_cpu_baseline:
        cores = torch.get_num_threads()   # the threads torch's and numpy's BLAS matmuls run on
        pure_ops.bert_layer(x_host, weights, heads=HEADS)  # warm-up
        n_cpu, t0 = 0, time.perf_counter()
        while n_cpu < 8 and time.perf_counter() - t0 < 20.0:
            pure_ops.bert_layer(x_host, weights, heads=HEADS)
            n_cpu += 1
        cpu_ms = (time.perf_counter() - t0) / n_cpu * 1e3
        cpu_baseline = {"value": round(cpu_ms, 2), "unit": "ms", "cores": cores, "kind": "port",
                        "omp_num_threads": os.environ.get("OMP_NUM_THREADS"), "os_cpu_count": os.cpu_count(),
                        "sample": f"{n_cpu} runs of the same layer (same seed, B=8 S=128) through the numpy restatement of "
                                  f"the reference's pure expansions, BLAS matmuls on {cores} threads"}

    result = {
        "metric": "BERT-base encoder layer latency (B=8, S=128, fp32) via ONNXModel",
        "value": round(ms_per_step, 5), "unit": "ms", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 5), "higher_is_better": False, "scaling": "weak", "vs_baseline": None,
        "dtype": "f32", "data": "synthetic",
        "config": {"workload": "BERT-base encoder layer, B=8 S=128 H=768 heads=12 FFN=3072, "
                               "ONNX graph of MatMul/Add/Reshape/Transpose/Div/Softmax/LayerNormalization/Gelu",
                   "launches_per_step": compiled.num_launches, "replay": "host_launches" if mode == "eager" else "hip_graph",
                   "warm_ms": WARM_MS, "warm_steps": warm_steps,
                   "kernel_us_per_step": round(layer_us, 2) if layer_us else None,
                   "max_rel_err_vs_oracle": err},
        "roofline": roofline, "cpu_baseline": cpu_baseline, "kernels": kernels,
    }
    print(json.dumps(result))


if __name__ == "__main__":
    main()
