"""Benchmark of the MI355X block-FP8 path (one GPU).

Headline (BASELINE.json metric): block-FP8 GEMM 4096x4096x8192, e4m3fn
operands with 1x128 activation / 128x128 weight fp32 scales, bf16 output.
One step = one w8a8_block_fp8_matmul call on inputs already resident in HBM
(the activations are quantised by act_quant once, before timing).

Prints ONE JSON line on stdout; progress goes to stderr. The line carries:
  roofline      the GEMM kernel's achieved TFLOP/s (algorithmic 2MNK per
                launch / mean launch time from HIP events around back-to-back
                launches on the launch stream) against dense FP8 MFMA peak;
  cpu_baseline  the reference's PyTorch CPU dequantise-then-matmul path
                (finegrained-fp8-helion/bench.py:11-14, restated in
                oracle/torch_ref.py) on a row sample of the same workload;
  secondary     act-quant, decode-shaped, medium, small, weight-quantiser and MLP-chain
                rows.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

PEAK_FP8_TFLOPS = 5000.0   # MI355X dense FP8 MFMA
PEAK_HBM_GBS = 8000.0      # MI355X HBM3E
METRIC = "TFLOP/s + % FP8 MFMA peak, block-FP8 GEMM 4096x4096x8192, 1 GPU"


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def parse():
    p = argparse.ArgumentParser()
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=50)
    # The GPU clock and power state settle over the first ~100 ms of
    # sustained MFMA work: after 200 warmup steps (~22 ms) the headline step
    # still measured 112-113 us, after 1000 or 3000 steps 109.5-110.3 us
    # (the kernel alone: 110 us either way).
    p.add_argument("--warmup", type=int, default=1000)
    p.add_argument("--no-cpu-baseline", action="store_true")
    p.add_argument("--no-secondary", action="store_true")
    p.add_argument("--only", default=None,
                   help="profile helper: run only one workload "
                        "(gemm|act_quant|decode|decode_graph[_m1|_m1_wide][_two_op]|decode_fused|"
                        "weight_quant|"
                        "weight_quant_bf16|mlp|"
                        "mlp_il|mlp_gateup|"
                        "mlp_down|medium|small|prefill|deep_gemm|deep_decode|copy|shapes|"
                        "shapes_streamed)"
                        " for --steps steps and exit without JSON")
    return p.parse_args()


def time_events(fn, steps, warmup, torch):
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    st = torch.cuda.current_stream()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record(st)
    for _ in range(steps):
        fn()
    e1.record(st)
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / steps  # ms per call


def time_steady(fn, steps, torch, warm_ms=25.0, min_warmup=200):
    """time_events after a warm-up of at least min_warmup calls and warm_ms
    of GPU time: the shader clock takes ~10 ms of MFMA load to settle after
    an HBM-bound leg, which 200 calls of a 5-30 us GEMM do not cover."""
    done, spent = 0, 0.0
    batch = min(50, min_warmup)
    while done < min_warmup or spent < warm_ms:
        spent += time_events(fn, batch, 0, torch) * batch
        done += batch
    return time_events(fn, steps, 0, torch)


def gemm_launcher(A, B, As, Bs, out, torch):
    """Direct C-ABI launch of the GEMM on the current stream (no Python-side
    allocation or validation), used to time the kernel itself."""
    from hf_kernels_helion_amd import _native
    lib = _native.load()
    M, K = A.shape
    N = B.shape[0]
    ws_bytes = lib.fp8b_gemm_workspace_size(M, N, K, 128, 128)
    ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=A.device)
    stream = torch.cuda.current_stream().cuda_stream
    args = (A.data_ptr(), A.stride(0), B.data_ptr(), B.stride(0), As.data_ptr(), As.stride(0),
            As.stride(1), Bs.data_ptr(), Bs.stride(0), Bs.stride(1), out.data_ptr(),
            out.stride(0), _native.BF16, M, N, K, 128, 128,
            ws.data_ptr() if ws_bytes else None, ws_bytes, stream)
    fn = lib.fp8b_w8a8_block_matmul

    def run():
        st = fn(*args)
        if st:
            _native.check(st, "fp8b_w8a8_block_matmul")
    return run, ws


def cpu_baseline(A, B, As, Bs, torch):
    from oracle import torch_ref
    torch.set_num_threads(os.cpu_count() or 1)
    R = 512
    M, K = A.shape
    N = B.shape[0]
    a, a_s = A[:R].contiguous(), As[:R].contiguous()
    torch_ref.dequant_matmul(a, B, a_s, Bs)  # warmup
    times = []
    t_start = time.perf_counter()
    while len(times) < 20 and (time.perf_counter() - t_start) < 12.0:
        t0 = time.perf_counter()
        torch_ref.dequant_matmul(a, B, a_s, Bs)
        times.append(time.perf_counter() - t0)
    t = sum(times) / len(times)
    cpu_model = "unknown CPU"
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                cpu_model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    return {
        "value": 2.0 * R * N * K / t / 1e12,
        "unit": "TFLOP/s",
        "cores": torch.get_num_threads(),
        "kind": "port",
        "sample": (f"{R} of {M} rows of the {M}x{N}x{K} workload: dequantise A rows and all of B "
                   f"with their block scales, fp32 matmul, bf16 cast (bench.py:11-14 restated); "
                   f"mean of {len(times)} iterations, {t * 1e3:.1f} ms each, "
                   f"os.cpu_count()={os.cpu_count()}, {cpu_model}"),
        "decode_32x4096x14336": cpu_decode_step(torch),
        "mlp_chain_3001": cpu_mlp_sample(torch),
    }


def cpu_mlp_sample(torch):
    """The M = 3001 MLP chain on the host, on a sample of 128 of
    its rows: CPU act-quant, dequantise-then-matmul against the gate/up
    weights [28672, 4096], silu_and_mul, act-quant, dequantise-then-matmul
    against the down weights [4096, 14336], as the reference's bench.py:11-14
    does per call; whole sampled chains, mean of up to 3 (about 10 s at most)."""
    from oracle import torch_ref
    from hf_kernels_helion_amd.finegrained_fp8_helion import synthetic
    R, H, I = 128, 4096, 14336
    x = synthetic.activations(R, H, seed=52)
    w13, s13 = synthetic.weights(2 * I, H, seed=50)
    w2, s2 = synthetic.weights(H, I, seed=51)

    def chain():
        q, s = torch_ref.act_quant(x, 128)
        h = torch_ref.dequant_matmul(q, w13, s, s13)
        a = torch_ref.silu_and_mul(h)
        q2, s2a = torch_ref.act_quant(a, 128)
        return torch_ref.dequant_matmul(q2, w2, s2a, s2)
    chain()  # warmup
    times = []
    t_start = time.perf_counter()
    while len(times) < 3 and (time.perf_counter() - t_start) < 10.0:
        t0 = time.perf_counter()
        chain()
        times.append(time.perf_counter() - t0)
    t = sum(times) / len(times)
    flop = 2.0 * R * (2 * I * H + H * I)
    return {"ms": round(t * 1e3, 1), "TFLOP/s": round(flop / t / 1e12, 4), "rows": R,
            "chains": len(times),
            "sample": f"{R} of 3001 rows; the weights are dequantised on every call"}


def cpu_decode_step(torch):
    """The decode configuration (C4) on the host: the CPU act-quant of the
    bf16 [32, 14336] activations (oracle/torch_ref.act_quant), then the
    dequantise-then-matmul of bench.py:11-14 against the [4096, 14336]
    weights with 128x128 block scales; whole steps, mean of up to 10 (about
    5 s at most), same thread count as the GEMM baseline."""
    from oracle import torch_ref
    from hf_kernels_helion_amd.finegrained_fp8_helion import synthetic
    M, N, K = 32, 4096, 14336
    x = synthetic.activations(M, K, seed=30)
    W, Bs = synthetic.weights(N, K, seed=31)
    q, s = torch_ref.act_quant(x, 128)
    torch_ref.dequant_matmul(q, W, s, Bs)  # warmup
    tq, tg = [], []
    t_start = time.perf_counter()
    while len(tg) < 10 and (time.perf_counter() - t_start) < 5.0:
        t0 = time.perf_counter()
        q, s = torch_ref.act_quant(x, 128)
        t1 = time.perf_counter()
        torch_ref.dequant_matmul(q, W, s, Bs)
        tg.append(time.perf_counter() - t1)
        tq.append(t1 - t0)
    aq, gm = sum(tq) / len(tq), sum(tg) / len(tg)
    byt = 2.0 * M * K + N * K + 4.0 * (N // 128) * (K // 128) + 2.0 * M * N
    return {"us": round((aq + gm) * 1e6, 1), "GB/s": round(byt / (aq + gm) / 1e9, 2),
            "act_quant_us": round(aq * 1e6, 1), "steps": len(tg)}


def load_traffic(key):
    f = ROOT / "profiles" / "traffic.json"
    if not f.exists():
        return None
    try:
        return json.loads(f.read_text()).get(key)
    except Exception:
        return None


def main():
    args = parse()
    if args.gpus != 1:
        print(f"bench.py measures one GPU only: --gpus {args.gpus} is not supported "
              "(across GPUs act-quant "
              "would shard by rows and the GEMM by output columns, or by K with one "
              "all-reduce of the output; that path is not built)", file=sys.stderr)
        sys.exit(2)

    import torch
    from hf_kernels_helion_amd import finegrained_fp8_helion as fp8
    from hf_kernels_helion_amd.finegrained_fp8_helion import synthetic

    assert torch.cuda.is_available(), "bench.py needs a ROCm GPU"
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    steps, warmup = args.steps, args.warmup

    if args.only:
        run_only(args.only, steps, warmup, torch, fp8, synthetic, dev)
        return

    # ---- headline: 4096x4096x8192 --------------------------------------
    M, N, K = 4096, 4096, 8192
    log(f"generating inputs {M}x{N}x{K}")
    x = synthetic.activations(M, K)
    W, Bs = synthetic.weights(N, K)
    Ad, As = fp8.act_quant(x.to(dev), 128)
    Bd, Bsd = W.to(dev), Bs.to(dev)
    flops = 2.0 * M * N * K

    def step():
        return fp8.w8a8_block_fp8_matmul(Ad, Bd, As, Bsd, [128, 128], torch.bfloat16)

    for _ in range(warmup):
        step()
    torch.cuda.synchronize()
    st = torch.cuda.current_stream()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    e0.record(st)
    for _ in range(steps):
        step()
    e1.record(st)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    ms = e0.elapsed_time(e1) / steps
    value = flops / (ms * 1e-3) / 1e12
    log(f"headline: {ms * 1e3:.1f} us/step, {value:.1f} TFLOP/s (wall {wall:.3f}s)")

    out = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    run, _ws = gemm_launcher(Ad, Bd, As, Bsd, out, torch)
    k_ms = time_events(run, steps, warmup, torch)
    achieved = flops / (k_ms * 1e-3) / 1e12
    log(f"kernel: {k_ms * 1e3:.1f} us/launch, {achieved:.1f} TFLOP/s "
        f"({100 * achieved / PEAK_FP8_TFLOPS:.1f}% of FP8 peak)")
    torch.testing.assert_close(out.float(), step().float(), rtol=0, atol=0)

    result = {
        "metric": METRIC,
        "value": round(value, 2),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": steps,
        "warmup": warmup,
        "ms_per_step": round(ms, 5),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp8_e4m3fn x fp8_e4m3fn -> fp32 acc -> bf16",
        "data": "synthetic: A~N(0,1) bf16 act-quantised per 1x128, W~N(0,0.02) quantised per "
                "128x128 block, seeds 1234/5678",
        "config": {"workload": "block-FP8 GEMM M=4096 N=4096 K=8192 (BASELINE configs[2])",
                   "M": M, "N": N, "K": K, "block_size": [128, 128], "out_dtype": "bf16",
                   "pct_fp8_peak": round(100 * value / PEAK_FP8_TFLOPS, 2)},
        "roofline": {
            "bound": "mfma",
            "achieved": round(achieved, 2),
            "peak": PEAK_FP8_TFLOPS,
            "unit": "TFLOP/s",
            "frac": round(achieved / PEAK_FP8_TFLOPS, 4),
            "traffic": load_traffic("gemm_4096x4096x8192"),
            "kernel": "gemm_pipe256_kernel",
            "launch_us": round(k_ms * 1e3, 2),
        },
    }

    if not args.no_secondary:
        result["secondary"] = secondary(torch, fp8, synthetic, dev)

    if not args.no_cpu_baseline:
        log("cpu baseline ...")
        result["cpu_baseline"] = cpu_baseline(Ad.cpu(), Bd.cpu(), As.cpu(), Bsd.cpu(), torch)
        log(f"cpu baseline: {result['cpu_baseline']['value']:.3f} TFLOP/s")
    else:
        result["cpu_baseline"] = None
    print(json.dumps(result), flush=True)


def _gpu_weights(N, K, seed, dev, torch, synthetic, block_n=128):
    g = torch.Generator(device=dev).manual_seed(seed)
    W = torch.randn(N, K, generator=g, device=dev) * 0.02
    return synthetic.quantize_weight_blockwise(W, block_n, 128)


def _gpu_acts(M, K, seed, dev, torch):
    g = torch.Generator(device=dev).manual_seed(seed)
    return torch.randn(M, K, generator=g, device=dev).to(torch.bfloat16)


def secondary(torch, fp8, synthetic, dev):
    res = {}
    # act-quant 4096x8192; 4 input/output sets (384 MB) rotate past the 256 MB MALL
    M, K = 4096, 8192
    xs = [_gpu_acts(M, K, 10 + i, dev, torch) for i in range(4)]
    it = [0]

    def aq():
        i = it[0] = (it[0] + 1) % 4
        return fp8.act_quant(xs[i], 128)
    ms_eager = time_events(aq, 200, 200, torch)
    # Eight launches (each input set twice) captured in a HIP graph: replays
    # cost GPU time only, without the per-op host dispatch between launches.
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            [fp8.act_quant(xs[i % 4], 128) for i in range(8)]
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        gouts = [fp8.act_quant(xs[i % 4], 128) for i in range(8)]
    graph.replay()
    eager = [fp8.act_quant(xs[i], 128) for i in range(4)]
    torch.cuda.synchronize()
    assert all(torch.equal(g[0].view(torch.uint8), e[0].view(torch.uint8)) and torch.equal(g[1], e[1])
               for g, e in zip(gouts, eager + eager)), "act_quant replay differs"
    # five windows of 50 replays after 20 warm-up replays; the median window
    windows = [time_events(graph.replay, 50, 20 if w == 0 else 0, torch) / 8 for w in range(5)]
    ms = sorted(windows)[2]
    del graph, gouts, eager
    byt = 3.0 * M * K + 4.0 * M * K / 128
    res["act_quant_4096x8192"] = {"us": round(ms * 1e3, 2), "GB/s": round(byt / ms / 1e6, 1),
                                  "pct_hbm_peak": round(100 * byt / ms / 1e6 / PEAK_HBM_GBS, 1),
                                  "eager_us": round(ms_eager * 1e3, 2),
                                  "windows_us": [round(w * 1e3, 2) for w in windows],
                                  "includes": "HIP-graph replay of 8 launches over 4 input "
                                              "sets (384 MB, past the 256 MB MALL); median of "
                                              "5 windows of 50 replays"}
    log(f"act_quant: {res['act_quant_4096x8192']}")
    del xs

    # decode 32x4096x14336 with act-quant in-op; 5 weight copies (294 MB)
    M, N, K = 32, 4096, 14336
    ws_ = [_gpu_weights(N, K, 20 + i, dev, torch, synthetic) for i in range(5)]
    xd = _gpu_acts(M, K, 30, dev, torch)
    it[0] = 0

    def dec():
        i = it[0] = (it[0] + 1) % 5
        q, s = fp8.act_quant(xd, 128)
        return fp8.w8a8_block_fp8_matmul(q, ws_[i][0], s, ws_[i][1], [128, 128], torch.bfloat16)
    ms_eager = time_events(dec, 50, 5, torch)

    # The same five steps captured once in a HIP graph (how a decode loop is
    # served): replays cost GPU time only, without per-op host dispatch.
    # Two forms: the op that quantises in-op (act_quant_w8a8_block_fp8_matmul:
    # one kernel quantises the bf16 rows inside the decode GEMM, then the
    # split-K sum), which is the C4 step, and act_quant then the GEMM (two
    # ops) beside it; every replay equals the eager two-op result bit for bit.
    def dec_two_op():
        outs = []
        for i in range(5):
            q, s = fp8.act_quant(xd, 128)
            outs.append(fp8.w8a8_block_fp8_matmul(q, ws_[i][0], s, ws_[i][1], [128, 128],
                                                  torch.bfloat16))
        return outs

    def dec_fused():
        return [fp8.act_quant_w8a8_block_fp8_matmul(xd, ws_[i][0], ws_[i][1], [128, 128],
                                                    torch.bfloat16) for i in range(5)]

    def graph_time(fn, ref):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(3):
                fn()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            gouts = fn()
        for _ in range(2):  # every replay equals the eager two-op result
            graph.replay()
            eager = ref()
            torch.cuda.synchronize()
            assert all(torch.equal(x_, y_) for x_, y_ in zip(gouts, eager)), "replay differs"
        # 200 replays (1000 steps) after 40: the step time at a steady clock
        # (100 steps after 5 replays read ~0.7 us higher), ~20 ms of GPU time
        t = time_events(graph.replay, 200, 40, torch) / 5
        del graph, gouts
        return t
    ms_two = graph_time(dec_two_op, dec_two_op)
    ms = graph_time(dec_fused, dec_two_op)
    byt = 2.0 * M * K + N * K + 4.0 * (N // 128) * (K // 128) + 2.0 * M * N
    res["decode_32x4096x14336"] = {"us": round(ms * 1e3, 2), "GB/s": round(byt / ms / 1e6, 1),
                                   "pct_hbm_peak": round(100 * byt / ms / 1e6 / PEAK_HBM_GBS, 1),
                                   "two_op_us": round(ms_two * 1e3, 2),
                                   "eager_two_op_us": round(ms_eager * 1e3, 2),
                                   "includes": "bf16 activations in, quantised in-op: "
                                               "act_quant_w8a8_block_fp8_matmul (one kernel "
                                               "+ split-K sum); two_op_us = act_quant then "
                                               "the GEMM; HIP-graph replay of 5 steps over 5 "
                                               "weight copies"}
    log(f"decode: {res['decode_32x4096x14336']}")

    # The same weights at one activation row (batch-1 decode): the op runs the
    # skinny GEMM with the act-quant inside it; act_quant then the GEMM beside.
    x1 = _gpu_acts(1, K, 31, dev, torch)

    def one_fused():
        return [fp8.act_quant_w8a8_block_fp8_matmul(x1, ws_[i][0], ws_[i][1], [128, 128],
                                                    torch.bfloat16) for i in range(5)]

    def one_two_op():
        outs = []
        for i in range(5):
            q, s = fp8.act_quant(x1, 128)
            outs.append(fp8.w8a8_block_fp8_matmul(q, ws_[i][0], s, ws_[i][1], [128, 128],
                                                  torch.bfloat16))
        return outs
    ms1 = graph_time(one_fused, one_two_op)
    ms1_two = graph_time(one_two_op, one_two_op)
    byt1 = 2.0 * K + N * K + 4.0 * (N // 128) * (K // 128) + 2.0 * N
    res["decode_1x4096x14336"] = {"us": round(ms1 * 1e3, 2),
                                  "GB/s": round(byt1 / ms1 / 1e6, 1),
                                  "pct_hbm_peak": round(100 * byt1 / ms1 / 1e6 / PEAK_HBM_GBS, 1),
                                  "two_op_us": round(ms1_two * 1e3, 2),
                                  "includes": "one activation row, quantised in-op (one kernel); "
                                              "two_op_us = act_quant then the GEMM; HIP-graph "
                                              "replay of 5 steps over the same 5 weight copies"}
    log(f"decode M=1: {res['decode_1x4096x14336']}")
    del ws_

    for name, (M, N, K) in {"medium_2048x2048x4096": (2048, 2048, 4096),
                            "small_512x512x2048": (512, 512, 2048)}.items():
        W, Bs = _gpu_weights(N, K, 40, dev, torch, synthetic)
        q, s = fp8.act_quant(_gpu_acts(M, K, 41, dev, torch), 128)
        # warm-up by GPU time, as for the harness shapes below: after the
        # HBM-bound decode legs the shader clock ramps over ~10 ms of MFMA load
        ms = time_steady(lambda: fp8.w8a8_block_fp8_matmul(q, W, s, Bs, [128, 128],
                                                           torch.bfloat16), 50, torch)
        tf = 2.0 * M * N * K / ms / 1e9
        res[name] = {"us": round(ms * 1e3, 2), "TFLOP/s": round(tf, 1),
                     "pct_fp8_peak": round(100 * tf / PEAK_FP8_TFLOPS, 1)}
        log(f"{name}: {res[name]}")

    # the reference harness's own input recipe (scripts/rebench_llm.py:128-131:
    # randn*0.3 -> e4m3fn operands, U(0.5,1) scales) over the reference's seven
    # fp8 tuning shapes (scripts/aot_tune.py:134-136; C1-C3 among them), beside
    # the reference's published B200 Helion figures where it has them
    # (results/triton_aot/fp8.json:2-28; other hardware, context only)
    b200 = {(512, 512, 2048): 16.5, (1024, 1024, 2048): None, (2048, 2048, 4096): 199.1,
            (4096, 2048, 4096): None, (4096, 4096, 8192): 187.4, (8192, 4096, 8192): None,
            (8192, 8192, 8192): None}
    harness = {}
    for (M, N, K), ref_tf in b200.items():
        A, B, As, Bs = [t.to(dev) for t in synthetic.harness_operands(M, N, K, seed=0)]
        # warm-up by GPU time: the shader clock ramps over ~10 ms of MFMA load
        ms = time_steady(lambda: fp8.w8a8_block_fp8_matmul(A, B, As, Bs, [128, 128],
                                                           torch.bfloat16), 50, torch)
        tf = 2.0 * M * N * K / ms / 1e9
        harness[f"{M}x{N}x{K}"] = {"us": round(ms * 1e3, 2), "TFLOP/s": round(tf, 1),
                                   "pct_fp8_peak": round(100 * tf / PEAK_FP8_TFLOPS, 1)}
        if ref_tf is not None:
            harness[f"{M}x{N}x{K}"]["reference_b200_helion_TFLOP/s"] = ref_tf
        del A, B, As, Bs
    res["harness_inputs"] = harness
    log(f"harness inputs: {harness}")

    # Context for the fraction of peak: the vendor library's plain fp8 GEMM
    # (torch._scaled_mm -> hipBLASLt, one per-tensor scale, no per-K-block
    # scale products) on the same operand bytes. It does less arithmetic than
    # the block-scaled path, so it bounds from above what a block-scaled
    # kernel with the same tiles can reach on this chip under its power limit.
    vendor = {}
    one = torch.ones((), device=dev)
    for (M, N, K) in ((4096, 4096, 8192), (2048, 2048, 4096)):
        x_ = _gpu_acts(M, K, 70, dev, torch)
        A_, As_ = fp8.act_quant(x_, 128)
        W_, Bs_ = _gpu_weights(N, K, 71, dev, torch, synthetic)
        try:
            f_v = lambda: torch._scaled_mm(A_, W_.t(), scale_a=one, scale_b=one,
                                           out_dtype=torch.bfloat16)
            ms_v = time_steady(f_v, 50, torch)
        except Exception as e:  # the vendor op is context only
            vendor[f"{M}x{N}x{K}"] = {"error": str(e)[:120]}
            continue
        ms_b = time_steady(lambda: fp8.w8a8_block_fp8_matmul(A_, W_, As_, Bs_, [128, 128],
                                                             torch.bfloat16), 50, torch)
        fl = 2.0 * M * N * K
        vendor[f"{M}x{N}x{K}"] = {"hipblaslt_plain_fp8_us": round(ms_v * 1e3, 2),
                                  "hipblaslt_plain_fp8_TFLOP/s": round(fl / ms_v / 1e9, 1),
                                  "block_fp8_us": round(ms_b * 1e3, 2),
                                  "block_fp8_TFLOP/s": round(fl / ms_b / 1e9, 1)}
        del x_, A_, As_, W_, Bs_
    res["vendor_plain_fp8_context"] = vendor
    log(f"vendor plain fp8 context: {vendor}")

    # deep-gemm layout (one weight scale per row and K-block, block_n = 1):
    # the headline shape and the decode shape (5 weight copies, as above)
    from hf_kernels_helion_amd import deep_gemm_helion as dg
    for name, (M, N, K, copies) in {"deep_gemm_4096x4096x8192": (4096, 4096, 8192, 1),
                                    "deep_gemm_32x4096x14336": (32, 4096, 14336, 5)}.items():
        wl = [_gpu_weights(N, K, 60 + i, dev, torch, synthetic, block_n=1)
              for i in range(copies)]
        q, s = fp8.act_quant(_gpu_acts(M, K, 61, dev, torch), 128)
        it[0] = 0

        def dgf():
            i = it[0] = (it[0] + 1) % copies
            return dg.gemm_fp8_fp8_bf16_nt(q, wl[i][0], s, wl[i][1], 128)
        ms = time_steady(dgf, 50, torch, min_warmup=20)
        tf = 2.0 * M * N * K / ms / 1e9
        byt = M * K + N * K + 4.0 * (M + N) * (K // 128) + 2.0 * M * N
        res[name] = {"us": round(ms * 1e3, 2), "TFLOP/s": round(tf, 1),
                     "pct_fp8_peak": round(100 * tf / PEAK_FP8_TFLOPS, 1),
                     "GB/s": round(byt / ms / 1e6, 1),
                     "pct_hbm_peak": round(100 * byt / ms / 1e6 / PEAK_HBM_GBS, 1)}
        log(f"{name}: {res[name]}")
        del wl

    # offline weight-block quantiser, fp32 [4096, 14336] -> e4m3fn + scales;
    # two inputs (470 MB) rotate past the MALL
    N, K = 4096, 14336
    wsrc = [torch.randn(N, K, device=dev) * 0.02 for _ in range(2)]
    it[0] = 0

    def wq():
        i = it[0] = (it[0] + 1) % 2
        return fp8.quantize_weight(wsrc[i])
    ms = time_events(wq, 20, 5, torch)
    byt = 4.0 * N * K + N * K + 4.0 * (N // 128) * (K // 128)
    res["weight_quant_4096x14336_f32"] = {"us": round(ms * 1e3, 2),
                                          "GB/s": round(byt / ms / 1e6, 1),
                                          "pct_hbm_peak": round(100 * byt / ms / 1e6 /
                                                                PEAK_HBM_GBS, 1)}
    log(f"weight_quant: {res['weight_quant_4096x14336_f32']}")
    # the same from bf16 weights (the usual checkpoint dtype); four inputs
    # (470 MB) rotate past the MALL
    wsrc = [(torch.randn(N, K, device=dev) * 0.02).to(torch.bfloat16) for _ in range(4)]
    it[0] = 0

    def wqb():
        i = it[0] = (it[0] + 1) % 4
        return fp8.quantize_weight(wsrc[i])
    ms = time_events(wqb, 20, 5, torch)
    byt = 2.0 * N * K + N * K + 4.0 * (N // 128) * (K // 128)
    res["weight_quant_4096x14336_bf16"] = {"us": round(ms * 1e3, 2),
                                           "GB/s": round(byt / ms / 1e6, 1),
                                           "pct_hbm_peak": round(100 * byt / ms / 1e6 /
                                                                 PEAK_HBM_GBS, 1)}
    log(f"weight_quant bf16: {res['weight_quant_4096x14336_bf16']}")
    del wsrc

    # MLP chain M=3001, H=4096, I=14336
    M, H, I = 3001, 4096, 14336
    w13, s13 = _gpu_weights(2 * I, H, 50, dev, torch, synthetic)
    w2, s2 = _gpu_weights(H, I, 51, dev, torch, synthetic)
    x = _gpu_acts(M, H, 52, dev, torch)
    # warm-up by GPU time (the legs before it are HBM-bound; see time_steady)
    ms = time_steady(lambda: fp8.fp8_mlp(x, w13, s13, w2, s2), 20, torch, min_warmup=10)
    fl = 2.0 * M * (2 * I * H + H * I)
    res["mlp_chain_3001"] = {"us": round(ms * 1e3, 2), "TFLOP/s": round(fl / ms / 1e9, 1),
                             "pct_fp8_peak": round(100 * fl / ms / 1e9 / PEAK_FP8_TFLOPS, 1)}
    log(f"mlp: {res['mlp_chain_3001']}")
    # the same chain with the gate/up weight interleaved once (outside the
    # timing): the gate/up GEMM's epilogue applies SiLU·up and the act-quant
    wi, si = fp8.interleave_gate_up(w13, s13)
    y0 = fp8.fp8_mlp(x, w13, s13, w2, s2)
    y1 = fp8.fp8_mlp(x, wi, si, w2, s2, gate_up_interleaved=True)
    assert torch.equal(y0, y1), "interleaved MLP chain differs from the default chain"
    del w13, s13, y0, y1
    ms = time_steady(lambda: fp8.fp8_mlp(x, wi, si, w2, s2, gate_up_interleaved=True),
                     20, torch, min_warmup=10)
    res["mlp_chain_3001_interleaved"] = {
        "us": round(ms * 1e3, 2), "TFLOP/s": round(fl / ms / 1e9, 1),
        "pct_fp8_peak": round(100 * fl / ms / 1e9 / PEAK_FP8_TFLOPS, 1),
        "equals_default_chain": True}
    log(f"mlp interleaved: {res['mlp_chain_3001_interleaved']}")
    return res


def run_only(what, steps, warmup, torch, fp8, synthetic, dev):
    """Run one workload for profiling (rocprofv3) without the other legs."""
    shapes = {"gemm": (4096, 4096, 8192), "medium": (2048, 2048, 4096),
              "small": (512, 512, 2048), "decode": (32, 4096, 14336),
              "decode_fused": (32, 4096, 14336), "mlp_gateup": (3001, 28672, 4096),
              "mlp_down": (3001, 4096, 14336), "prefill": (2048, 4096, 4096)}
    if what in shapes:
        M, N, K = shapes[what]
        x = _gpu_acts(M, K, 41, dev, torch)
        q, s = fp8.act_quant(x, 128)
        if what in ("decode", "decode_fused"):
            # five weight copies (294 MB) rotate past the 256 MB MALL, as in
            # the bench leg
            ws_ = [_gpu_weights(N, K, 20 + i, dev, torch, synthetic) for i in range(5)]
            it = [0]

            def fn():
                i = it[0] = (it[0] + 1) % 5
                if what == "decode_fused":
                    return fp8.act_quant_w8a8_block_fp8_matmul(x, ws_[i][0], ws_[i][1],
                                                               [128, 128], torch.bfloat16)
                q2, s2 = fp8.act_quant(x, 128)
                return fp8.w8a8_block_fp8_matmul(q2, ws_[i][0], s2, ws_[i][1], [128, 128],
                                                 torch.bfloat16)
        else:
            W, Bs = _gpu_weights(N, K, 40, dev, torch, synthetic)
            fn = lambda: fp8.w8a8_block_fp8_matmul(q, W, s, Bs, [128, 128], torch.bfloat16)
    elif what.startswith("decode_graph"):
        # the bench leg's decode step (five weight copies) as a HIP graph of
        # five steps, replayed --steps times: the in-op quantising op
        # (one kernel + split-K sum), or act_quant then the GEMM
        # (decode_graph[_two_op]); the same at one row
        # (decode_graph_m1[_two_op], 1x4096x14336: the skinny one-kernel
        # path) and at one row of a gate/up projection
        # (decode_graph_m1_wide[_two_op], 1x28672x4096: the small-grid one)
        two_op = what.endswith("_two_op")
        base = what[:-len("_two_op")] if two_op else what
        shapes_ = {"decode_graph": (32, 4096, 14336), "decode_graph_m1": (1, 4096, 14336),
                   "decode_graph_m1_wide": (1, 28672, 4096)}
        if base not in shapes_:
            raise SystemExit(f"unknown --only {what}")
        M, N, K = shapes_[base]
        ws_ = [_gpu_weights(N, K, 20 + i, dev, torch, synthetic) for i in range(5)]
        xd = _gpu_acts(M, K, 30, dev, torch)

        def five():
            for i in range(5):
                if not two_op:
                    fp8.act_quant_w8a8_block_fp8_matmul(xd, ws_[i][0], ws_[i][1], [128, 128],
                                                        torch.bfloat16)
                    continue
                q, s = fp8.act_quant(xd, 128)
                fp8.w8a8_block_fp8_matmul(q, ws_[i][0], s, ws_[i][1], [128, 128],
                                          torch.bfloat16)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(3):
                five()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            five()
        ms = time_events(graph.replay, steps, warmup, torch) / 5
        log(f"{what}: {ms * 1e3:.2f} us/step over {5 * steps} graph-replayed steps")
        return
    elif what in ("deep_gemm", "deep_decode"):
        from hf_kernels_helion_amd import deep_gemm_helion as dg
        M, N, K, copies = (4096, 4096, 8192, 1) if what == "deep_gemm" else (32, 4096, 14336, 5)
        wl = [_gpu_weights(N, K, 60 + i, dev, torch, synthetic, block_n=1) for i in range(copies)]
        q, s = fp8.act_quant(_gpu_acts(M, K, 61, dev, torch), 128)
        it = [0]

        def fn():
            i = it[0] = (it[0] + 1) % copies
            return dg.gemm_fp8_fp8_bf16_nt(q, wl[i][0], s, wl[i][1], 128)
    elif what == "copy":
        # calibration for the rocprofv3 FETCH_SIZE/WRITE_SIZE counters: a
        # plain 256 MiB device-to-device copy
        src = torch.empty(256 << 20, dtype=torch.uint8, device=dev)
        dst = torch.empty_like(src)
        fn = lambda: dst.copy_(src)
    elif what in ("weight_quant", "weight_quant_bf16"):
        # as the bench legs: two fp32 or four bf16 inputs (470 MB) rotate past
        # the MALL
        if what == "weight_quant":
            wsrc = [torch.randn(4096, 14336, device=dev) * 0.02 for _ in range(2)]
        else:
            wsrc = [(torch.randn(4096, 14336, device=dev) * 0.02).to(torch.bfloat16)
                    for _ in range(4)]
        it = [0]

        def fn():
            i = it[0] = (it[0] + 1) % len(wsrc)
            return fp8.quantize_weight(wsrc[i])
    elif what == "act_quant":
        # four input sets (384 MB with outputs) rotate past the MALL, as in
        # the bench leg
        xs = [_gpu_acts(4096, 8192, 10 + i, dev, torch) for i in range(4)]
        it = [0]

        def fn():
            i = it[0] = (it[0] + 1) % 4
            return fp8.act_quant(xs[i], 128)
    elif what == "mlp":
        M, H, I = 3001, 4096, 14336
        w13, s13 = _gpu_weights(2 * I, H, 50, dev, torch, synthetic)
        w2, s2 = _gpu_weights(H, I, 51, dev, torch, synthetic)
        x = _gpu_acts(M, H, 52, dev, torch)
        fn = lambda: fp8.fp8_mlp(x, w13, s13, w2, s2)
    elif what == "mlp_il":
        M, H, I = 3001, 4096, 14336
        w13, s13 = _gpu_weights(2 * I, H, 50, dev, torch, synthetic)
        wi, si = fp8.interleave_gate_up(w13, s13)
        del w13, s13
        w2, s2 = _gpu_weights(H, I, 51, dev, torch, synthetic)
        x = _gpu_acts(M, H, 52, dev, torch)
        fn = lambda: fp8.fp8_mlp(x, wi, si, w2, s2, gate_up_interleaved=True)
    elif what == "shapes":
        # the block-FP8 GEMM over LLM projection shapes against the vendor's
        # plain fp8 GEMM (torch._scaled_mm -> hipBLASLt, one per-tensor
        # scale) on the same operand bytes, weights MALL-resident, steady
        # clock, both as HIP-graph replays of 10 calls (GPU time without the
        # host dispatch): an upper bound for the planner's tile choices
        one = torch.ones((), device=dev)

        def graph_time_events(fn, n, w, torch):
            for _ in range(3):
                fn()
            torch.cuda.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                for _ in range(10):
                    fn()
            for _ in range(max(1, w // 10)):
                g.replay()
            torch.cuda.synchronize()
            e0 = torch.cuda.Event(enable_timing=True)
            e1 = torch.cuda.Event(enable_timing=True)
            reps = max(1, n // 10)
            e0.record()
            for _ in range(reps):
                g.replay()
            e1.record()
            torch.cuda.synchronize()
            return e0.elapsed_time(e1) / (10 * reps)
        log(f"{'M':>5} {'N':>6} {'K':>6} {'block_us':>9} {'vendor_us':>10} {'ratio':>6}")
        # (4096, 11008): LLaMA-2-7B's down projection, 86 K-blocks (scale
        # windows by 4-byte lanes)
        for (N, K) in ((4096, 4096), (28672, 4096), (4096, 14336), (6144, 4096), (8192, 8192),
                       (2048, 7168), (7168, 2048), (4096, 11008)):
            W, Bs = _gpu_weights(N, K, 80, dev, torch, synthetic)
            for M in (256, 512, 1024, 2048, 4096, 8192):
                A, As = fp8.act_quant(_gpu_acts(M, K, 81, dev, torch), 128)
                f_b = lambda: fp8.w8a8_block_fp8_matmul(A, W, As, Bs, [128, 128],
                                                        torch.bfloat16)
                f_v = lambda: torch._scaled_mm(A, W.t(), scale_a=one, scale_b=one,
                                               out_dtype=torch.bfloat16)
                n = max(5, min(steps, int(3e-3 / (2.0 * M * N * K / 2e15))))
                tb = min(graph_time_events(f_b, n, warmup, torch) for _ in range(2))
                tv = min(graph_time_events(f_v, n, warmup, torch) for _ in range(2))
                log(f"{M:5d} {N:6d} {K:6d} {tb * 1e3:9.1f} {tv * 1e3:10.1f} {tb / tv:6.2f}")
                del A, As
            del W, Bs
        return
    elif what == "shapes_streamed":
        # decode and small-prefill shapes (M <= 256) with the weights streamed
        # from HBM, as in a forward pass over a model's layers: each call of a
        # HIP graph reads its own weight copy (about 600 MB of copies, past
        # the 256 MB MALL). The block-FP8 GEMM against the vendor's plain fp8
        # GEMM (torch._scaled_mm -> hipBLASLt, one per-tensor scale) on the
        # same operand bytes; per call, best of four timed replays
        one = torch.ones((), device=dev)

        def graph_us(calls):
            for c in calls:
                c()
            torch.cuda.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                for c in calls:
                    c()
            for _ in range(max(1, warmup // 10)):
                g.replay()
            torch.cuda.synchronize()
            best = float("inf")
            for _ in range(4):
                e0 = torch.cuda.Event(enable_timing=True)
                e1 = torch.cuda.Event(enable_timing=True)
                e0.record()
                for _ in range(5):
                    g.replay()
                e1.record()
                torch.cuda.synchronize()
                best = min(best, e0.elapsed_time(e1) * 1e3 / (5 * len(calls)))
            return best

        log(f"{'M':>5} {'N':>6} {'K':>6} {'copies':>6} {'block_us':>9} {'vendor_us':>10} {'ratio':>6}")
        for (N, K) in ((4096, 4096), (28672, 4096), (4096, 14336), (6144, 4096), (8192, 8192),
                       (7168, 2048), (7168, 8192), (11008, 4096)):
            W0, Bs = _gpu_weights(N, K, 90, dev, torch, synthetic)
            copies = max(2, (600 << 20) // (N * K))
            Ws = [W0] + [W0.clone() for _ in range(copies - 1)]
            for M in (1, 16, 32, 64, 128, 256):
                A, As = fp8.act_quant(_gpu_acts(M, K, 91, dev, torch), 128)
                tb = graph_us([
                    (lambda W=W: fp8.w8a8_block_fp8_matmul(A, W, As, Bs, [128, 128],
                                                           torch.bfloat16)) for W in Ws])
                try:
                    tv = graph_us([
                        (lambda W=W: torch._scaled_mm(A, W.t(), scale_a=one, scale_b=one,
                                                      out_dtype=torch.bfloat16)) for W in Ws])
                except RuntimeError:
                    tv = float("nan")  # the vendor GEMM rejects this M
                log(f"{M:5d} {N:6d} {K:6d} {copies:6d} {tb:9.1f} {tv:10.1f} {tb / tv:6.2f}")
                del A, As
            del W0, Ws, Bs
            torch.cuda.empty_cache()
        return
    else:
        raise SystemExit(f"unknown --only {what}")
    ms = time_events(fn, steps, warmup, torch)
    log(f"{what}: {ms * 1e3:.2f} us/step over {steps} steps")


if __name__ == "__main__":
    main()
