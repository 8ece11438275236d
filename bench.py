"""Benchmark of the gfx950 executor's hot path (one MI355X).

Workload: the W8A8 GEMM -- activations f32
[4096, 4096] ~ N(0,1) quantized per row to int8, weights [4096, 4096]
~ N(0, 0.02) quantized per output channel (packed once, frozen), int32
accumulation, f32 dequant.  One step = quantize the activations + the int8
GEMM with its dequant epilogue, inputs resident in HBM.  ``value`` is the
whole job's throughput in int8 tera-ops per second (2*M*N*K per step).

The JSON line also carries:
  roofline      the dominant kernel (the int8 MFMA GEMM): algorithmic ops
                per launch / its mean duration measured here with HIP events
                around back-to-back launches on the stream it runs on,
                against MI355X's dense int8 peak (5.0 POP/s); traffic from
                profiles/ when measured;
  cpu_baseline  the oracle's W8A8 (scalar C, 1 thread) timed on this host on
                a bounded row sample of the same GEMM;
  extra         the decode-shaped GEMM (M = 32), causal attention fwd+bwd at
                BASELINE config 3, softmax-xent and AdamW, each with its
                roofline fraction; and the LoRA training steps through the
                plan engine: the MLP (configs[0], us/step and rows/s) and the
                12-layer decoder (configs[3], tokens/s relaxed and exact, with
                the step's algorithmic TFLOP/s against the bf16 MFMA peak).

--gpus N with N > 1 exits: this build measures one GPU.
"""
from __future__ import annotations

import argparse
import importlib
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_INT8_TOPS = 5000.0      # MI355X dense int8, POP/s x 1000
PEAK_BF16_TFLOPS = 2500.0    # dense bf16
PEAK_FP32_TFLOPS = 157.3     # fp32 MFMA
PEAK_HBM_GBS = 8000.0        # HBM3E


def parse():
    p = argparse.ArgumentParser()
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=50)
    p.add_argument("--warmup", type=int, default=5)
    p.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    p.add_argument("--no-extra", action="store_true", help="skip the secondary workloads")
    p.add_argument("--pmc-probe", action="store_true",
                   help="for rocprofv3 --pmc runs: one W8A8 step plus a 256 MiB device copy "
                        "(the counter calibration: a copy's known bytes)")
    p.add_argument("--attn-probe", action="store_true",
                   help="for rocprofv3 runs: BASELINE configs[2] attention fwd+bwd, bf16 x3, f32 x1")
    p.add_argument("--lora-probe", nargs="?", const="c4", choices=["c1", "c4", "c5"],
                   help="for rocprofv3 runs: BASELINE configs[3] (c4) or configs[4] (c5) decoder "
                        "LoRA plan, one staged step then resident steps (relaxed family)")
    return p.parse_args()


def lora_probe(which: str):
    """BASELINE configs[0] (c1), configs[3] (c4) or configs[4] (c5) through
    the plan engine for the profilers: build the LoRA plan, one staged step,
    then resident steps (200 for c1, five for c4, two for c5)."""
    import numpy as np
    import torch
    hip = importlib.import_module("see-ai_amd.hip")
    pw = importlib.import_module("see-ai_amd.planwriter")
    if which == "c1":
        eng = hip.Engine(pw.mlp_lora(hip.plan_self_hash).blob)
        eng.train_step(pw.normal(1, (32, 256)), pw.uniform_ints(2, 32, 256))
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(200):
            loss = eng.train_resident()
        dt = (time.perf_counter() - t0) / 200
        eng.close()
        print(f"lora probe: LoRA MLP (c1), 200 resident steps, {dt * 1e6:.1f} us/step, "
              f"loss {loss:.5f}", flush=True)
        return 0
    if which == "c5":
        img, T, n = pw.decoder_q8_lora(hip.plan_self_hash, relaxed=True), 4 * 2048, 2
    else:
        img, T, n = pw.decoder_lora(hip.plan_self_hash, relaxed=True), 8 * 1024, 5
    print(f"lora probe {which}: plan built", flush=True)
    eng = hip.Engine(img.blob)
    eng.set_attention_bf16(True)  # both configs train in bf16 activations
    del img
    tok = pw.uniform_ints(9, T + 1, 32000)
    eng.train_step(tok[:T].copy().view(np.float32), tok[1:].copy())
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(n):
        loss = eng.train_resident()
    dt = (time.perf_counter() - t0) / n
    fused, dropped = eng.fused_dispatches(), eng.dropped_stores()
    eng.close()
    print(f"lora probe: decoder LoRA ({which}) relaxed, {n} resident steps, "
          f"{dt * 1e3:.1f} ms/step, {T / dt:.0f} tokens/s, loss {loss:.4f}, "
          f"{fused} fused dispatches, {dropped} dead stores dropped", flush=True)
    return 0


def pmc_probe():
    """One quantize + GEMM at the bench shape, then a plain 256 MiB copy whose
    FETCH_SIZE / WRITE_SIZE readings calibrate the counters' byte scale."""
    import torch
    hip = importlib.import_module("see-ai_amd.hip")
    ctx = hip.Context(0)
    ctx.use_torch_stream()
    M = N = K = 4096
    X = torch.randn((M, K), device="cuda")
    W = torch.randn((K, N), device="cuda") * 0.02
    QA = torch.empty((M, K), dtype=torch.int8, device="cuda")
    sa = torch.empty(M, device="cuda")
    QWt = torch.empty((N, K), dtype=torch.int8, device="cuda")
    sw = torch.empty(N, device="cuda")
    C = torch.empty((M, N), device="cuda")
    ctx.call("seeai_w8a8_pack_weights", W.data_ptr(), QWt.data_ptr(), sw.data_ptr(), K, N)
    for _ in range(3):
        ctx.call("seeai_w8a8_quantize_rows", X.data_ptr(), QA.data_ptr(), sa.data_ptr(), M, K)
        ctx.call("seeai_w8a8_gemm", QA.data_ptr(), sa.data_ptr(), QWt.data_ptr(), sw.data_ptr(),
                 C.data_ptr(), None, M, N, K)
    src = torch.empty(64 * 1024 * 1024, device="cuda")  # 256 MiB
    dst = torch.empty_like(src)
    for _ in range(3):
        dst.copy_(src)
    torch.cuda.synchronize()
    ctx.close()
    print("pmc probe: 3 x (quantize 4096x4096 + W8A8 GEMM 4096^3), 3 x copy 256 MiB", flush=True)
    return 0


def attention_step(ctx, dt, q, k, v, do, o, st, dq, dk, dv, B, S, H, d, parts=None):
    """One causal attention fwd + bwd as a plan runs it: forward, dQ, then
    dK and dV as one fused pass (an adjacent dK / dV pair fuses in a range,
    in the relaxed and the exact family).  `parts` picks a subset ("fwd",
    "dq", "dkdv") for per-kernel timing."""
    P = lambda t: t.data_ptr()
    parts = parts or ("fwd", "dq", "dkdv")
    if "fwd" in parts:
        ctx.call("seeai_attn_fwd", dt, P(q), P(k), P(v), P(o), P(st), B, S, H, d, None)
    if "dq" in parts:
        ctx.call("seeai_attn_dq", dt, P(q), P(k), P(v), P(do), P(st), P(dq), B, S, H, d)
    if "dkdv" in parts:
        ctx.call("seeai_attn_dkdv" if dt else "seeai_attn_dkdv_f32", P(q), P(k), P(v), P(do),
                 P(st), P(dk), P(dv), B, S, H, d)


def attention_step_bf16(ctx, q, k, v, do, o, st, dq, dk, dv, B, S, H, d, parts=None):
    """One causal attention fwd + bwd on bf16 operands held in HBM as bf16
    (what a model trained in bf16 activations holds): the forward, dQ with
    the stats delta, and the fused dK / dV pass."""
    P = lambda t: t.data_ptr()
    parts = parts or ("fwd", "dq", "dkdv")
    if "fwd" in parts:
        ctx.call("seeai_attn_fwd_bf16", P(q), P(k), P(v), P(o), P(st), B, S, H, d, None)
    if "dq" in parts:
        ctx.call("seeai_attn_dq_bf16", P(q), P(k), P(v), P(do), P(st), P(dq), B, S, H, d)
    if "dkdv" in parts:
        ctx.call("seeai_attn_dkdv_bf16", P(q), P(k), P(v), P(do), P(st), P(dk), P(dv), B, S, H, d)


def attn_probe():
    """BASELINE configs[2] per path for the profilers: causal attention fwd +
    dQ + dK + dV at B16 H16 S2048 d64 -- on bf16 operands held as bf16 three
    times, on f32 operands through the relaxed bf16 kernels once, exact (f32)
    once."""
    import torch
    hip = importlib.import_module("see-ai_amd.hip")
    ctx = hip.Context(0)
    ctx.use_torch_stream()
    B, S, H, d = 16, 2048, 16, 64
    g = torch.Generator(device="cuda").manual_seed(20261202)
    q, k, v, do = (torch.randn((B * S, H * d), device="cuda", generator=g) for _ in range(4))
    o, st = torch.empty_like(q), torch.empty((B * H * S, 4), device="cuda")
    dq, dk, dv = torch.empty_like(q), torch.empty_like(q), torch.empty_like(q)
    qb, kb, vb, dob = (x.to(torch.bfloat16) for x in (q, k, v, do))
    for _ in range(3):
        attention_step_bf16(ctx, qb, kb, vb, dob, o, st, dq, dk, dv, B, S, H, d)
    for dt in (1, 0):
        attention_step(ctx, dt, q, k, v, do, o, st, dq, dk, dv, B, S, H, d)
    torch.cuda.synchronize()
    ctx.close()
    print("attention probe: B16 H16 S2048 d64 causal, 3 x bf16-held fwd+bwd, 1 x relaxed bf16 on "
          "f32 operands, 1 x f32 fwd+bwd", flush=True)
    return 0


def load_traffic(name: str):
    path = os.path.join(ROOT, "profiles", "traffic.json")
    if not os.path.exists(path):
        return None
    with open(path) as f:
        return json.load(f).get(name)


def main():
    args = parse()
    if args.pmc_probe:
        return pmc_probe()
    if args.attn_probe:
        return attn_probe()
    if args.lora_probe:
        return lora_probe(args.lora_probe)
    if args.gpus != 1:
        print(f"bench.py measures one GPU; --gpus {args.gpus} is not supported by this build "
              "(the path shards by GEMM column blocks / attention (b, h) -- see DESIGN.md)",
              file=sys.stderr)
        return 2
    import numpy as np
    import torch

    hip = importlib.import_module("see-ai_amd.hip")
    torch.cuda.set_device(0)
    ctx = hip.Context(0)
    ctx.use_torch_stream()
    ev = lambda: torch.cuda.Event(enable_timing=True)  # noqa: E731

    M = N = K = 4096
    g = torch.Generator(device="cuda").manual_seed(20261201)
    X = torch.randn((M, K), device="cuda", generator=g)
    W = torch.randn((K, N), device="cuda", generator=g) * 0.02
    QA = torch.empty((M, K), dtype=torch.int8, device="cuda")
    sa = torch.empty(M, dtype=torch.float32, device="cuda")
    QWt = torch.empty((N, K), dtype=torch.int8, device="cuda")
    sw = torch.empty(N, dtype=torch.float32, device="cuda")
    C = torch.empty((M, N), dtype=torch.float32, device="cuda")
    ctx.call("seeai_w8a8_pack_weights", W.data_ptr(), QWt.data_ptr(), sw.data_ptr(), K, N)

    def quantize():
        ctx.call("seeai_w8a8_quantize_rows", X.data_ptr(), QA.data_ptr(), sa.data_ptr(), M, K)

    def gemm():
        ctx.call("seeai_w8a8_gemm", QA.data_ptr(), sa.data_ptr(), QWt.data_ptr(), sw.data_ptr(),
                 C.data_ptr(), None, M, N, K)

    for _ in range(args.warmup):
        quantize()
        gemm()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i in range(args.steps):
        quantize()
        gemm()
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    # The GEMM kernel's mean duration: HIP events (on torch's current stream,
    # the one the library launches on) around the same number of GEMM-only
    # launches back to back.
    g_start, g_end = ev(), ev()
    g_start.record()
    for i in range(args.steps):
        gemm()
    g_end.record()
    torch.cuda.synchronize()
    gemm_ms = g_start.elapsed_time(g_end) / args.steps
    # The activation quantize alone (HBM-bound: reads 4MK bytes, writes MK + 4M).
    q_start, q_end = ev(), ev()
    q_start.record()
    for i in range(args.steps):
        quantize()
    q_end.record()
    torch.cuda.synchronize()
    quant_ms = q_start.elapsed_time(q_end) / args.steps
    quant_bytes = 4 * M * K + M * K + 4 * M
    ms_per_step = wall * 1000.0 / args.steps
    ops = 2.0 * M * N * K
    value = ops / (ms_per_step * 1e-3) / 1e12
    achieved = ops / (gemm_ms * 1e-3) / 1e12

    line = {
        "metric": "int8 GEMM TOPS + LoRA train-step tokens/s on 1 MI355X; % of MFMA/HBM roofline",
        "value": round(value, 2),
        "unit": "TOPS (int8, quantize + GEMM + dequant per step)",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 5),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "int8 (int32 accumulate, f32 dequant)",
        "data": "synthetic: X ~ N(0,1), W ~ N(0,0.02), seeded on device",
        "config": {"workload": "W8A8 GEMM M=4096 K=4096 N=4096 (BASELINE configs[1])",
                   "M": M, "N": N, "K": K, "parallelism": "single GPU"},
        "roofline": {
            "kernel": "GemmI8DmaKernel<256,256,4,2,4,1,false>",
            "bound": "mfma",
            "achieved": round(achieved, 1),
            "peak": PEAK_INT8_TOPS,
            "unit": "TFLOP/s",
            "op": "int8 multiply-accumulate counted as 2 ops",
            "frac": round(achieved / PEAK_INT8_TOPS, 4),
            "algorithmic_per_launch": ops,
            "kernel_ms": round(gemm_ms, 5),
            "traffic": load_traffic("w8a8_4096"),
        },
        "quantize": {"kernel": "QuantizeRowsBlockKernel<4>", "ms": round(quant_ms, 5),
                     "bytes": quant_bytes, "GB_s": round(quant_bytes / quant_ms / 1e6, 1),
                     "hbm_frac": round(quant_bytes / quant_ms / 1e6 / PEAK_HBM_GBS, 4)},
    }

    if not args.no_cpu:
        line["cpu_baseline"] = cpu_baseline(M, N, K)
    if not args.no_extra:
        line["extra"] = extras(ctx, torch, hip)
    print(json.dumps(line), flush=True)
    ctx.close()
    return 0


def host_threads():
    """The host threads this process may use, capped at the 16 a one-GPU
    box grants (its OMP_NUM_THREADS)."""
    try:
        n = len(os.sched_getaffinity(0))
    except AttributeError:
        n = os.cpu_count() or 1
    cap = int(os.environ.get("OMP_NUM_THREADS", "16") or 16)
    return max(1, min(n, cap, 16))


def cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline(M, N, K):
    """The reported CPU baseline: the oracle (the repository's C restatement
    of the reference executor, bit-matched to it) on this host, for all five
    configs: the W8A8 step (quantize + int32 GEMM + dequant, configs[1]) on
    a row sample; the config-1 train step; one-block slices of configs[3]
    and configs[4] at full widths; configs[2]'s attention on sampled (b, h)
    units -- each at all threads and at one, on the same workload.
    Each measurement is a median of repeats after a warm-up.  The oracle's
    chunks are the reference's ParallelFor chunks, so every thread count
    computes the same bits."""
    import numpy as np
    from oracle.oracle import oracle
    orc = oracle()
    threads = host_threads()
    r = np.random.default_rng(1)

    def median_s(fn, reps, warm=True):
        if warm:
            fn()
        ts = []
        for _ in range(reps):
            t0 = time.perf_counter()
            fn()
            ts.append(time.perf_counter() - t0)
        return float(np.median(ts))

    out = {"kind": "port", "cores": threads, "host_threads_available": os.cpu_count(),
           "cpu_model": cpu_model()}
    # W8A8: weights packed once, outside the step, as on the GPU.
    W = (r.standard_normal((K, N)) * 0.02).astype(np.float32)
    QW, sw = orc.quantize_cols(W)
    w8 = {}
    for th, rows, reps in [(threads, 1024, 3), (1, 256, 1)]:
        X = r.standard_normal((rows, K)).astype(np.float32)
        orc.set_threads(th)

        def step(X=X):
            QA, sa = orc.quantize_rows(X)
            orc.gemm_w8a8(QA, sa, QW, sw)
        dt = median_s(step, reps)
        w8[th] = (2.0 * rows * N * K / dt / 1e12, rows, dt)
    out.update({"value": round(w8[threads][0], 4), "unit": "TOPS",
                "sample": f"W8A8 step on {w8[threads][1]} of the {M} activation rows (quantize + "
                          f"int32 GEMM + dequant against all {N}x{K} weights), median of 3, "
                          f"{threads} threads; CPU {out['cpu_model']}",
                "one_thread": {"value": round(w8[1][0], 4), "unit": "TOPS",
                               "sample": f"{w8[1][1]} rows, {w8[1][2]:.2f} s"}})
    # Train steps through the oracle's instruction interpreter (the CPU
    # executor's arithmetic and order).
    from tests.engine_oracle import OracleEngine
    pw = importlib.import_module("see-ai_amd.planwriter")
    hip = importlib.import_module("see-ai_amd.hip")
    steps = {}
    img = pw.mlp_lora(hip.plan_self_hash)
    x, y = pw.normal(1, (32, 256)), pw.uniform_ints(2, 32, 256)
    for th in (threads, 1):
        orc.set_threads(th)
        eng = OracleEngine(orc, img.blob)
        dt = median_s(lambda: eng.train_step(x, y), 5)
        steps[f"c1_{th}t"] = {"ms_per_step": round(dt * 1e3, 3), "rows_s": round(32 / dt, 1),
                              "threads": th}
    # configs[3] and configs[4] at full widths, one block and one sequence
    # (the whole steps are 12 blocks x 8 sequences of 1024 and 16 blocks x 4
    # sequences of 2048): tokens/s of the slice, all threads and one thread
    # on the same slice.
    slices = [("c4_slice", pw.decoder_lora,
               dict(vocab=32000, dim=768, heads=12, ffn=3072, layers=1, seq=512, batch=1, rank=8),
               "configs[3] widths (d768, 12 heads, FFN 3072, vocab 32000), 1 block"),
              ("c5_slice", pw.decoder_q8_lora,
               dict(vocab=32000, dim=2048, heads=32, ffn=5632, layers=1, seq=128, batch=1,
                    rank=16),
               "configs[4] widths (d2048, 32 heads, SiLU-gated FFN 5632, int8 base, vocab "
               "32000), 1 block")]
    for key, make, cfg, what in slices:
        seq = cfg["seq"]
        img = make(hip.plan_self_hash, relaxed=False, **cfg)
        t = pw.uniform_ints(9, seq + 1, 32000)
        xb, yb = t[:seq].copy().view(np.float32), t[1:].copy()
        for th in (threads, 1):
            orc.set_threads(th)
            eng = OracleEngine(orc, img.blob)
            # the one-thread run follows the warm all-threads one on the same plan
            dt = median_s(lambda: eng.train_step(xb, yb), 2 if th > 1 else 1, warm=th > 1)
            steps[f"{key}_{th}t"] = {"s_per_step": round(dt, 3), "tokens_s": round(seq / dt, 1),
                                     "threads": th,
                                     "sample": f"{what}, B1 x S{seq}, exact family"}
            del eng
        del img
    # causal attention fwd + bwd (the tiled family: forward, dQ,
    # dK, dV) on (b, h) units of the B16 H16 S2048 d64 grid -- every unit is
    # the same work -- scaled to the 256 units of the grid.
    S2, d2 = 2048, 64
    att = {}
    for th, units in ((threads, 4), (1, 1)):
        orc.set_threads(th)
        q2, k2, v2, do2 = (r.standard_normal((S2, units * d2)).astype(np.float32)
                           for _ in range(4))

        def attn_step():
            _, st = orc.attn_fwd_tiled(q2, k2, v2, 1, S2, units, d2)
            _, st = orc.attn_dq_tiled(q2, k2, v2, do2, st, 1, S2, units, d2)
            orc.attn_dk_tiled(q2, k2, v2, do2, st, 1, S2, units, d2)
            orc.attn_dv_tiled(q2, k2, do2, st, 1, S2, units, d2)
        dt = median_s(attn_step, 1, warm=th > 1) * 256 / units
        att[th] = {"ms_fwd_bwd": round(dt * 1e3, 1), "TFLOP_s": round(412518187008 / dt / 1e12, 5),
                   "threads": th,
                   "sample": f"{units} of the 256 (b, h) units of B16 H16 S2048 d64, scaled x "
                             f"{256 // units}"}
    steps["attention_c3_all_threads"] = att[threads]
    steps["attention_c3_1t"] = att[1]
    orc.set_threads(1)
    orc.pool_stop()  # the host threads end here, before the GPU extras
    out["train_steps"] = steps
    return out


def extras(ctx, torch, hip):
    out = {}
    ev = lambda: torch.cuda.Event(enable_timing=True)  # noqa: E731

    def timed(fn, iters, warm=2):
        for _ in range(warm):
            fn()
        torch.cuda.synchronize()
        a, b = ev(), ev()
        a.record()
        for _ in range(iters):
            fn()
        b.record()
        torch.cuda.synchronize()
        return a.elapsed_time(b) / iters

    # Decode-shaped W8A8: HBM-bound on the weight stream.  Each call takes the
    # next of 20 weight matrices (20 x 16.8 MB = 336 MB, more than the
    # 256 MB last-level cache), so the weight stream comes from HBM; the
    # single-matrix figure (cache-resident) is reported beside it.
    M, N, K = 32, 4096, 4096
    QA = torch.randint(-127, 128, (M, K), dtype=torch.int8, device="cuda")
    QWs = [torch.randint(-127, 128, (N, K), dtype=torch.int8, device="cuda") for _ in range(20)]
    sa, sw = torch.rand(M, device="cuda"), torch.rand(N, device="cuda")
    C = torch.empty((M, N), device="cuda")
    turn = [0]

    def rotating():
        turn[0] = (turn[0] + 1) % len(QWs)
        ctx.call("seeai_w8a8_gemm", QA.data_ptr(), sa.data_ptr(), QWs[turn[0]].data_ptr(),
                 sw.data_ptr(), C.data_ptr(), None, M, N, K)
    ms = timed(rotating, 200, 20)
    ms_resident = timed(lambda: ctx.call("seeai_w8a8_gemm", QA.data_ptr(), sa.data_ptr(),
                                         QWs[0].data_ptr(), sw.data_ptr(), C.data_ptr(), None,
                                         M, N, K), 200)
    alg_bytes = M * K + N * K + 4 * M * N + 4 * (M + N)
    out["w8a8_m32"] = {"ms": round(ms, 5), "TOPS": round(2 * M * N * K / ms / 1e9, 1),
                       "GB_s": round(alg_bytes / ms / 1e6, 1),
                       "hbm_frac": round(alg_bytes / ms / 1e6 / PEAK_HBM_GBS, 4),
                       "weights": "20 matrices in rotation (from HBM)",
                       "ms_one_matrix_cache_resident": round(ms_resident, 5)}
    del QWs

    # A reference point, not this build's code: the vendor library's int8
    # GEMM (hipBLASLt, through torch._int_mm) on the same box and shapes,
    # int32 output with no quantize and no dequant, the weight passed
    # K-contiguous as W8A8 packs it.
    ref = {}
    for (m, n, kk) in [(4096, 4096, 4096), (32, 4096, 4096)]:
        a = torch.randint(-127, 128, (m, kk), dtype=torch.int8, device="cuda")
        wt = torch.randint(-127, 128, (n, kk), dtype=torch.int8, device="cuda")
        try:
            ms_v = timed(lambda: torch._int_mm(a, wt.t()), 50, 5)
            ref[f"{m}x{n}x{kk}"] = {"ms": round(ms_v, 5),
                                    "TOPS": round(2 * m * n * kk / ms_v / 1e9, 1)}
        except RuntimeError as e:  # a build of torch without the int8 path
            ref[f"{m}x{n}x{kk}"] = {"error": str(e)[:120]}
        del a, wt
    out["w8a8_vendor_reference"] = dict(
        ref, note="hipBLASLt int8 GEMM via torch._int_mm: int32 output, no quantize or dequant")

    # Causal attention fwd+bwd, BASELINE config 3 (B16 H16 S2048 d64).
    B, S, H, d = 16, 2048, 16, 64
    flops = 412518187008.0  # causal-exact fwd + bwd
    q, k, v, do = (torch.randn((B * S, H * d), device="cuda") for _ in range(4))
    o, st = torch.empty_like(q), torch.empty((B * H * S, 4), device="cuda")
    dq, dk, dv = torch.empty_like(q), torch.empty_like(q), torch.empty_like(q)
    # bf16 operands held as bf16 (the models trained in bf16 activations)
    qb, kb, vb, dob = (x.to(torch.bfloat16) for x in (q, k, v, do))
    args_ = (ctx, qb, kb, vb, dob, o, st, dq, dk, dv, B, S, H, d)
    ms = timed(lambda: attention_step_bf16(*args_), 5, 1)
    tf = flops / ms / 1e9
    out["attention_bf16"] = {
        "ms_fwd_bwd": round(ms, 3), "TFLOP_s": round(tf, 1),
        "mfma_frac": round(tf / PEAK_BF16_TFLOPS, 4),
        "config": "B16 H16 S2048 d64 causal, Q/K/V/dO bf16 in HBM",
        "ms_parts": {part: round(timed(lambda part=part: attention_step_bf16(*args_, parts=(part,)),
                                       5, 1), 4) for part in ("fwd", "dq", "dkdv")}}
    del qb, kb, vb, dob
    # f32 operands: the relaxed family on the bf16 kernels (rounding while
    # staging), and the exact family
    for dt, name in [(1, "attention_bf16_f32_operands"), (0, "attention_f32")]:
        args_ = (ctx, dt, q, k, v, do, o, st, dq, dk, dv, B, S, H, d)
        ms = timed(lambda: attention_step(*args_), 3, 1)
        tf = flops / ms / 1e9
        peak = PEAK_BF16_TFLOPS if dt else PEAK_FP32_TFLOPS
        out[name] = {"ms_fwd_bwd": round(ms, 3), "TFLOP_s": round(tf, 1),
                     "mfma_frac": round(tf / peak, 4), "config": "B16 H16 S2048 d64 causal"}
        out[name]["ms_parts"] = {
            part: round(timed(lambda part=part: attention_step(*args_, parts=(part,)), 3, 1), 4)
            for part in ("fwd", "dq", "dkdv")}
    del q, k, v, do, o, st, dq, dk, dv

    # Softmax cross-entropy fwd at the decoders' 8192 x 32000 logits.
    Nr, Cc = 8192, 32000
    logits = torch.randn((Nr, Cc), device="cuda") * 3
    labels = torch.randint(0, Cc, (Nr,), dtype=torch.int32, device="cuda")
    probs = torch.empty_like(logits)
    loss = torch.empty(1, device="cuda")
    ms = timed(lambda: ctx.call("seeai_xent_fwd", logits.data_ptr(), labels.data_ptr(),
                                loss.data_ptr(), probs.data_ptr(), Nr, Cc, 0), 10)
    by = 2 * Nr * Cc * 4
    out["xent_fwd_8192x32000"] = {"ms": round(ms, 4), "GB_s": round(by / ms / 1e6, 1),
                                  "hbm_frac": round(by / ms / 1e6 / PEAK_HBM_GBS, 4)}
    del logits, probs

    # AdamW over config 5's 4,194,304 LoRA parameters (28 B/param).
    n = 4194304
    p, gr, m, vv = (torch.randn(n, device="cuda") for _ in range(4))
    vv.abs_()
    sp = hip.StepParams(1e-3, 0.9, 0.999, 1e-8, 0.01, 0, 3)
    import ctypes
    ms = timed(lambda: ctx.call("seeai_adamw_step", p.data_ptr(), gr.data_ptr(), m.data_ptr(),
                                vv.data_ptr(), n, ctypes.byref(sp), ctypes.c_float(0.0)), 50)
    by = 28 * n
    out["adamw_4M"] = {"ms": round(ms, 4), "GB_s": round(by / ms / 1e6, 1),
                       "hbm_frac": round(by / ms / 1e6 / PEAK_HBM_GBS, 4)}
    del p, gr, m, vv
    out.update(lora_steps(torch, hip))
    return out


def decoder_step_flops(layers, dim, ffn, vocab, T, batch, seq, heads, ffn_mats=2):
    """Algorithmic FLOP of one decoder LoRA training step: 2*T*P for the
    frozen products' forward plus 2*T*P for their dX (P = frozen GEMM
    parameters; an approximation: the step skips the dX below layer 0's
    LoRA sites), plus causal-exact attention fwd + bwd (3 x 4*d*pairs per
    (b, h) and layer).  LoRA products are negligible and not counted."""
    P = layers * (4 * dim * dim + ffn_mats * dim * ffn) + dim * vocab
    d = dim // heads
    pairs = seq * (seq + 1) // 2
    attn = layers * batch * heads * 3 * 4 * d * pairs
    return 4.0 * T * P + attn


def lora_steps(torch, hip):
    """The plan engine on BASELINE configs[0] (the LoRA MLP, one 32-row
    step) and configs[3] (the 12-layer decoder, 8 x 1024 tokens per step),
    plans from the in-repo plan writer, inputs resident.  The decoder runs
    the relaxed family as written (bf16 MFMA where the plan marks it) and,
    with relaxed execution switched off, the exact family."""
    import numpy as np
    pw = importlib.import_module("see-ai_amd.planwriter")
    out = {}

    def steps_per_s(eng, n, warm):
        for _ in range(warm):
            eng.train_resident()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(n):
            loss = eng.train_resident()
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) / n, loss

    img = pw.mlp_lora(hip.plan_self_hash)
    eng = hip.Engine(img.blob)
    eng.train_step(pw.normal(1, (32, 256)), pw.uniform_ints(2, 32, 256))
    dt, loss = steps_per_s(eng, 200, 10)
    out["lora_mlp_c1"] = {"us_per_step": round(dt * 1e6, 1), "rows_s": round(32 / dt),
                          "gemm_flop_per_step": 27394048, "loss": loss,
                          "bound": "launch latency (25 instructions per step)"}
    eng.close()
    del eng, img

    t0 = time.perf_counter()
    img = pw.decoder_lora(hip.plan_self_hash, relaxed=True)
    build_s = time.perf_counter() - t0
    eng = hip.Engine(img.blob)
    del img
    T = 8 * 1024
    tok = pw.uniform_ints(9, T + 1, 32000)
    eng.train_step(tok[:T].copy().view(np.float32), tok[1:].copy())
    flops = decoder_step_flops(12, 768, 3072, 32000, T, 8, 1024, 12)
    # configs[3] trains in bf16 activations: relaxed attention on the bf16
    # kernels; the exact leg runs every instruction in the exact family.
    for name, allow, n in [("lora_decoder_c4_relaxed", True, 10),
                           ("lora_decoder_c4_exact", False, 3)]:
        eng.set_relaxed(allow)
        eng.set_attention_bf16(allow)
        dt, loss = steps_per_s(eng, n, 2)
        tf = flops / dt / 1e12
        out[name] = {"ms_per_step": round(dt * 1e3, 2), "tokens_s": round(T / dt),
                     "TFLOP_s": round(tf, 1), "bf16_mfma_frac": round(tf / PEAK_BF16_TFLOPS, 4),
                     "flop_per_step": flops, "loss": loss, "steps_timed": n,
                     "config": "12 layers, d768, 12 heads, FFN 3072, vocab 32000, B8 x S1024, "
                               "LoRA r8 on Q/V",
                     "plan_build_s": round(build_s, 1)}
    # A fresh batch every step through the feeder (the reference's
    # BatchPipeline): the next batch's check and upload overlap the current
    # step, relaxed family as above.
    eng.set_relaxed(True)
    eng.set_attention_bf16(True)
    n = 10
    toks = np.stack([pw.uniform_ints(100 + i, T + 1, 32000) for i in range(n + 2)])
    xs = toks[:, :T].copy().view(np.float32)
    ys = toks[:, 1:].copy()
    eng.train_steps(xs[:2], ys[:2])  # warm: the feeder's buffers and thread
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    losses = eng.train_steps(xs[2:], ys[2:])
    torch.cuda.synchronize()
    dt = (time.perf_counter() - t0) / n
    resident = out["lora_decoder_c4_relaxed"]["ms_per_step"]
    out["lora_decoder_c4_relaxed_fed"] = {
        "ms_per_step": round(dt * 1e3, 2), "tokens_s": round(T / dt), "steps_timed": n,
        "loss": float(losses[-1]),
        "vs_resident": round(dt * 1e3 / resident, 4),
        "feed": "fresh token batch per step: checked and uploaded on the feeder stream while "
                "the previous step runs"}
    eng.close()
    del eng

    # 16 layers, d2048, 32 heads, SiLU-gated FFN 5632, RMSNorm,
    # frozen int8 base (per-column scales), LoRA r16 on Q/K/V/O, 4 x 2048
    # tokens per step; the relaxed family (bf16 MFMA over the exact int8
    # levels).  The exact family at this size is parity-tested at a small
    # shape, not timed.
    t0 = time.perf_counter()
    img = pw.decoder_q8_lora(hip.plan_self_hash, relaxed=True)
    build_s = time.perf_counter() - t0
    t0 = time.perf_counter()
    eng = hip.Engine(img.blob)
    load_s = time.perf_counter() - t0
    eng.set_attention_bf16(True)  # configs[4]: bf16 activations
    del img
    T = 4 * 2048
    tok = pw.uniform_ints(10, T + 1, 32000)
    eng.train_step(tok[:T].copy().view(np.float32), tok[1:].copy())
    flops = decoder_step_flops(16, 2048, 5632, 32000, T, 4, 2048, 32, ffn_mats=3)
    n = 3
    dt, loss = steps_per_s(eng, n, 1)
    tf = flops / dt / 1e12
    out["lora_decoder_c5_relaxed"] = {
        "ms_per_step": round(dt * 1e3, 2), "tokens_s": round(T / dt), "TFLOP_s": round(tf, 1),
        "bf16_mfma_frac": round(tf / PEAK_BF16_TFLOPS, 4), "flop_per_step": flops, "loss": loss,
        "steps_timed": n, "fused_dispatches": eng.fused_dispatches(),
        "dropped_stores": eng.dropped_stores(),
        "config": "16 layers, d2048, 32 heads, SiLU-gated FFN 5632, RMSNorm, vocab 32000, "
                  "B4 x S2048, int8 base (per-column scales), LoRA r16 on Q/K/V/O",
        "plan_build_s": round(build_s, 1), "plan_load_s": round(load_s, 1)}
    eng.close()
    return out


if __name__ == "__main__":
    sys.exit(main())
