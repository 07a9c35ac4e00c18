#!/usr/bin/env python3
"""Benchmark of the quantized GEMV hot path on one MI355X.

Workload: the GEMVs of one Llama-3-8B-shaped
Q4_K_M decode step at B=1 -- 32 layers x {q 4096x4096, k 1024x4096, v 1024x4096,
o 4096x4096, gate 14336x4096, up 14336x4096, down 4096x14336} plus the
lm_head 128256x4096.  Q4_K_M type rule used here: attn_v, ffn_down and the
lm_head are Q6_K in every layer, everything else Q4_K (4.876 GB of packed
weights per token).  Weights are random N(0, 0.02) fp32 drawn on the device and
quantized on the device with LoraMerge's Q4_K / Q6_K quantizers; activations are
N(0, 1) fp32.  All inputs are resident in HBM before timing starts.

A "step" is one decode token's 225 GEMVs, issued as a decode step can issue
them (independent GEMVs on one input share a launch: [q,k,v], [gate,up]),
captured once into a HIP graph and replayed.  value = algorithmic bytes per step / step time (GB/s), where
algorithmic bytes = packed weight bytes + 4*(cols + rows) per GEMV.

Extra measurements in the same JSON line:
  roofline      the dominant kernel (the grouped Q4_K [gate, up] GEMV, one launch
                over 2 x 14336x4096), timed with HIP events on its stream over
                all 32 layers' launches
  cpu_baseline  the CPU oracle (C restatement of Juno's Java matVecQ4Kraw /
                matVecQ6Kraw, one task per row on a thread pool) on one layer's
                GEMVs, on the host cores of this machine
  batched       the same step with B = 32 activations per GEMV
"""
from __future__ import annotations

import argparse
import ctypes
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_HBM_GBS = 8000.0
Q8_0, Q4_K, Q6_K = 8, 12, 14
BLOCK = {Q8_0: (32, 34), Q4_K: (256, 144), Q6_K: (256, 210)}
PEAK_MFMA_F16_TFLOPS = 2500.0  # dense fp16 MFMA

HIDDEN, FFN, KV, VOCAB, LAYERS = 4096, 14336, 1024, 128256, 32
# (name, rows, cols, type)
LAYER = [("attn_q", HIDDEN, HIDDEN, Q4_K), ("attn_k", KV, HIDDEN, Q4_K), ("attn_v", KV, HIDDEN, Q6_K),
         ("attn_output", HIDDEN, HIDDEN, Q4_K), ("ffn_gate", FFN, HIDDEN, Q4_K), ("ffn_up", FFN, HIDDEN, Q4_K),
         ("ffn_down", HIDDEN, FFN, Q6_K)]
HEAD = ("output", VOCAB, HIDDEN, Q6_K)


def packed_bytes(rows, cols, t):
    qk, bb = BLOCK[t]
    return rows * (cols // qk) * bb


def algo_bytes(rows, cols, t, B=1):
    return packed_bytes(rows, cols, t) + 4 * B * (rows + cols)


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def build_model(torch, be, seed=0):
    """Device-resident packed weights for all layers + head."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    mats = []
    for layer in range(LAYERS):
        for name, rows, cols, t in LAYER:
            w = torch.randn(rows * cols, generator=g, device="cuda", dtype=torch.float32).mul_(0.02)
            mats.append((f"blk.{layer}.{name}", rows, cols, t,
                         be.quantize_dev(t, w.data_ptr(), rows, cols, torch.cuda.current_stream().cuda_stream)))
            del w
    name, rows, cols, t = HEAD
    w = torch.randn(rows * cols, generator=g, device="cuda", dtype=torch.float32).mul_(0.02)
    mats.append((name, rows, cols, t, be.quantize_dev(t, w.data_ptr(), rows, cols,
                                                       torch.cuda.current_stream().cuda_stream)))
    del w
    torch.cuda.synchronize()
    return mats


def make_step(torch, L, mats, B, stream, grouped=True):
    """Buffers and a launcher for one decode step's GEMVs at batch B.

    B = 1 issues the GEMVs the way a decode step can: per layer one grouped
    launch for [q, k, v] (same input), [o], one for [gate, up] (same input),
    [down]; then the lm_head.  Each stage has its own input vector, as in a
    real step (attention-norm output, attention output, FFN-norm output,
    SwiGLU product).  B > 1 groups the same way through the batched group
    entry point (one MFMA launch per group at B >= 3)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    x_attn = torch.randn(B, HIDDEN, generator=g, device="cuda")
    x_o = torch.randn(B, HIDDEN, generator=g, device="cuda")
    x_ffn = torch.randn(B, HIDDEN, generator=g, device="cuda")
    x_down = torch.randn(B, FFN, generator=g, device="cuda")
    x_head = torch.randn(B, HIDDEN, generator=g, device="cuda")
    src = {"attn_q": x_attn, "attn_k": x_attn, "attn_v": x_attn, "attn_output": x_o,
           "ffn_gate": x_ffn, "ffn_up": x_ffn, "ffn_down": x_down, "output": x_head}
    ys = {m[0]: torch.empty(B, m[1], device="cuda") for m in mats}
    by_name = {m[0]: m for m in mats}
    stages = []
    for layer in range(LAYERS):
        for names in (["attn_q", "attn_k", "attn_v"], ["attn_output"], ["ffn_gate", "ffn_up"], ["ffn_down"]):
            stages.append([f"blk.{layer}.{n}" for n in names])
    stages.append(["output"])
    if not grouped:
        stages = [[m[0]] for m in mats]

    def xin(name):
        return src[name.split(".")[-1]]

    packed = []
    for st in stages:
        n = len(st)
        hs = (ctypes.c_void_p * n)(*[by_name[nm][4].handle for nm in st])
        xp = (ctypes.c_void_p * n)(*[xin(nm).data_ptr() for nm in st])
        yp = (ctypes.c_void_p * n)(*[ys[nm].data_ptr() for nm in st])
        packed.append((st, n, hs, xp, yp))

    keep = (src, ys)  # the kernels write through raw pointers: keep the tensors alive

    def launch():
        assert keep
        s = ctypes.c_void_p(stream.cuda_stream)
        for st, n, hs, xp, yp in packed:
            if B == 1:
                rc = L.jh_qmatvec_group_dev(n, hs, xp, yp, s)
            else:
                rc = L.jh_qmatvec_batched_group_dev(n, hs, xp, B, yp, s)
            if rc:
                raise RuntimeError(L.jh_last_error().decode())
    return launch, len(packed)


def time_graph(torch, launch, stream, steps, warmup):
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        launch()  # eager run once (also validates arguments)
        stream.synchronize()
        with torch.cuda.graph(g, stream=stream):
            launch()
        for _ in range(warmup):
            g.replay()
        stream.synchronize()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(stream)
        for _ in range(steps):
            g.replay()
        e1.record(stream)
        stream.synchronize()
        torch.cuda.synchronize()
        wall = time.perf_counter() - t0
    return e0.elapsed_time(e1) / steps, wall / steps * 1e3


def dominant_kernel(torch, L, mats, stream, reps):
    """Average launch duration of the dominant kernel: the grouped Q4_K [gate, up]
    GEMV of a layer (2 x 14336x4096, one staged launch, B=1).  HIP events on the
    launch stream around graph replays of all 32 layers' launches, so every
    launch streams matrices no other launch in the replay touches."""
    pairs = [([m for m in mats if m[0] == f"blk.{l}.ffn_gate"][0], [m for m in mats if m[0] == f"blk.{l}.ffn_up"][0])
             for l in range(LAYERS)]
    x = torch.randn(HIDDEN, device="cuda")
    ys = [torch.empty(FFN, device="cuda") for _ in range(2)]
    s = ctypes.c_void_p(stream.cuda_stream)
    args = []
    for ga, ua in pairs:
        hs = (ctypes.c_void_p * 2)(ga[4].handle, ua[4].handle)
        xp = (ctypes.c_void_p * 2)(x.data_ptr(), x.data_ptr())
        yp = (ctypes.c_void_p * 2)(ys[0].data_ptr(), ys[1].data_ptr())
        args.append((hs, xp, yp))
    def launch():
        for hs, xp, yp in args:
            if L.jh_qmatvec_group_dev(2, hs, xp, yp, s):
                raise RuntimeError(L.jh_last_error().decode())

    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        launch()  # eager pass first: validates the arguments outside the capture
        stream.synchronize()
        with torch.cuda.graph(g, stream=stream):
            launch()
        g.replay()
        stream.synchronize()
        e0.record(stream)
        for _ in range(reps):
            g.replay()
        e1.record(stream)
        stream.synchronize()
    avg_ms = e0.elapsed_time(e1) / (reps * len(args))
    per_launch = 2 * packed_bytes(FFN, HIDDEN, Q4_K) + 4 * (HIDDEN + 2 * FFN)
    del g  # the graph goes before the buffers it writes
    torch.cuda.synchronize()
    return avg_ms, per_launch, pairs


def d2h_packed(torch, dev):
    """Copy a matrix's packed bytes to host memory."""
    import numpy as np
    n = dev.nbytes()
    src = torch.empty(n, dtype=torch.uint8, device="cuda")
    hip = ctypes.CDLL("libamdhip64.so.7")  # the runtime torch already loaded
    torch.cuda.synchronize()
    rc = hip.hipMemcpy(ctypes.c_void_p(src.data_ptr()), ctypes.c_void_p(dev.device_pointer()),
                       ctypes.c_size_t(n), 3)  # device to device
    if rc != 0:
        raise RuntimeError(f"hipMemcpy failed: rc={rc}")
    return src.cpu().numpy()


def host_cpus():
    """Threads the reference's CPU path would use on this host, and the CPU
    model.  matVecQ4Kraw runs its rows on IntStream.parallel(), i.e.
    ForkJoinPool.commonPool() (availableProcessors - 1 workers) plus the
    calling thread (LlamaTransformerHandler.java:1436): availableProcessors
    threads.  The JVM's availableProcessors is the CPUs this process may run
    on (what `nproc` prints), limited by a cgroup CPU quota when one is set."""
    nproc = len(os.sched_getaffinity(0))
    quota = None
    try:
        with open("/sys/fs/cgroup/cpu.max") as f:
            q, period = f.read().split()[:2]
        if q != "max":
            quota = max(1, -(-int(q) // int(period)))
    except (OSError, ValueError):
        pass
    model = "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    return nproc, quota, model


def cpu_baseline(torch, mats, budget_s):
    """CPU oracle (C restatement of the Java path) on layer 0's seven GEMVs,
    on as many threads as the JVM's common pool plus the caller would use."""
    import numpy as np

    import oracle
    nproc, quota, model = host_cpus()
    # Without a cgroup quota, the pool stays within the 16 host CPUs a one-GPU
    # box grants per GPU (more would time-share the cores of other jobs).
    threads = min(nproc, quota) if quota else min(nproc, 16)
    layer0 = [m for m in mats if m[0].startswith("blk.0.")]
    host = []
    for name, rows, cols, t, dev in layer0:
        hbuf = d2h_packed(torch, dev)
        host.append((name, rows, cols, t, hbuf, np.random.default_rng(3).standard_normal(cols).astype(np.float32)))
    layer_bytes = sum(algo_bytes(r, c, t) for _, r, c, t, _, _ in host)
    t0 = time.perf_counter()
    reps = 0
    while True:
        for _, rows, cols, t, raw, x in host:
            oracle.matvec(t, raw, x, 0, rows, cols, nthreads=threads)
        reps += 1
        if time.perf_counter() - t0 >= budget_s:
            break
    dt = time.perf_counter() - t0
    gbs = layer_bytes * reps / dt / 1e9
    return {"value": round(gbs, 3), "unit": "GB/s", "cores": threads, "kind": "port",
            "nproc": nproc, "cgroup_cpu_quota": quota, "cpu_model": model,
            "sample": f"C++ restatement of Juno's Java CPU path: matVecQ4Kraw/matVecQ6Kraw as restated in "
                      f"oracle/juno_oracle.c (-O2 -ffp-contract=off, one task per row on {threads} threads, "
                      f"like ForkJoinPool.commonPool() plus the caller) on layer 0's 7 GEMVs "
                      f"({layer_bytes / 1e6:.1f} MB), {reps} reps in {dt:.1f} s",
            "tok_s_equiv": round(gbs * 1e9 / step_bytes(1), 4)}


def step_bytes(B):
    tot = sum(algo_bytes(r, c, t, B) for _, r, c, t in LAYER) * LAYERS
    return tot + algo_bytes(HEAD[1], HEAD[2], HEAD[3], B)


def step_flops(B):
    """Algorithmic GEMV flops of one 8B step at batch B: 2 B rows cols per GEMV."""
    return 2 * B * (sum(r * c for _, r, c, _ in LAYER) * LAYERS + HEAD[1] * HEAD[2])


def mfma_counters():
    """Counter-based MFMA figures of the batched [gate, up] kernel at B = 32 / 64
    from the committed rocprofv3 --pmc summary (profiles/)."""
    p = os.path.join(ROOT, "profiles", "mfma_group_q4k_gate_up_b32_b64_counters.json")
    try:
        with open(p) as f:
            d = json.load(f)
    except (OSError, ValueError):
        return {}
    keep = ("kernel", "avg_us", "mfma_issued_frac_of_2p5PF", "mfma_algorithmic_frac_of_2p5PF",
            "mfma_busy_frac_per_simd", "valu_active_frac_per_simd", "traffic_over_algorithmic")
    return {b: dict({k: v[k] for k in keep}, source="rocprofv3 --pmc SQ_INSTS_VALU_MFMA_MOPS_F16 / "
                    "SQ_VALU_MFMA_BUSY_CYCLES (profiles/mfma_group_q4k_gate_up_b32_b64_counters.json)")
            for b, v in d.get("kernels", {}).items()}


def hbm_stream_copy(torch, stream, reps=20):
    """STREAM-style copy on this GPU: 2 GiB of fp32 into another 2 GiB buffer
    (torch's copy kernel), HIP events around `reps` copies; bytes = read + write.
    The measured ceiling that HBM-bound kernels are compared with, beside the
    8 TB/s published peak."""
    n = 1 << 29
    a = torch.ones(n, device="cuda")
    b = torch.empty(n, device="cuda")
    with torch.cuda.stream(stream):
        for _ in range(2):
            b.copy_(a)
        stream.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(stream)
        for _ in range(reps):
            b.copy_(a)
        e1.record(stream)
        stream.synchronize()
    ms = e0.elapsed_time(e1) / reps
    moved = 2 * 4 * n
    del a, b
    torch.cuda.synchronize()
    gbs = moved / (ms * 1e-3) / 1e9
    return {"GB_s": round(gbs, 1), "bytes_per_copy": moved, "ms_per_copy": round(ms, 4),
            "frac_of_peak": round(gbs / PEAK_HBM_GBS, 4)}


def batch_sweep(torch, L, mats, stream, steps):
    """the 8B GEMV step at B in {8, 16, 32, 64} (grouped like
    B = 1; fp16 MFMA from B = 3).  MFMA utilisation = algorithmic flops over the
    dense fp16 peak; the kernels issue twice that (x as hi + lo fp16 limbs)."""
    out = {}
    counters = mfma_counters()
    for B in (8, 16, 32, 64):
        launch, _ = make_step(torch, L, mats, B, stream)
        ms, _ = time_graph(torch, launch, stream, steps, 2)
        tf = step_flops(B) / (ms * 1e-3) / 1e12
        out[f"b{B}"] = {"ms_per_step": round(ms, 4), "tok_s": round(B * 1e3 / ms, 1),
                        "GB_s": round(step_bytes(B) / (ms * 1e-3) / 1e9, 1), "algorithmic_TFLOP_s": round(tf, 1),
                        "mfma_util": round(tf / PEAK_MFMA_F16_TFLOPS, 4) if B >= 3 else None,
                        "mfma_issued_util": round(2 * tf / PEAK_MFMA_F16_TFLOPS, 4) if B >= 3 else None}
        if f"b{B}" in counters:
            out[f"b{B}"]["gate_up_kernel_counters"] = counters[f"b{B}"]
    return out


def rotated_gemv(torch, be, L, stream, qtype, rows, cols, B, seed, outliers=False, min_bytes=512 << 20, reps=5):
    """One GEMV shape timed over enough packed copies (>= min_bytes in all) that
    no launch finds its weights in the 256 MB memory-side cache; returns
    (us per GEMV, algorithmic GB/s)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    one = packed_bytes(rows, cols, qtype)
    n = max(2, -(-min_bytes // one))
    w = torch.randn(rows * cols, generator=g, device="cuda").mul_(0.02)
    if outliers:  # 1 % of the entries at 10x (seeded choice)
        idx = torch.randperm(rows * cols, generator=g, device="cuda")[: rows * cols // 100]
        w[idx] *= 10
    cur = torch.cuda.current_stream().cuda_stream
    mats = [be.quantize_dev(qtype, w.data_ptr(), rows, cols, cur) for _ in range(n)]
    del w
    x = torch.randn(B, cols, generator=g, device="cuda")
    y = torch.empty(B, rows, device="cuda")
    s = ctypes.c_void_p(stream.cuda_stream)
    torch.cuda.synchronize()

    def launch():
        for m in mats:
            if L.jh_qmatvec_batched_dev(m.handle, ctypes.c_void_p(x.data_ptr()), B, ctypes.c_void_p(y.data_ptr()), 0,
                                        rows, s):
                raise RuntimeError(L.jh_last_error().decode())
    ms, _ = time_graph(torch, launch, stream, reps, 1)
    for m in mats:
        m.close()
    torch.cuda.synchronize()
    us = ms * 1e3 / n
    return us, algo_bytes(rows, cols, qtype, B) / (us * 1e-6) / 1e9


def shape_sweeps(torch, be, L, stream):
    """BASELINE config 1 (single Q4_K GEMV at the TinyLlama up-projection shape)
    and config 5 (Phi-3-mini-shaped Q8_0 and Q6_K GEMVs with 1 % outliers at 10x,
    B = 1 and 32), each over rotated copies."""
    us, gbs = rotated_gemv(torch, be, L, stream, Q4_K, 5632, 2048, 1, 21)
    cfg1 = {"shape": "5632x2048", "type": "Q4_K", "batch": 1, "us": round(us, 2), "GB_s": round(gbs, 1),
            "pct_of_peak": round(100 * gbs / PEAK_HBM_GBS, 2)}
    phi = {}
    shapes = {"qkv": (9216, 3072), "o": (3072, 3072), "gate_up": (16384, 3072), "down": (3072, 8192),
              "lm_head": (32064, 3072)}
    for qt, tn in ((Q8_0, "Q8_0"), (Q6_K, "Q6_K")):
        for name, (r, c) in shapes.items():
            for B in (1, 32):
                us, gbs = rotated_gemv(torch, be, L, stream, qt, r, c, B, 30 + r + c + B, outliers=True)
                phi[f"{tn}.{name}.b{B}"] = {"us": round(us, 2), "GB_s": round(gbs, 1)}
    return {"config1_tinyllama_up_q4k": cfg1, "config5_phi3": phi}


def parity_spot_check(torch, L, mats, stream):
    """Gate GEMV of layer 0 against the oracle (rel-err metric of the tests)."""
    import numpy as np

    import oracle
    name, rows, cols, t, dev = [m for m in mats if m[0] == "blk.0.ffn_gate"][0]
    hraw = d2h_packed(torch, dev)
    x = np.random.default_rng(9).standard_normal(cols).astype(np.float32)
    dx = torch.from_numpy(x).cuda()
    dy = torch.empty(rows, device="cuda")
    L.jh_qmatvec_batched_dev(dev.handle, dx.data_ptr(), 1, dy.data_ptr(), 0, rows, None)
    torch.cuda.synchronize()
    y = dy.cpu().numpy().astype(np.float64)
    ref = oracle.matvec(t, hraw, x, 0, rows, cols).astype(np.float64)
    deq = oracle.dequantize(t, hraw, rows, cols).astype(np.float64)
    scale = np.abs(deq) @ np.abs(x.astype(np.float64))
    return float((np.abs(y - ref) / np.maximum(np.abs(ref), 1e-3 * scale)).max())


def profile_mode(torch, L, be):
    """Launches for hardware-counter runs (rocprofv3 --pmc): 8 layers' grouped
    [gate, up] Q4_K GEMVs, eagerly, 4 times each, then the calibration copy."""
    g = torch.Generator(device="cuda")
    g.manual_seed(0)
    mats = []
    for layer in range(8):
        pair = []
        for name in ("ffn_gate", "ffn_up"):
            w = torch.randn(FFN * HIDDEN, generator=g, device="cuda").mul_(0.02)
            pair.append(be.quantize_dev(Q4_K, w.data_ptr(), FFN, HIDDEN, torch.cuda.current_stream().cuda_stream))
            del w
        mats.append(pair)
    torch.cuda.synchronize()
    x = torch.randn(HIDDEN, device="cuda")
    ys = [torch.empty(FFN, device="cuda") for _ in range(2)]
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for _ in range(4):
        for ga, ua in mats:
            hs = (ctypes.c_void_p * 2)(ga.handle, ua.handle)
            xp = (ctypes.c_void_p * 2)(x.data_ptr(), x.data_ptr())
            yp = (ctypes.c_void_p * 2)(ys[0].data_ptr(), ys[1].data_ptr())
            if L.jh_qmatvec_group_dev(2, hs, xp, yp, s):
                raise RuntimeError(L.jh_last_error().decode())
    torch.cuda.synchronize()
    # calibration: an elementwise kernel that reads 1 GiB and writes 1 GiB
    a = torch.empty(1 << 28, device="cuda")
    a.fill_(1.0)
    b = torch.empty_like(a)
    torch.mul(a, 2.0, out=b)
    torch.cuda.synchronize()
    per_launch = 2 * packed_bytes(FFN, HIDDEN, Q4_K) + 4 * (HIDDEN + 2 * FFN)
    print(json.dumps({"profile": "gemv_staged Q4_K [gate, up]", "launches": 32,
                      "algorithmic_bytes_per_launch": per_launch,
                      "calibration": "torch.mul 2^28 fp32: reads 1073741824 B, writes 1073741824 B"}), flush=True)


def profile_mfma_mode(torch, L, be):
    """Launches for MFMA counter runs (rocprofv3 --pmc): 8 layers' grouped
    Q4_K [gate, up] GEMVs at B = 32 (mfma_group<false, 1, 1, ..>) and at B = 64
    (mfma_group<false, 2, 1, ..>), eagerly, 4 times each, then the calibration copy."""
    g = torch.Generator(device="cuda")
    g.manual_seed(0)
    mats = []
    for layer in range(8):
        pair = []
        for name in ("ffn_gate", "ffn_up"):
            w = torch.randn(FFN * HIDDEN, generator=g, device="cuda").mul_(0.02)
            pair.append(be.quantize_dev(Q4_K, w.data_ptr(), FFN, HIDDEN, torch.cuda.current_stream().cuda_stream))
            del w
        mats.append(pair)
    torch.cuda.synchronize()
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    out = {}
    for B in (32, 64):
        x = torch.randn(B, HIDDEN, device="cuda")
        ys = [torch.empty(B, FFN, device="cuda") for _ in range(2)]
        for _ in range(4):
            for ga, ua in mats:
                hs = (ctypes.c_void_p * 2)(ga.handle, ua.handle)
                xp = (ctypes.c_void_p * 2)(x.data_ptr(), x.data_ptr())
                yp = (ctypes.c_void_p * 2)(ys[0].data_ptr(), ys[1].data_ptr())
                if L.jh_qmatvec_batched_group_dev(2, hs, xp, B, yp, s):
                    raise RuntimeError(L.jh_last_error().decode())
        torch.cuda.synchronize()
        kernel, ksplit = ctypes.c_int(), ctypes.c_int()
        hs = (ctypes.c_void_p * 2)(mats[0][0].handle, mats[0][1].handle)
        L.jh_qmatvec_batched_plan(2, hs, B, ctypes.byref(kernel), ctypes.byref(ksplit))
        out[f"b{B}"] = {"launches": 32, "ksplit": ksplit.value, "algorithmic_flops_per_launch": 2 * B * 2 * FFN * HIDDEN,
                        "issued_f16_mfma_flops_per_launch": 2 * 2 * B * 2 * FFN * HIDDEN,
                        "algorithmic_bytes_per_launch": 2 * packed_bytes(FFN, HIDDEN, Q4_K) + 4 * B * (HIDDEN + 2 * FFN)}
    a = torch.empty(1 << 28, device="cuda")
    a.fill_(1.0)
    b = torch.empty_like(a)
    torch.mul(a, 2.0, out=b)
    torch.cuda.synchronize()
    print(json.dumps({"profile": "mfma_group Q4_K [gate, up]", **out,
                      "calibration": "torch.mul 2^28 fp32: reads 1073741824 B, writes 1073741824 B"}), flush=True)


def measured_traffic():
    """HBM bytes per launch of the dominant kernel from the committed rocprofv3
    --pmc summary (FETCH_SIZE + WRITE_SIZE, calibrated; see profiles/)."""
    p = os.path.join(ROOT, "profiles", "gemv_staged_q4k_gate_up_counters.json")
    try:
        with open(p) as f:
            d = json.load(f)
        return int(d["traffic_bytes_per_launch"]), "rocprofv3 --pmc FETCH_SIZE/WRITE_SIZE (profiles/gemv_staged_q4k_gate_up_counters.json)"
    except (OSError, KeyError, ValueError):
        return None, None


def decode_step_8b(torch, be, stream, steps, mats, B):
    """Full decode steps at the Llama-3-8B shape (32 layers, hidden 4096, 32 / 8
    heads of 128, FFN 14336, vocab 128256, rope theta 500000) on the bench's own
    packed matrices, with N(0.5..1.5) norm weights and a Q6_K token embedding:
    B = 1 through LlamaDecoder (from the residual stream), B > 1 through
    LlamaBatchPipeline (token rows, one step for all B requests).  Every request
    is at position 511 over a KV cache pre-filled with N(0, 1); the step is one
    captured graph.  Every op of the step is a HIP kernel."""
    from juno_amd import decode as D
    from juno_amd.pipeline import LlamaBatchPipeline
    cfg = D.LlamaConfig(hidden_dim=HIDDEN, num_layers=LAYERS, num_heads=32, num_kv_heads=8, head_dim=128,
                        intermediate_size=FFN, vocab_size=VOCAB, rms_norm_eps=1e-5, rope_theta=500000.0)
    by = {m[0]: m[4] for m in mats}
    g = torch.Generator(device="cuda")
    g.manual_seed(10)
    norm = lambda: torch.rand(HIDDEN, generator=g, device="cuda").add_(0.5)
    names = {"q": "attn_q", "k": "attn_k", "v": "attn_v", "o": "attn_output", "gate": "ffn_gate", "up": "ffn_up",
             "down": "ffn_down"}
    layers = [D.LlamaLayerWeights(norm(), norm(), {k: by[f"blk.{l}.{v}"] for k, v in names.items()})
              for l in range(LAYERS)]
    emb = None
    if B > 1:
        src = torch.randn(VOCAB * HIDDEN, generator=g, device="cuda")
        emb = be.quantize_dev(Q6_K, src.data_ptr(), VOCAB, HIDDEN, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        del src
    w = D.LlamaWeights(cfg, layers, norm(), by["output"], token_embd=emb)
    if B == 1:
        dec = D.LlamaDecoder(w, max_seq=512)
        dec.k_cache.normal_(generator=g)
        dec.v_cache.normal_(generator=g)
        dec.x.normal_(generator=g)
        dec.pos.fill_(511)
        x0 = dec.x.clone()

        def full():
            dec.x.copy_(x0)  # the step updates the residual stream in place
            dec.enqueue_step(stream)
        ms, _ = time_graph(torch, full, stream, steps, 3)
        del dec
    else:
        pipe = LlamaBatchPipeline(w, max_seq=512, max_batch=B)
        pipe.k_cache.normal_(generator=g)
        pipe.v_cache.normal_(generator=g)
        pipe.meta.copy_(torch.tensor([[(97 * b) % VOCAB for b in range(B)], [511] * B, list(range(B))],
                                     dtype=torch.int32))
        ms, _ = time_graph(torch, lambda: pipe.enqueue(B, stream), stream, steps, 3)
        del pipe
    if emb is not None:
        emb.close()
    torch.cuda.synchronize()
    return {"config": f"llama3-8b-q4_k_m-full-decode-step-b{B}-ctx512", "batch": B, "ms_per_step": round(ms, 4),
            "tok_s": round(B * 1e3 / ms, 1)}


def tinyllama_step(torch, stream, steps):
    """TinyLlama-1.1B-shaped Q4_K_M full decode step (22 layers,
    hidden 2048, 32 / 4 heads, head_dim 64, FFN 5632, vocab 32000; Q6_K for
    attn_v, ffn_down and the output), B = 1, at position 511 over a KV cache
    pre-filled with N(0, 1): every op of the step is a HIP kernel, the step is
    one captured graph.  Also times the step's GEMV launches alone (the tok/s
    bound the GEMVs set)."""
    from juno_amd import decode as D
    cfg = D.LlamaConfig(hidden_dim=2048, num_layers=22, num_heads=32, num_kv_heads=4, head_dim=64,
                        intermediate_size=5632, vocab_size=32000)
    w = D.LlamaWeights.random(cfg, seed=7, embeddings=True)
    dec = D.LlamaDecoder(w, max_seq=512)
    g = torch.Generator(device="cuda")
    g.manual_seed(8)
    dec.k_cache.normal_(generator=g)
    dec.v_cache.normal_(generator=g)
    dec.x.normal_(generator=g)
    dec.pos.fill_(511)
    x0 = dec.x.clone()
    gemv_bytes = sum(m.nbytes() for lw in w.layers for m in lw.mats.values()) + w.output.nbytes()

    def full():
        dec.x.copy_(x0)  # the step updates the residual stream in place
        dec.enqueue_step(stream)

    gate = torch.empty(cfg.intermediate_size, device="cuda")
    up = torch.empty(cfg.intermediate_size, device="cuda")

    def gemvs_only():  # the step's projections alone (gate and up as a plain group)
        for lw in w.layers:
            m = lw.mats
            dec._group([m["q"], m["k"], m["v"]], [dec.xn] * 3, [dec.q, dec.k, dec.v], ctypes.c_void_p(stream.cuda_stream))
            dec._group([m["o"]], [dec.att], [dec.proj], ctypes.c_void_p(stream.cuda_stream))
            dec._group([m["gate"], m["up"]], [dec.xn] * 2, [gate, up], ctypes.c_void_p(stream.cuda_stream))
            dec._group([m["down"]], [dec.hid], [dec.proj], ctypes.c_void_p(stream.cuda_stream))
        dec._group([w.output], [dec.xn], [dec.logits], ctypes.c_void_p(stream.cuda_stream))

    ms, _ = time_graph(torch, full, stream, steps, 3)
    gemv_ms, _ = time_graph(torch, gemvs_only, stream, steps, 3)
    out = {"config": "tinyllama-1.1b-q4_k_m-full-decode-step-b1-ctx512", "layers": cfg.num_layers,
           "ms_per_step": round(ms, 4), "tok_s": round(1e3 / ms, 1),
           "gemv_ms_per_step": round(gemv_ms, 4), "gemv_tok_s_bound": round(1e3 / gemv_ms, 1),
           "gemv_bytes_per_step": gemv_bytes, "gemv_GB_s": round(gemv_bytes / (gemv_ms * 1e-3) / 1e9, 1),
           "launches_per_step": cfg.num_layers * 6 + 3,
           "ops": "residual + rmsnorm + grouped q/k/v (one launch; layer 0: rmsnorm, then the group), rope + KV "
                  "append + GQA (2 kernels), o, residual + rmsnorm + gate/up + silu*up (one launch), down; final "
                  "residual + rmsnorm + output projection (one launch), position increment"}
    del dec
    out["batched"] = tinyllama_batch_step(torch, stream, steps, w, cfg, 32)
    w.close()
    return out


def tinyllama_batch_step(torch, stream, steps, w, cfg, B):
    """forwardBatch of B requests through the same TinyLlama-shaped model: one
    decode step for all B (token embedding rows, batched GEMVs, batched rope +
    KV append + attention over B cache slots), each request at position 511
    over its own pre-filled KV cache; one captured graph per step."""
    from juno_amd.pipeline import LlamaBatchPipeline
    pipe = LlamaBatchPipeline(w, max_seq=512, max_batch=B)
    g = torch.Generator(device="cuda")
    g.manual_seed(9)
    pipe.k_cache.normal_(generator=g)
    pipe.v_cache.normal_(generator=g)
    rows = torch.tensor([[(97 * b) % cfg.vocab_size for b in range(B)], [511] * B, list(range(B))],
                        dtype=torch.int32)
    pipe.meta.copy_(rows)
    ms, _ = time_graph(torch, lambda: pipe.enqueue(B, stream), stream, steps, 3)
    del pipe
    return {"config": f"tinyllama-1.1b-q4_k_m-forward-batch-b{B}-ctx512", "batch": B, "ms_per_step": round(ms, 4),
            "tok_s": round(B * 1e3 / ms, 1),
            "launches_per_step": cfg.num_layers * 9 + 3}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--cpu-budget", type=float, default=15.0, help="seconds of CPU-baseline work")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-batched", action="store_true")
    ap.add_argument("--profile-mfma", action="store_true",
                    help="counter-collection mode for the batched MFMA kernel: [gate, up] at B = 32 and 64")
    ap.add_argument("--profile", action="store_true",
                    help="counter-collection mode: only the dominant kernel (eager launches over 8 layers' "
                         "[gate, up]) and a 1 GiB elementwise copy that calibrates FETCH_SIZE / WRITE_SIZE")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) > 1:
        print("bench.py measures one GPU only: this build has no multi-GPU path "
              "(the GEMV would shard by rows, one slice of every matrix per GPU).", file=sys.stderr)
        sys.exit(2)

    import torch

    from juno_amd import _lib
    from juno_amd import matvec as mv
    L = _lib.load()
    ctx = mv.GpuContext.shared(0)
    be = ctx.create_mat_vec()
    info = mv.device_info(0)
    log(f"device {info}")
    if args.profile:
        profile_mode(torch, L, be)
        return
    if args.profile_mfma:
        profile_mfma_mode(torch, L, be)
        return
    t0 = time.perf_counter()
    mats = build_model(torch, be)
    log(f"model built: {len(mats)} matrices, {sum(m[4].nbytes() for m in mats) / 1e9:.3f} GB packed, "
        f"{time.perf_counter() - t0:.1f} s")
    stream = torch.cuda.Stream()
    stream_copy = hbm_stream_copy(torch, stream)
    log(f"HBM STREAM copy: {stream_copy}")

    launch, nlaunch = make_step(torch, L, mats, 1, stream)
    ms, wall_ms = time_graph(torch, launch, stream, args.steps, args.warmup)
    sb = step_bytes(1)
    gbs = sb / (ms * 1e-3) / 1e9
    log(f"B=1 step: {ms:.4f} ms (wall {wall_ms:.4f} ms, {nlaunch} grouped launches)  {gbs:.1f} GB/s  "
        f"{1e3 / ms:.1f} tok/s")

    avg_ms, per_launch, _ = dominant_kernel(torch, L, mats, stream, reps=max(args.steps, 20))
    ach = per_launch / (avg_ms * 1e-3) / 1e9
    log(f"gate+up Q4_K grouped GEMV: {avg_ms * 1e3:.2f} us/launch  {ach:.1f} GB/s")

    batched = None
    if not args.no_batched:
        launch32, _ = make_step(torch, L, mats, 32, stream)
        ms32, _ = time_graph(torch, launch32, stream, max(args.steps // 5, 3), 2)
        sb32 = step_bytes(32)
        batched = {"B": 32, "ms_per_step": round(ms32, 4), "tok_s": round(32 * 1e3 / ms32, 1),
                   "GB_s": round(sb32 / (ms32 * 1e-3) / 1e9, 1)}
        log(f"B=32 step: {ms32:.4f} ms  {batched}")

    sweep = None
    if not args.no_batched:
        sweep = batch_sweep(torch, L, mats, stream, max(args.steps // 5, 3))
        log(f"batched sweep: {sweep}")
    shapes = shape_sweeps(torch, be, L, stream)
    log(f"shape sweeps: {shapes}")

    full8b = {"b1": decode_step_8b(torch, be, stream, max(args.steps // 2, 10), mats, 1)}
    log(f"8B full decode step, B=1: {full8b['b1']}")
    if not args.no_batched:
        full8b["b32"] = decode_step_8b(torch, be, stream, max(args.steps // 5, 3), mats, 32)
        log(f"8B full decode step, B=32: {full8b['b32']}")

    tiny = tinyllama_step(torch, stream, max(args.steps // 2, 10))
    log(f"TinyLlama decode step: {tiny}")

    traffic, traffic_src = measured_traffic()
    parity = parity_spot_check(torch, L, mats, stream)
    log(f"parity spot check (layer-0 gate vs oracle): max rel-err {parity:.2e}")

    cpu = None if args.no_cpu_baseline else cpu_baseline(torch, mats, args.cpu_budget)
    if cpu:
        log(f"cpu baseline: {cpu}")

    line = {
        "metric": "Q4_K GEMV effective HBM GB/s (% of peak); decode tok/s at 8B shapes, B=1/32",
        "value": round(gbs, 1),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic: N(0,0.02) weights quantized on device with LoraMerge Q4_K/Q6_K; N(0,1) activations",
        "config": {"workload": "llama3-8b-q4_k_m-decode-gemvs-b1", "hidden": HIDDEN, "ffn": FFN,
                   "kv_dim": KV, "vocab": VOCAB, "layers": LAYERS, "batch": 1,
                   "gemvs_per_step": len(mats), "launches_per_step": nlaunch,
                   "q6k_rule": "attn_v, ffn_down, output in every layer",
                   "algorithmic_bytes_per_step": sb},
        "pct_of_peak": round(100 * gbs / PEAK_HBM_GBS, 2),
        "tok_s": round(1e3 / ms, 1),
        "roofline": {"bound": "hbm", "achieved": round(ach, 1), "peak": PEAK_HBM_GBS, "unit": "GB/s",
                     "frac": round(ach / PEAK_HBM_GBS, 4), "traffic": traffic, "traffic_source": traffic_src,
                     "kernel": "gemv_staged<Q4_K> [gate, up] 2x14336x4096 B=1 (one launch)",
                     "avg_launch_us": round(avg_ms * 1e3, 3),
                     "algorithmic_bytes_per_launch": per_launch},
        "cpu_baseline": cpu,
        "hbm_stream_copy": stream_copy,
        "batched": batched,
        "batched_sweep": sweep,
        "shape_sweeps": shapes,
        "decode_step_8b": full8b,
        "decode_step_tinyllama": tiny,
        "parity_max_rel_err": parity,
        "device": info["name"],
    }
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
