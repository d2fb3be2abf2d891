"""Benchmark of the WhisperDRZ attention hot path on one MI355X.

Headline (the JSON line's ``value``): BASELINE config 2 — encoder self-attention at
Whisper-large-v3 shape, B=16 x H=20 x L=1500 x D=64, bf16, 32 sequential layers each with its
own seeded inputs resident in HBM. One "step" = the 32 layers. Reported in TFLOP/s of
algorithmic work (4*B*H*L^2*D per layer) and as a fraction of the bf16 dense MFMA peak.

The same line carries, under ``decode``, the decoder paths (configs 3, 4, 5) in GB/s of
algorithmic HBM bytes (only valid K/V rows are counted), each with 32 distinct per-layer caches
captured into one hipGraph and replayed, and under ``cpu_baseline`` the reference's CPU torch
path (torch SDPA, fp32) timed on this host's cores on a bounded sample. Under ``dtw_prep`` it
carries the DTW alignment inputs (compute_attention and _dtw_prep_batch) in GB/s of algorithmic
HBM bytes, and under ``log_mel`` the GPU log-mel front end in GB/s of its samples and mel, each
with its own roofline and CPU baseline.

Under ``cross_fill`` it times the encoder output's projection into every layer's cross cache (the
key/value GEMM and ``wdrz_kv_fill``, with its own HBM roofline).
Under ``decode_step`` it times a whole captured large-v3 decode step (64 streams) with and without
the fused add + LayerNorm.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu] [--only enc|dec|dtw|mel|step|fill]
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

import numpy as np
import torch

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

METRIC = "enc-attn TFLOP/s + decode-attn HBM GB/s at large-v3 shape, % of MI355X roofline"
# MI355X published peaks (dense, no sparsity).
PEAK_BF16_TFLOPS = 2500.0
PEAK_HBM_GBS = 8000.0

H, D = 20, 64
E = 2  # bytes per bf16 element
N_LAYERS = 32


def log(msg: str) -> None:
    print(msg, file=sys.stderr, flush=True)


_TRAFFIC_FILE = os.path.join(ROOT, "profiles", "pmc_traffic.json")


def measured_traffic(kernel: str):
    """HBM bytes per launch of `kernel` from the committed rocprofv3 FETCH_SIZE/WRITE_SIZE passes
    (profiles/pmc_traffic.json; calibrated against a copy of known size), or None."""
    try:
        with open(_TRAFFIC_FILE) as f:
            k = json.load(f)["kernels"].get(kernel)
    except (OSError, ValueError, KeyError):
        return None
    return None if k is None else int(k["traffic_bytes"])


def summed_traffic(kernels):
    """`measured_traffic` of several kernels together, None where any of them was not measured."""
    each = [measured_traffic(k) for k in kernels or ()]
    return sum(each) if each and None not in each else None


def timed_events(fn, iters: int, stream: torch.cuda.Stream) -> float:
    """Milliseconds per call of fn() over `iters` calls, timed with HIP events on `stream`."""
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    start.record(stream)
    for _ in range(iters):
        fn()
    end.record(stream)
    torch.cuda.synchronize()
    return start.elapsed_time(end) / iters


# --------------------------------------------------------------------------------------------
# config 2: encoder self-attention
# --------------------------------------------------------------------------------------------


def bench_encoder(dev, steps: int, warmup: int) -> dict:
    from whisperdrz_amd import scaled_dot_product_attention

    B, L = 16, 1500
    flop_layer = 4.0 * B * H * L * L * D
    log(f"[bench] encoder: generating {N_LAYERS} layers of B={B} H={H} L={L} bf16 inputs")
    layers = []
    for i in range(N_LAYERS):
        g = torch.Generator(device=dev).manual_seed(2000 + i)
        qkv = torch.randn((3, B, L, H, D), generator=g, device=dev, dtype=torch.float32).to(torch.bfloat16)
        layers.append(tuple(x.permute(0, 2, 1, 3) for x in qkv))  # [B, H, L, D] views of [B, L, H, D]
    outs = [None] * N_LAYERS

    def step():
        for i, (q, k, v) in enumerate(layers):
            outs[i] = scaled_dot_product_attention(q, k, v, scale=0.125)

    stream = torch.cuda.current_stream()
    for _ in range(warmup):
        step()
    ms_step = timed_events(step, steps, stream)
    ms_launch = ms_step / N_LAYERS
    tflops = flop_layer * N_LAYERS / (ms_step * 1e-3) / 1e12
    achieved = flop_layer / (ms_launch * 1e-3) / 1e12
    log(f"[bench] encoder: {ms_step:.3f} ms/step, {tflops:.1f} TFLOP/s ({100 * tflops / PEAK_BF16_TFLOPS:.1f}% of bf16 peak)")
    del layers, outs
    torch.cuda.empty_cache()

    # one 30-s window (B=1): a grid smaller than the chip, served by the key-split kernel
    single = []
    for i in range(8):
        g = torch.Generator(device=dev).manual_seed(2500 + i)
        qkv = torch.randn((3, 1, L, H, D), generator=g, device=dev, dtype=torch.float32).to(torch.bfloat16)
        single.append(tuple(x.permute(0, 2, 1, 3) for x in qkv))

    def step1():
        for q, k, v in single:
            scaled_dot_product_attention(q, k, v, scale=0.125)

    for _ in range(warmup):
        step1()
    us1 = timed_events(step1, steps, stream) * 1e3 / len(single)
    t1 = 4.0 * H * L * L * D / (us1 * 1e-6) / 1e12
    log(f"[bench] encoder, one window (B=1): {us1:.1f} us per layer, {t1:.1f} TFLOP/s")
    del single
    torch.cuda.empty_cache()
    return {
        "ms_per_step": ms_step,
        "tflops": tflops,
        "single_window": {"workload": "one encoder layer B=1 H=20 L=1500 D=64 bf16 (dense_split4_kernel<Bf16>)",
                          "us_per_layer": round(us1, 2), "tflops": round(t1, 1)},
        "roofline": {
            "bound": "mfma",
            "achieved": round(achieved, 2),
            "peak": PEAK_BF16_TFLOPS,
            "unit": "TFLOP/s",
            "frac": round(achieved / PEAK_BF16_TFLOPS, 4),
            "traffic": measured_traffic("dense_pipe_kernel<wdrz::Bf16, 3>"),
            "traffic_source": "profiles/pmc_traffic.json (rocprofv3 FETCH_SIZE/WRITE_SIZE passes)",
            "kernel": "dense_pipe_kernel<Bf16, 3>",
            "flop_per_launch": flop_layer,
            "ms_per_launch": ms_launch,
            # softmax exponentials per layer (B*H*L^2) and their rate: the VALU side of the kernel
            "exp_per_launch": float(B * H * L * L),
            "exp_per_s": round(B * H * L * L / (ms_launch * 1e-3), 1),
        },
    }


def bench_config1(dev, steps: int, warmup: int) -> dict:
    """Config 1 (the reference's CPU-runnable case) on the GPU: one encoder layer, B=1 H=20
    L=1500 D=64 in fp32, non-causal, scale 1/8 (dense_f32_kernel: every fp32 product is six bf16
    matrix products, so its roofline is a sixth of the bf16 matrix peak); 8 seeded input sets in
    rotation."""
    from whisperdrz_amd import scaled_dot_product_attention

    B, L, n_sets = 1, 1500, 8
    flop = 4.0 * B * H * L * L * D
    sets = []
    for i in range(n_sets):
        g = torch.Generator(device=dev).manual_seed(1000 + i)
        qkv = torch.randn((3, B, L, H, D), generator=g, device=dev, dtype=torch.float32)
        sets.append(tuple(x.permute(0, 2, 1, 3) for x in qkv))

    def run():
        for q, k, v in sets:
            scaled_dot_product_attention(q, k, v, scale=0.125)

    stream = torch.cuda.current_stream()
    for _ in range(warmup):
        run()
    us = timed_events(run, steps, stream) * 1e3 / n_sets
    tflops = flop / (us * 1e-6) / 1e12
    log(f"[bench] config1 fp32 dense (B=1 H=20 L=1500): {us:.1f} us per layer, {tflops:.2f} TFLOP/s "
        f"({100 * 6 * tflops / PEAK_BF16_TFLOPS:.1f}% of a sixth of the bf16 matrix peak)")
    del sets
    torch.cuda.empty_cache()
    return {
        "workload": "config1: one encoder self-attention layer B=1 H=20 L=1500 D=64 fp32, non-causal, scale 1/8 "
                    "(the shape of cpu_baseline), 8 seeded input sets in rotation",
        "us_per_layer": round(us, 2),
        "tflops": round(tflops, 3),
        "roofline": {"bound": "mfma", "achieved": round(tflops, 3), "peak": round(PEAK_BF16_TFLOPS / 6, 1),
                     "unit": "TFLOP/s", "frac": round(6 * tflops / PEAK_BF16_TFLOPS, 4), "traffic": measured_traffic("dense_f32_kernel<false>"),
                     "traffic_source": "profiles/pmc_traffic.json (rocprofv3 FETCH_SIZE/WRITE_SIZE passes)",
                     "kernel": "dense_f32_kernel<false> (six v_mfma_f32_32x32x16_bf16 products per fp32 product)"},
    }


# --------------------------------------------------------------------------------------------
# configs 3, 4, 5: decoder cached self-attention, cross-attention, draft verify
# --------------------------------------------------------------------------------------------


def _lengths(seed, n, lo, hi):
    """Attended lengths L_i ~ U{lo..hi} (inclusive) from the seed: the draw the parity tests use."""
    return np.random.default_rng(seed).integers(lo, hi + 1, size=n, dtype=np.int64)


def host_cores() -> int:
    """Threads for the CPU baselines: every core this process may run on (no cap)."""
    return len(os.sched_getaffinity(0))


def _projected_cross_cache(xa, dev, seed):
    """Cross K/V of one layer as config 4 states them: the simulated encoder output xa
    [B, L, 1280] projected with this layer's seeded W_k, W_v ~ N(0, 1/1280) (unit-variance K/V),
    stored head-major [B, H, L, D] and viewed as [B, L, H, D]."""
    Bn, Ln, n_state = xa.shape
    g = torch.Generator(device=dev).manual_seed(seed)
    w = (torch.randn((2, n_state, n_state), generator=g, device=dev) * n_state ** -0.5).to(torch.bfloat16)
    kv = torch.empty((2, Bn, H, Ln, D), dtype=torch.bfloat16, device=dev)
    for j in range(2):
        kv[j].copy_((xa @ w[j]).view(Bn, Ln, H, D).permute(0, 2, 1, 3))
    return kv[0].permute(0, 2, 1, 3), kv[1].permute(0, 2, 1, 3)


def _head_major_cache(n_slots, Lmax, dev, seed):
    """K and V caches stored head-major [n_slots, H, Lmax, D], viewed as [n_slots, Lmax, H, D]."""
    g = torch.Generator(device=dev).manual_seed(seed)
    kv = torch.randn((2, n_slots, H, Lmax, D), generator=g, device=dev, dtype=torch.float32).to(torch.bfloat16)
    return kv[0].permute(0, 2, 1, 3), kv[1].permute(0, 2, 1, 3)


def bench_decode(dev, steps: int, warmup: int) -> dict:
    from whisperdrz_amd import flash_attn_with_kvcache, kvcache_workspace_size
    from whisperdrz_amd.attention import _WORKSPACES

    Bs, Lself, Lcross = 64, 448, 1500
    res = {}
    slots = torch.arange(Bs, dtype=torch.int32, device=dev)

    def q_new(seed, sq):
        g = torch.Generator(device=dev).manual_seed(seed)
        t = torch.randn((3, Bs, sq, H, D), generator=g, device=dev, dtype=torch.float32).to(torch.bfloat16)
        return t[0], t[1], t[2]

    def run_graph(name, body, bytes_per_layer, extra=None, kernels=()):
        torch.cuda.synchronize()
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            for _ in range(3):
                body()
        torch.cuda.current_stream().wait_stream(s)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            body()
        stream = torch.cuda.current_stream()
        for _ in range(warmup):
            graph.replay()
        ms = timed_events(graph.replay, steps, stream)
        gbs = bytes_per_layer * N_LAYERS / (ms * 1e-3) / 1e9
        log(f"[bench] {name}: {ms * 1e3 / N_LAYERS:.2f} us/layer, {gbs:.0f} GB/s ({100 * gbs / PEAK_HBM_GBS:.1f}% of HBM)")
        out = {
            "us_per_layer": round(ms * 1e3 / N_LAYERS, 3),
            "GB_per_s": round(gbs, 1),
            "roofline": {
                "bound": "hbm",
                "achieved": round(gbs, 1),
                "peak": PEAK_HBM_GBS,
                "unit": "GB/s",
                "frac": round(gbs / PEAK_HBM_GBS, 4),
                "traffic": summed_traffic(kernels),
                "traffic_source": "profiles/pmc_traffic.json (rocprofv3 FETCH_SIZE/WRITE_SIZE passes)",
                "bytes_per_layer": bytes_per_layer,
            },
            "graph": f"{N_LAYERS} layers in one hipGraph",
        }
        if extra:
            out.update(extra)
        del graph
        return out

    # shared per-layer caches: 32 distinct self caches (capacity 448) and cross caches (1500)
    log("[bench] decode: generating 32 self caches (64 x 448, K/V ~ N(0,1)) and 32 cross caches "
        "(64 x 1500, projected per layer from one N(0,1) encoder output), head-major bf16")
    self_kv = [_head_major_cache(Bs, Lself, dev, 3000 + i) for i in range(N_LAYERS)]
    gx = torch.Generator(device=dev).manual_seed(3999)
    xa = torch.randn((Bs, Lcross, H * D), generator=gx, device=dev, dtype=torch.float32).to(torch.bfloat16)
    cross_kv = [_projected_cross_cache(xa, dev, 4000 + i) for i in range(N_LAYERS)]
    del xa
    for sq in (1, 5):
        _WORKSPACES.reserve(dev, max(kvcache_workspace_size(Bs, sq, H, D, Lself),
                                     kvcache_workspace_size(Bs, sq, H, D, Lcross)))

    # ---- config 3: self-attention decode, sq=1, L_i ~ U[1,448] including the new token ----
    L3 = _lengths(3, Bs, 1, Lself)
    cs3 = torch.from_numpy((L3 - 1).astype(np.int32)).to(dev)
    q3 = [q_new(5000 + i, 1) for i in range(N_LAYERS)]
    o3 = [torch.empty((Bs, 1, H, D), dtype=torch.bfloat16, device=dev) for _ in range(N_LAYERS)]

    def body3():
        for i in range(N_LAYERS):
            q, k, v = q3[i]
            flash_attn_with_kvcache(q, self_kv[i][0], self_kv[i][1], k=k, v=v, cache_seqlens=cs3,
                                    cache_batch_idx=slots, softmax_scale=0.125, causal=True, out=o3[i])

    sumL3 = int(L3.sum())
    bytes3 = 2 * H * D * E * sumL3 + 2 * H * D * E * Bs + 2 * H * D * E * Bs + 8 * Bs
    res["config3_self_decode"] = run_graph("config3 self sq=1", body3, bytes3, {"sum_L": sumL3},
                                           kernels=("kv_attn_kernel<wdrz::Bf16, 1, true, false>",))

    # ---- config 4: cross-attention decode, sq=1, 1500 keys per stream ----
    q4 = [q_new(6000 + i, 1)[0] for i in range(N_LAYERS)]
    o4 = [torch.empty((Bs, 1, H, D), dtype=torch.bfloat16, device=dev) for _ in range(N_LAYERS)]

    def body4():
        for i in range(N_LAYERS):
            flash_attn_with_kvcache(q4[i], cross_kv[i][0], cross_kv[i][1], cache_batch_idx=slots,
                                    softmax_scale=0.125, causal=False, out=o4[i])

    bytes4 = 2 * Bs * Lcross * H * D * E + 2 * H * D * E * Bs + 4 * Bs
    res["config4_cross_decode"] = run_graph(
        "config4 cross sq=1", body4, bytes4,
        {"inputs": "per layer K = xa W_k, V = xa W_v with xa ~ N(0,1) [64, 1500, 1280] bf16 (one simulated "
                   "encoder output) and seeded W_k, W_v ~ N(0, 1/1280) [1280, 1280] per layer; queries ~ N(0,1)"},
        kernels=("kv_attn_kernel<wdrz::Bf16, 1, false, true>",))

    # ---- config 5: 5-token draft verify (self, causal within the draft) + cross ----
    sq = 5
    L5 = _lengths(5, Bs, sq, Lself)
    cs5 = torch.from_numpy((L5 - sq).astype(np.int32)).to(dev)
    q5 = [q_new(7000 + i, sq) for i in range(N_LAYERS)]
    qx5 = [q_new(8000 + i, sq)[0] for i in range(N_LAYERS)]
    o5 = [torch.empty((Bs, sq, H, D), dtype=torch.bfloat16, device=dev) for _ in range(N_LAYERS)]
    ox5 = [torch.empty((Bs, sq, H, D), dtype=torch.bfloat16, device=dev) for _ in range(N_LAYERS)]

    def body5():
        for i in range(N_LAYERS):
            q, k, v = q5[i]
            flash_attn_with_kvcache(q, self_kv[i][0], self_kv[i][1], k=k, v=v, cache_seqlens=cs5,
                                    cache_batch_idx=slots, softmax_scale=0.125, causal=True, out=o5[i])
            flash_attn_with_kvcache(qx5[i], cross_kv[i][0], cross_kv[i][1], cache_batch_idx=slots,
                                    softmax_scale=0.125, causal=False, out=ox5[i])

    sumL5 = int(L5.sum())
    bytes5_self = 2 * H * D * E * sumL5 + 4 * H * D * E * Bs * sq + 8 * Bs
    bytes5_cross = 2 * Bs * Lcross * H * D * E + 2 * H * D * E * Bs * sq + 4 * Bs
    res["config5_verify_self_plus_cross"] = run_graph(
        "config5 verify sq=5 (self+cross)", body5, bytes5_self + bytes5_cross,
        {"sum_L": sumL5, "bytes_self_per_layer": bytes5_self, "bytes_cross_per_layer": bytes5_cross},
        kernels=("kv_mq_kernel<wdrz::Bf16, true, 8, 4>", "kv_mq_kernel<wdrz::Bf16, false, 8, 4>"),
    )
    # ---- prefill: a 224-token prompt into empty self caches (the window's first call) ----
    sqp = 224
    csp = torch.zeros(Bs, dtype=torch.int32, device=dev)
    qp = [q_new(9000 + i, sqp) for i in range(8)]

    def bodyp():
        for i in range(8):
            q, k, v = qp[i]
            flash_attn_with_kvcache(q, self_kv[i][0], self_kv[i][1], k=k, v=v, cache_seqlens=csp,
                                    cache_batch_idx=slots, softmax_scale=0.125, causal=True)

    for _ in range(warmup):
        bodyp()
    us_p = timed_events(bodyp, steps, torch.cuda.current_stream()) * 1e3 / 8
    flop_p = 4.0 * Bs * H * D * sqp * (sqp + 1) / 2
    log(f"[bench] prefill sq={sqp} into empty caches: {us_p:.1f} us/layer, {flop_p / us_p / 1e6:.1f} TFLOP/s")
    bytes_p = 6 * Bs * sqp * H * D * E  # Q, new K and V read, K and V appended, O written
    res["prefill_self_sq224"] = {
        "workload": "64 streams append a 224-token prompt to empty 448-row self caches (causal), bf16; "
                    "kv_prefill_kernel in 256-query blocks",
        "us_per_layer": round(us_p, 2), "tflops": round(flop_p / us_p / 1e6, 2),
        "roofline": {"bound": "hbm", "achieved": round(bytes_p / us_p / 1e3, 1), "peak": PEAK_HBM_GBS,
                     "unit": "GB/s", "frac": round(bytes_p / us_p / 1e3 / PEAK_HBM_GBS, 4),
                     "traffic": measured_traffic("kv_prefill_kernel<wdrz::Bf16, true>"), "bytes_per_layer": bytes_p}}

    # ---- the same prompt's cross-attention over the 1500 encoder rows ----
    def bodyc():
        for i in range(8):
            flash_attn_with_kvcache(qp[i][0], cross_kv[i][0], cross_kv[i][1], cache_batch_idx=slots,
                                    softmax_scale=0.125, causal=False)

    for _ in range(warmup):
        bodyc()
    us_c = timed_events(bodyc, steps, torch.cuda.current_stream()) * 1e3 / 8
    flop_c = 4.0 * Bs * H * D * sqp * Lcross
    bytes_c = 2 * Bs * Lcross * H * D * E + 2 * Bs * sqp * H * D * E  # K, V once; Q read, O written
    log(f"[bench] prefill cross sq={sqp} over {Lcross} rows: {us_c:.1f} us/layer, {flop_c / us_c / 1e6:.1f} TFLOP/s, "
        f"{bytes_c / us_c / 1e3:.0f} GB/s")
    res["prefill_cross_sq224"] = {
        "workload": f"64 streams, {sqp} prompt queries over {Lcross} cross rows (non-causal), bf16; "
                    "dense_pipe_kernel<Bf16, 2> through the slot map (256-query items)",
        "us_per_layer": round(us_c, 2), "tflops": round(flop_c / us_c / 1e6, 2),
        "roofline": {"bound": "hbm", "achieved": round(bytes_c / us_c / 1e3, 1), "peak": PEAK_HBM_GBS,
                     "unit": "GB/s", "frac": round(bytes_c / us_c / 1e3 / PEAK_HBM_GBS, 4), "traffic": None,
                     "bytes_per_layer": bytes_c}}
    del self_kv, cross_kv, qp
    torch.cuda.empty_cache()
    return res


# --------------------------------------------------------------------------------------------
# CPU baseline: the reference's CPU torch path (torch SDPA, fp32), bounded sample
# --------------------------------------------------------------------------------------------


# --------------------------------------------------------------------------------------------
# DTW alignment prep (_dtw_prep_batch, dtw_align.py:700-753)
# --------------------------------------------------------------------------------------------

DTW_B, DTW_H, DTW_T, DTW_A = 16, 10, 448, 1500  # chunks x large-v3 alignment heads x text x audio


def _dtw_inputs(dev, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    w = 2.5 * torch.randn((DTW_B, DTW_H, DTW_T, DTW_A), generator=g, device=dev)
    rng = np.random.default_rng(seed)
    lens = [int(x) for x in rng.integers(DTW_T // 2, DTW_T + 1, DTW_B)]
    return w, lens, [DTW_A] * DTW_B


def dtw_bytes(lens, caps) -> int:
    """Algorithmic HBM bytes of one prep: every valid score read once (4 B per column < cap of
    every row of every head) and the [B, T, max cap] result written once."""
    read = sum(4 * DTW_H * DTW_T * c for c in caps)
    return read + 4 * DTW_B * DTW_T * max(caps)


def bench_dtw(dev, steps: int, warmup: int) -> dict:
    from whisperdrz_amd import dtw_prep
    from oracle.dtw_oracle import dtw_prep_torch

    n_in = 4
    log(f"[bench] dtw prep: {n_in} distinct score tensors [{DTW_B}, {DTW_H}, {DTW_T}, {DTW_A}] fp32")
    inputs = [_dtw_inputs(dev, 5000 + i) for i in range(n_in)]
    outs = [None] * n_in

    def step():
        for i, (w, lens, caps) in enumerate(inputs):
            outs[i] = dtw_prep(w, lens, caps, 7)

    stream = torch.cuda.current_stream()
    for _ in range(warmup):
        step()
    ms = timed_events(step, steps, stream) / n_in
    nbytes = dtw_bytes(inputs[0][1], inputs[0][2])
    gbs = nbytes / (ms * 1e-3) / 1e9
    log(f"[bench] dtw prep: {ms * 1e3:.1f} us per prep, {gbs:.0f} GB/s algorithmic ({100 * gbs / PEAK_HBM_GBS:.1f}% of HBM)")
    # The reference's op sequence (torch ops; sort-based median in place of its Triton kernel)
    # on the same GPU, for comparison.
    w, lens, caps = inputs[0]
    dtw_prep_torch(w, lens, caps)
    ms_torch = timed_events(lambda: dtw_prep_torch(w, lens, caps), 3, stream)
    log(f"[bench] dtw prep: torch op sequence on the GPU {ms_torch * 1e3:.0f} us ({ms_torch / ms:.1f}x)")
    del inputs, outs
    torch.cuda.empty_cache()
    qk = bench_dtw_qk(dev, steps, warmup)
    dec_attn = bench_dtw_decoder_attention(dev, steps, warmup)
    mf = bench_median_filter(dev, steps, warmup)
    return {
        "workload": f"_dtw_prep_batch: B={DTW_B} chunks x H={DTW_H} alignment heads x T_text={DTW_T} x "
        f"T_audio={DTW_A} fp32 scores, caps={DTW_A}, lens ~ U[{DTW_T // 2},{DTW_T}], median width 7; "
        f"{n_in} distinct inputs in rotation",
        "us_per_prep": round(ms * 1e3, 2),
        "GB_per_s": round(gbs, 1),
        "roofline": {
            "bound": "hbm",
            "achieved": round(gbs, 1),
            "peak": PEAK_HBM_GBS,
            "unit": "GB/s",
            "frac": round(gbs / PEAK_HBM_GBS, 4),
            "traffic": summed_traffic(DTW_KERNELS),
            "traffic_source": "profiles/pmc_traffic.json (rocprofv3 FETCH_SIZE/WRITE_SIZE passes)",
            "bytes_per_prep": nbytes,
            "kernels": list(DTW_KERNELS),
        },
        "torch_ops_gpu_us": round(ms_torch * 1e3, 1),
        "compute_attention": qk,
        "decoder_attention": dec_attn,
        "median_filter": mf,
    }


def bench_median_filter(dev, steps: int, warmup: int) -> dict:
    """median_filter (dtw_align.py:156-167), width 7, on the prep's [16, 10, 448, 1500] fp32 scores:
    HBM-bound, the scores read once and the result written once."""
    from oracle.dtw_oracle import median_filter_torch
    from whisperdrz_amd import median_filter

    g = torch.Generator(device=dev).manual_seed(6600)
    x = torch.randn((DTW_B, DTW_H, DTW_T, DTW_A), generator=g, device=dev)
    stream = torch.cuda.current_stream()
    for _ in range(warmup):
        median_filter(x, 7)
    us = timed_events(lambda: median_filter(x, 7), steps, stream) * 1e3
    median_filter_torch(x, 7)
    us_torch = timed_events(lambda: median_filter_torch(x, 7), 3, stream) * 1e3
    nbytes = 2 * x.numel() * 4
    gbs = nbytes / (us * 1e-6) / 1e9
    log(f"[bench] median_filter width 7: {us:.1f} us, {gbs:.0f} GB/s ({100 * gbs / PEAK_HBM_GBS:.1f}% of HBM); "
        f"torch sort-based form {us_torch:.0f} us")
    del x
    torch.cuda.empty_cache()
    return {
        "us": round(us, 2),
        "roofline": {"bound": "hbm", "achieved": round(gbs, 1), "peak": PEAK_HBM_GBS, "unit": "GB/s",
                     "frac": round(gbs / PEAK_HBM_GBS, 4), "traffic": measured_traffic("median_filter_kernel<3>"),
                     "bytes_per_call": nbytes, "kernel": "median_filter_kernel<3>"},
        "torch_sort_gpu_us": round(us_torch, 1),
    }


def bench_dtw_decoder_attention(dev, steps: int, warmup: int) -> dict:
    """The uncached decoder forward that feeds the alignment (dtw_align.py:1183, model.py:288):
    per layer a causal self-attention over the padded text [16, 20, 448, 64] and a cross-attention
    of those 448 rows over the 1500 encoder rows, bf16, 8 distinct layers in rotation. Algorithmic
    FLOP: 4*B*H*T*T*D/2 for the causal half (keys at or before each query) + 4*B*H*T*A*D."""
    from whisperdrz_amd import scaled_dot_product_attention

    B, T, A, n_l = DTW_B, DTW_T, DTW_A, 8
    g = torch.Generator(device=dev).manual_seed(6500)
    layers = []
    for _ in range(n_l):
        q, k, v = (torch.randn((B, H, T, D), generator=g, device=dev).to(torch.bfloat16) for _ in range(3))
        kx, vx = (torch.randn((B, H, A, D), generator=g, device=dev).to(torch.bfloat16) for _ in range(2))
        layers.append((q, k, v, kx, vx))
    stream = torch.cuda.current_stream()

    def self_attn():
        for q, k, v, _, _ in layers:
            scaled_dot_product_attention(q, k, v, is_causal=True, scale=0.125)

    def cross_attn():
        for q, _, _, kx, vx in layers:
            scaled_dot_product_attention(q, kx, vx, is_causal=False, scale=0.125)

    for _ in range(warmup):
        self_attn()
        cross_attn()
    us_self = timed_events(self_attn, steps, stream) * 1e3 / n_l
    us_cross = timed_events(cross_attn, steps, stream) * 1e3 / n_l
    f_self = 4.0 * B * H * T * T * D / 2
    f_cross = 4.0 * B * H * T * A * D
    t_self = f_self / (us_self * 1e-6) / 1e12
    t_cross = f_cross / (us_cross * 1e-6) / 1e12
    log(f"[bench] dtw decoder attention: causal self {us_self:.1f} us/layer ({t_self:.0f} TFLOP/s), "
        f"cross {us_cross:.1f} us/layer ({t_cross:.0f} TFLOP/s)")
    del layers
    torch.cuda.empty_cache()

    def roof(t, kernel):
        return {"bound": "mfma", "achieved": round(t, 1), "peak": PEAK_BF16_TFLOPS, "unit": "TFLOP/s",
                "frac": round(t / PEAK_BF16_TFLOPS, 4), "traffic": None, "kernel": kernel}

    return {
        "workload": f"uncached decoder attention for DTW: B={B} chunks, H={H}, T_text={T}, T_audio={A}, bf16",
        "causal_self_us_per_layer": round(us_self, 2),
        "causal_self_roofline": roof(t_self, "dense_mfma_kernel<Bf16, true>"),
        "cross_us_per_layer": round(us_cross, 2),
        "cross_roofline": roof(t_cross, "dense_pipe_kernel<Bf16, 2> (256-query items)"),
    }


# large-v3 alignment heads (layer, head), decoded from the reference's LARGE_V3_ALIGNMENT_HEADS
# bitmask (dtw_align.py:43-60): one head in each of 10 layers.
DTW_HEADS = [(7, 0), (10, 17), (12, 18), (13, 12), (16, 1), (17, 14), (19, 11), (21, 4), (24, 1), (25, 6)]


def bench_dtw_qk(dev, steps: int, warmup: int) -> dict:
    """compute_attention at the bench shape: the 10 alignment heads' Q/K slices read in place from
    per-layer captures [16, 448, 1280] / [16, 1500, 1280] bf16, fp32 scores written."""
    from whisperdrz_amd import compute_attention, dtw_attention_prep, dtw_prep

    n_layers, n_heads = 32, H
    mask = torch.zeros(n_layers, n_heads, dtype=torch.bool)
    for l, h in DTW_HEADS:
        mask[l, h] = True
    g = torch.Generator(device=dev).manual_seed(6000)
    q_out = [None] * n_layers
    k_out = [None] * n_layers
    for l, _ in DTW_HEADS:
        q_out[l] = torch.randn((DTW_B, DTW_T, n_heads * D), generator=g, device=dev).to(torch.bfloat16)
        k_out[l] = torch.randn((DTW_B, DTW_A, n_heads * D), generator=g, device=dev).to(torch.bfloat16)
    stream = torch.cuda.current_stream()
    for _ in range(warmup):
        compute_attention(q_out, k_out, mask)
    ms = timed_events(lambda: compute_attention(q_out, k_out, mask), steps, stream)
    nbytes = 4 * DTW_B * DTW_H * DTW_T * DTW_A + 2 * DTW_B * DTW_H * (DTW_T + DTW_A) * D
    gbs = nbytes / (ms * 1e-3) / 1e9

    def torch_ref():  # the reference's gather + fp32 batched matmul (dtw_align.py:565-585)
        s = D ** -0.25
        qs = torch.stack([q_out[l].view(DTW_B, DTW_T, n_heads, D)[:, :, h] for l, h in DTW_HEADS]).float() * s
        ks = torch.stack([k_out[l].view(DTW_B, DTW_A, n_heads, D)[:, :, h] for l, h in DTW_HEADS]).float() * s
        return (qs @ ks.transpose(-1, -2)).transpose(0, 1).contiguous()

    torch_ref()
    ms_torch = timed_events(torch_ref, 3, stream)
    log(f"[bench] compute_attention: {ms * 1e3:.1f} us, {gbs:.0f} GB/s ({100 * gbs / PEAK_HBM_GBS:.1f}% of HBM); "
        f"torch gather + fp32 matmul {ms_torch * 1e3:.0f} us")
    # The fused entry (scores recomputed inside both prep passes, never stored) against the
    # two-call chain compute_attention -> dtw_prep, on the bench's lengths and caps.
    rng = np.random.default_rng(5000)
    lens = [int(x) for x in rng.integers(DTW_T // 2, DTW_T + 1, DTW_B)]
    caps = [DTW_A] * DTW_B
    for _ in range(warmup):
        dtw_attention_prep(q_out, k_out, mask, lens, caps)
    ms_fused = timed_events(lambda: dtw_attention_prep(q_out, k_out, mask, lens, caps), steps, stream)
    ms_chain = timed_events(lambda: dtw_prep(compute_attention(q_out, k_out, mask), lens, caps), steps, stream)
    log(f"[bench] fused attention+prep: {ms_fused * 1e3:.1f} us; chain compute_attention + dtw_prep "
        f"{ms_chain * 1e3:.1f} us")
    del q_out, k_out
    torch.cuda.empty_cache()
    return {
        "us": round(ms * 1e3, 2),
        "roofline": {
            "bound": "hbm",
            "achieved": round(gbs, 1),
            "peak": PEAK_HBM_GBS,
            "unit": "GB/s",
            "frac": round(gbs / PEAK_HBM_GBS, 4),
            "traffic": measured_traffic("dtw_qk_kernel<wdrz::Bf16>"),
            "bytes_per_call": nbytes,
            "kernel": "dtw_qk_kernel<Bf16>",
        },
        "torch_gpu_us": round(ms_torch * 1e3, 1),
        "fused_attention_prep_us": round(ms_fused * 1e3, 2),
        "chain_attention_then_prep_us": round(ms_chain * 1e3, 2),
    }


# --------------------------------------------------------------------------------------------
# a whole decode step (large-v3 decoder, random weights, 64 streams, one captured hipGraph)
# --------------------------------------------------------------------------------------------


def bench_decode_step(dev, steps: int, warmup: int) -> dict:
    from whisperdrz_amd.decoder import BucketedDecodeGraphs, TextDecoderStack
    from whisperdrz_amd.kv_cache import KVSlotPool

    Bs, n_vocab, n_layer = 64, 51866, 32
    steps = min(steps, 20)
    torch.manual_seed(0)
    log("[bench] decode step: large-v3 decoder (random weights, bf16), 64 streams, 32 layers")
    with torch.device(dev):
        dec = TextDecoderStack(n_vocab, 448, H * D, H, n_layer).to(torch.bfloat16).eval()
    pool = KVSlotPool(n_layer, Bs, H, D, self_len=448, cross_len=1500, dtype=torch.bfloat16, device=dev)
    pool.arena.view(torch.bfloat16).normal_()
    lens0 = torch.from_numpy(_lengths(8, Bs, 1, 400).astype(np.int32)).to(dev)
    tokens = torch.randint(0, n_vocab, (Bs, 1), device=dev)
    slots = torch.arange(Bs, device=dev)
    res = {}
    for fused in (True, False):
        dec.fused_small_ops = fused
        for c in pool.self_kv:
            c.seq_lens.copy_(lens0)
        graphs = BucketedDecodeGraphs(dec, pool, n_vocab, buckets=[Bs])
        with torch.no_grad():
            graphs.capture(Bs)
            positions = lens0.long()
            for c in pool.self_kv:
                c.seq_lens.copy_(lens0)
            for _ in range(warmup):
                graphs.forward(tokens, positions, slots)
            ms = timed_events(lambda: graphs.forward(tokens, positions, slots), steps, torch.cuda.current_stream())
        res["fused" if fused else "unfused"] = ms
        log(f"[bench] decode step ({'fused add+LayerNorm' if fused else 'torch add, LayerNorm'}): {ms:.3f} ms "
            f"per step, {Bs / ms * 1e3:.0f} tokens/s")
        del graphs
    # the step's logits (model.py:609-613): [64, 1280] x [1280, 51866] against the tied embedding,
    # a plain library GEMM (hipBLASLt), timed on its own: 32 launches in one graph
    with torch.no_grad():
        h = torch.randn((Bs, H * D), device=dev).to(torch.bfloat16)
        w = dec.token_embedding.weight.to(torch.bfloat16)
        logits = torch.empty((Bs, n_vocab), dtype=torch.bfloat16, device=dev)
        torch.matmul(h, w.T, out=logits)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for _ in range(N_LAYERS):
                torch.matmul(h, w.T, out=logits)
        g.replay()
        ms_l = timed_events(g.replay, 10, torch.cuda.current_stream()) / N_LAYERS
        del g
    lbytes = n_vocab * H * D * 2 + Bs * H * D * 2 + Bs * n_vocab * 2
    res["logits_us"] = ms_l * 1e3
    res["logits_gbs"] = lbytes / (ms_l * 1e-3) / 1e9
    log(f"[bench] decode step logits GEMM: {ms_l * 1e3:.1f} us, {res['logits_gbs']:.0f} GB/s "
        f"({100 * res['logits_gbs'] / PEAK_HBM_GBS:.1f}% of HBM)")
    del dec, pool
    torch.cuda.empty_cache()
    return {
        "workload": "one cached decode step of the large-v3 decoder (random bf16 weights, 32 layers, vocab "
        "51866), 64 streams, self lengths U[1,400], cross 1500, captured in one hipGraph",
        "ms_per_step": round(res["fused"], 4),
        "tokens_per_s": round(Bs / res["fused"] * 1e3, 1),
        "ms_per_step_unfused_small_ops": round(res["unfused"], 4),
        "logits": {
            "workload": "tied-embedding logits [64, 1280] x [1280, 51866] bf16 (model.py:609-613), hipBLASLt",
            "us": round(res["logits_us"], 2),
            "roofline": {"bound": "hbm", "achieved": round(res["logits_gbs"], 1), "peak": PEAK_HBM_GBS, "unit": "GB/s",
                         "frac": round(res["logits_gbs"] / PEAK_HBM_GBS, 4), "traffic": None,
                         "bytes": n_vocab * H * D * 2 + Bs * H * D * 2 + Bs * n_vocab * 2},
        },
    }


# --------------------------------------------------------------------------------------------
# cross-attention fill after the encoder (prefill_flash, model.py:851-862)
# --------------------------------------------------------------------------------------------

FILL_B, FILL_L = 16, 1500


def bench_cross_fill(dev, steps: int, warmup: int) -> dict:
    """The encoder output of 16 windows projected into every layer's cross cache: per layer one
    key / value GEMM ([16*1500, 1280] x [1280, 2560], hipBLASLt) and one wdrz_kv_fill into the
    head-major slots. The fill alone is HBM-bound: it reads and writes 2 x 16 x 1500 x 1280 bf16."""
    import torch.nn.functional as F

    from whisperdrz_amd.decoder import TextDecoderStack
    from whisperdrz_amd.kv_cache import KVSlotPool

    torch.manual_seed(0)
    with torch.device(dev):
        dec = TextDecoderStack(51866, 448, H * D, H, N_LAYERS).to(torch.bfloat16).eval()
    pool = KVSlotPool(N_LAYERS, FILL_B, H, D, self_len=448, cross_len=FILL_L, dtype=torch.bfloat16, device=dev)
    g = torch.Generator(device=dev).manual_seed(9000)
    xa = torch.randn((FILL_B, FILL_L, H * D), generator=g, device=dev).to(torch.bfloat16)
    slots = torch.arange(FILL_B, device=dev)
    stream = torch.cuda.current_stream()
    kvs = [torch.randn((FILL_B, FILL_L, 2, H, D), generator=g, device=dev).to(torch.bfloat16) for _ in range(4)]

    def fill_only():
        for i, c in enumerate(pool.cross_kv[:4]):
            c.set_cross_attention(kvs[i][:, :, 0], kvs[i][:, :, 1], slots)

    def fill_torch():  # the reference's index_put on the same views
        for i, c in enumerate(pool.cross_kv[:4]):
            c.k_cache[slots, :FILL_L] = kvs[i][:, :, 0]
            c.v_cache[slots, :FILL_L] = kvs[i][:, :, 1]

    def full():
        for blk, c in zip(dec.blocks, pool.cross_kv):
            w, b = blk.cross_attn.kv_weight()
            kv = F.linear(xa, w, b).view(FILL_B, FILL_L, 2, H, D)
            c.set_cross_attention(kv[:, :, 0], kv[:, :, 1], slots)

    with torch.no_grad():
        for _ in range(warmup):
            fill_only()
            full()
        us = timed_events(fill_only, steps, stream) * 1e3 / 4
        fill_torch()
        us_torch = timed_events(fill_torch, 3, stream) * 1e3 / 4
        ms_full = timed_events(full, max(3, steps // 4), stream)
    nbytes = 2 * 2 * FILL_B * FILL_L * H * D * E  # K and V, read once and written once
    gbs = nbytes / (us * 1e-6) / 1e9
    log(f"[bench] cross fill: wdrz_kv_fill {us:.1f} us per layer, {gbs:.0f} GB/s ({100 * gbs / PEAK_HBM_GBS:.1f}% of "
        f"HBM); torch index_put {us_torch:.1f} us; GEMM + fill for 32 layers {ms_full:.2f} ms")
    del dec, pool, kvs
    torch.cuda.empty_cache()
    return {
        "workload": f"prefill_flash cross fill: {FILL_B} windows x {FILL_L} encoder rows, 32 layers, per layer one "
        "[24000, 1280] x [1280, 2560] key/value GEMM (hipBLASLt) and one wdrz_kv_fill into head-major slots",
        "fill_us_per_layer": round(us, 2),
        "roofline": {
            "bound": "hbm",
            "achieved": round(gbs, 1),
            "peak": PEAK_HBM_GBS,
            "unit": "GB/s",
            "frac": round(gbs / PEAK_HBM_GBS, 4),
            "traffic": measured_traffic("kv_fill_kernel"),
            "bytes_per_layer": nbytes,
            "kernel": "kv_fill_kernel",
        },
        "torch_index_put_us_per_layer": round(us_torch, 1),
        "ms_32_layers_gemm_plus_fill": round(ms_full, 3),
    }


# --------------------------------------------------------------------------------------------
# log-mel front end (LogMelSpectrogram, audio.py:81-156)
# --------------------------------------------------------------------------------------------

MEL_B, MEL_N, MEL_MELS = 16, 480000, 128


def mel_bytes() -> int:
    """Bytes a batch cannot do without: the samples read once, the mel written once (fp32). The work
    beside them is small (a 400-point real FFT per frame), so the front end's roofline is HBM."""
    return 4 * MEL_B * (MEL_N + MEL_MELS * 3000)


def bench_logmel(dev, steps: int, warmup: int) -> dict:
    from whisperdrz_amd import log_mel_spectrogram

    g = torch.Generator(device=dev).manual_seed(7000)
    audio = [0.1 * torch.randn((MEL_B, MEL_N), generator=g, device=dev) for _ in range(2)]
    stream = torch.cuda.current_stream()
    for _ in range(warmup):
        for x in audio:
            log_mel_spectrogram(x, MEL_MELS, 3000)
    ms = timed_events(lambda: [log_mel_spectrogram(x, MEL_MELS, 3000) for x in audio], steps, stream) / len(audio)
    gbs = mel_bytes() / (ms * 1e-3) / 1e9
    log(f"[bench] log-mel: {ms * 1e3:.1f} us per {MEL_B} x 30 s windows ({MEL_B / ms * 1e3:.0f} windows/s), "
        f"{gbs:.0f} GB/s ({100 * gbs / PEAK_HBM_GBS:.1f}% of HBM)")
    del audio
    return {
        "workload": f"LogMelSpectrogram: {MEL_B} windows of 30 s (480000 samples, fp32, on the GPU) -> "
        f"[{MEL_B}, {MEL_MELS}, 3000]",
        "us_per_batch": round(ms * 1e3, 2),
        "windows_per_s": round(MEL_B / ms * 1e3, 1),
        "roofline": {
            "bound": "hbm",
            "achieved": round(gbs, 1),
            "peak": PEAK_HBM_GBS,
            "unit": "GB/s",
            "frac": round(gbs / PEAK_HBM_GBS, 4),
            "traffic": None,
            "bytes_per_batch": mel_bytes(),
            "kernel": "logmel_spec_kernel, logmel_finish_kernel",
        },
    }


def logmel_cpu_baseline(budget_s: float = 8.0) -> dict:
    """The reference's op sequence (torch.stft + filterbank + log) on the host cores, one window."""
    from oracle.mel_oracle import log_mel_torch, mel_filterbank

    cores = host_cores()
    torch.set_num_threads(cores)
    fb = mel_filterbank(MEL_MELS)
    x = 0.1 * torch.randn(MEL_N, generator=torch.Generator().manual_seed(1))
    log_mel_torch(x, fb, 3000)
    times = []
    t_end = time.perf_counter() + budget_s
    while len(times) < 3 or (time.perf_counter() < t_end and len(times) < 200):
        t0 = time.perf_counter()
        log_mel_torch(x, fb, 3000)
        times.append(time.perf_counter() - t0)
    med = float(np.median(times))
    log(f"[bench] log-mel cpu baseline: {med * 1e3:.2f} ms per window on {cores} threads")
    return {
        "value": round(1.0 / med, 1),
        "unit": "windows/s",
        "cores": cores,
        "kind": "port",
        "sample": f"torch CPU fp32 op sequence of LogMelSpectrogram (audio.py:141-156, torch.stft) on one 30-s "
        f"window, median of {len(times)} runs ({med * 1e3:.2f} ms each)",
    }


DTW_KERNELS = ("dtw_rowcol_kernel<6>", "dtw_col_merge_kernel", "dtw_seg_kernel")


def dtw_cpu_baseline(budget_s: float = 12.0) -> dict:
    """The reference's op sequence in torch fp32 on the host cores, on one chunk."""
    from oracle.dtw_oracle import dtw_prep_torch

    cores = host_cores()
    torch.set_num_threads(cores)
    g = torch.Generator().manual_seed(1)
    w = 2.5 * torch.randn((1, DTW_H, DTW_T, DTW_A), generator=g)
    lens, caps = [DTW_T - 17], [DTW_A]
    nbytes = 4 * DTW_H * DTW_T * DTW_A + 4 * DTW_T * DTW_A
    dtw_prep_torch(w, lens, caps)
    times = []
    t_end = time.perf_counter() + budget_s
    while len(times) < 3 or (time.perf_counter() < t_end and len(times) < 100):
        t0 = time.perf_counter()
        dtw_prep_torch(w, lens, caps)
        times.append(time.perf_counter() - t0)
    med = float(np.median(times))
    log(f"[bench] dtw cpu baseline: {med * 1e3:.1f} ms per chunk on {cores} threads -> {nbytes / med / 1e9:.2f} GB/s")
    return {
        "value": round(nbytes / med / 1e9, 3),
        "unit": "GB/s",
        "cores": cores,
        "kind": "port",
        "sample": f"torch CPU fp32 op sequence of _dtw_prep_batch (dtw_align.py:720-746, sort-based median "
        f"of dtw_align.py:65-78) on one chunk H={DTW_H} T={DTW_T} A={DTW_A}, median of {len(times)} runs "
        f"({med * 1e3:.1f} ms each)",
    }


def decode_cpu_baseline(budget_s: float = 15.0) -> dict:
    """The reference's CPU path for decode configs 3, 4 and 5 (``_sdpa_attn_with_kvcache``,
    model.py:20-76, as the oracle restates it) in torch fp32 on the host cores: one layer of
    each config at full size (64 streams, the same seeded lengths). Reported in the GPU line's
    unit: that config's algorithmic bytes per layer (counted in bf16, as the GPU line counts
    them) per second of CPU time."""
    from oracle.attention_oracle import kvcache_torch

    cores = host_cores()
    torch.set_num_threads(cores)
    Bs, Lself, Lcross = 64, 448, 1500
    g = torch.Generator().manual_seed(2)
    idx = torch.arange(Bs, dtype=torch.int32)
    L3 = _lengths(3, Bs, 1, Lself)
    L5 = _lengths(5, Bs, 5, Lself)
    kself, vself = (torch.randn((Bs, Lself, H, D), generator=g) for _ in range(2))
    kx, vx = (torch.randn((Bs, Lcross, H, D), generator=g) for _ in range(2))

    def new(sq):
        return tuple(torch.randn((Bs, sq, H, D), generator=g) for _ in range(3))

    q1, k1, v1 = new(1)
    q5, k5, v5 = new(5)
    qx5 = new(5)[0]
    cs3 = torch.from_numpy((L3 - 1).astype(np.int32))
    cs5 = torch.from_numpy((L5 - 5).astype(np.int32))
    cases = {
        "config3_self_decode": (lambda: kvcache_torch(q1, kself, vself, k1, v1, cs3, idx, 0.125),
                                2 * H * D * E * int(L3.sum()) + 4 * H * D * E * Bs + 8 * Bs),
        "config4_cross_decode": (lambda: kvcache_torch(q1, kx, vx, None, None, None, idx, 0.125),
                                 2 * Bs * Lcross * H * D * E + 2 * H * D * E * Bs + 4 * Bs),
        "config5_verify_self_plus_cross": (
            lambda: (kvcache_torch(q5, kself, vself, k5, v5, cs5, idx, 0.125),
                     kvcache_torch(qx5, kx, vx, None, None, None, idx, 0.125)),
            2 * H * D * E * int(L5.sum()) + 4 * H * D * E * Bs * 5 + 8 * Bs + 2 * Bs * Lcross * H * D * E
            + 2 * H * D * E * Bs * 5 + 4 * Bs),
    }
    out = {}
    per_case = budget_s / len(cases)
    for name, (fn, nbytes) in cases.items():
        fn()  # warm-up
        times = []
        t_end = time.perf_counter() + per_case
        while len(times) < 3 or (time.perf_counter() < t_end and len(times) < 50):
            t0 = time.perf_counter()
            fn()
            times.append(time.perf_counter() - t0)
        med = float(np.median(times))
        log(f"[bench] {name} cpu baseline: {med * 1e3:.1f} ms per layer on {cores} threads -> "
            f"{nbytes / med / 1e9:.2f} GB/s")
        out[name] = {
            "value": round(nbytes / med / 1e9, 3),
            "unit": "GB/s",
            "cores": cores,
            "kind": "port",
            "sample": f"torch CPU fp32 restatement of _sdpa_attn_with_kvcache (model.py:20-76: append, gather, "
            f"bottom-right mask, SDPA) on one full layer of the config (64 streams), median of {len(times)} runs "
            f"({med * 1e3:.1f} ms each); bytes = the GPU line's bf16 algorithmic bytes per layer",
        }
    return out


def _cpu_time(fn, budget_s: float, min_runs: int = 3):
    fn()  # warm-up
    times = []
    t_end = time.perf_counter() + budget_s
    while len(times) < min_runs or (time.perf_counter() < t_end and len(times) < 50):
        t0 = time.perf_counter()
        fn()
        times.append(time.perf_counter() - t0)
    return float(np.median(times)), len(times)


def extra_cpu_baselines(budget_s: float = 6.0) -> dict:
    """The reference's CPU paths beside the remaining rows, bounded samples in fp32 on the host
    cores: the decode step (one layer of the large-v3 decoder for 64 streams through the oracle's
    _sdpa_attn_with_kvcache restatement, scaled to 32 layers), the cross fill (one layer's key /
    value projection of one window and its index_put, scaled to 16 windows x 32 layers) and
    median_filter (the sort-based form of dtw_align.py:65-78 on one chunk's 10 heads)."""
    import torch.nn.functional as F

    from oracle.attention_oracle import kvcache_torch
    from oracle.dtw_oracle import median_filter_torch
    from whisperdrz_amd.decoder import ResidualAttentionBlock
    from whisperdrz_amd.kv_cache import FlashKVCache

    cores = host_cores()
    torch.set_num_threads(cores)
    out = {}
    torch.manual_seed(0)
    Bs = 64
    def ref_kv(q, kc, vc, k=None, v=None, cache_seqlens=None, cache_batch_idx=None, softmax_scale=None,
               causal=False):  # the restatement takes no causal flag (bottom-right is implied by the append)
        return kvcache_torch(q, kc, vc, k, v, cache_seqlens, cache_batch_idx, softmax_scale)

    blk = ResidualAttentionBlock(H * D, H, attn_kvcache=ref_kv).eval()
    sk, ck = FlashKVCache(Bs, 448, H, D, dtype=torch.float32), FlashKVCache(Bs, 1500, H, D, dtype=torch.float32)
    g = torch.Generator().manual_seed(3)
    ck.k_storage.normal_(generator=g)
    ck.v_storage.normal_(generator=g)
    sk.seq_lens.copy_(torch.from_numpy(_lengths(8, Bs, 1, 400).astype(np.int32)) - 1)
    x = torch.randn((Bs, 1, H * D), generator=g)
    slots = torch.arange(Bs)
    with torch.no_grad():
        med, n = _cpu_time(lambda: blk.forward_flash(x, sk, ck, slot_indices=slots), budget_s)
    out["decode_step"] = {"value": round(32 * med * 1e3, 1), "unit": "ms/step", "cores": cores, "kind": "port",
                          "sample": f"one decoder layer (self + cross attention through the torch restatement of "
                          f"_sdpa_attn_with_kvcache, MLP, LayerNorms) for 64 streams in fp32, median of {n} runs "
                          f"({med * 1e3:.1f} ms) x 32 layers; logits GEMM not included"}
    xa = torch.randn((1, FILL_L, H * D), generator=g)
    wk, wv, bv = torch.randn(H * D, H * D) / 36, torch.randn(H * D, H * D) / 36, torch.randn(H * D)
    fc = FlashKVCache(1, FILL_L, H, D, dtype=torch.float32)
    sl = torch.zeros(1, dtype=torch.long)

    def fill():
        k = F.linear(xa, wk).view(1, FILL_L, H, D)
        v = F.linear(xa, wv, bv).view(1, FILL_L, H, D)
        fc.k_cache[sl, :FILL_L] = k
        fc.v_cache[sl, :FILL_L] = v

    med, n = _cpu_time(fill, budget_s)
    out["cross_fill"] = {"value": round(med * FILL_B * 32 * 1e3, 1), "unit": "ms per 16 windows x 32 layers",
                         "cores": cores, "kind": "port",
                         "sample": f"one window's key/value projection + index_put into a head-major cache, fp32, "
                         f"median of {n} runs ({med * 1e3:.1f} ms) x 16 windows x 32 layers"}
    w = torch.randn((1, DTW_H, DTW_T, DTW_A), generator=g)
    med, n = _cpu_time(lambda: median_filter_torch(w, 7), budget_s)
    nbytes = 2 * w.numel() * 4
    out["median_filter"] = {"value": round(nbytes / med / 1e9, 3), "unit": "GB/s", "cores": cores, "kind": "port",
                            "sample": f"sort-based median_filter (dtw_align.py:65-78) width 7 on one chunk "
                            f"[1, 10, 448, 1500] fp32, median of {n} runs ({med * 1e3:.1f} ms)"}
    for k, v in out.items():
        log(f"[bench] {k} cpu baseline: {v['value']} {v['unit']}")
    return out


def cpu_baseline(budget_s: float = 12.0) -> dict:
    from oracle.attention_oracle import sdpa_torch

    cores = host_cores()
    torch.set_num_threads(cores)
    B, L = 1, 1500
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn((B, H, L, D), generator=g) for _ in range(3))
    flop = 4.0 * B * H * L * L * D
    sdpa_torch(q, k, v, scale=0.125)  # warm-up
    times = []
    t_end = time.perf_counter() + budget_s
    while len(times) < 5 or (time.perf_counter() < t_end and len(times) < 200):
        t0 = time.perf_counter()
        sdpa_torch(q, k, v, scale=0.125)
        times.append(time.perf_counter() - t0)
    med = float(np.median(times))
    tflops = flop / med / 1e12
    log(f"[bench] cpu baseline: torch SDPA fp32 {med * 1e3:.1f} ms per (B=1,H=20,L=1500) layer on {cores} threads -> {tflops:.3f} TFLOP/s")
    return {
        "value": round(tflops, 4),
        "unit": "TFLOP/s",
        "cores": cores,
        "kind": "port",
        "sample": f"torch CPU F.scaled_dot_product_attention fp32 (the reference's CPU path, model.py:288-296) on "
        f"one 30-s window layer B=1 H=20 L=1500 D=64, median of {len(times)} runs "
        f"({med * 1e3:.1f} ms each); config 2 is 16 such windows x 32 layers",
    }


# Algorithmic HBM bytes per launch of each kernel at the pmc_sample shapes (what the kernel must
# read and write at least), against which the measured traffic is compared.
_ALG_BYTES = {
    "dense_pipe_kernel<wdrz::Bf16, 3>": 4 * 16 * 1500 * 20 * 64 * 2,  # Q + K + V + O
    "kv_attn_kernel<wdrz::Bf16, 1, true, false>": 68526592,
    "kv_attn_kernel<wdrz::Bf16, 1, false, true>": 491847936,
    "kv_mq_kernel<wdrz::Bf16, true, 8, 4>": 75279872,
    "kv_mq_kernel<wdrz::Bf16, false, 8, 4>": 493158656,
    "dtw_rowcol_kernel<6>": 430080000,
    "dtw_seg_kernel": 430080000 + 43008000,
    "dtw_qk_kernel<wdrz::Bf16>": 430080000 + 2 * 16 * 10 * (448 + 1500) * 64,
    "kv_fill_kernel": 2 * 2 * 16 * 1500 * 1280 * 2,
    "median_filter_kernel<3>": 2 * 16 * 10 * 448 * 1500 * 4,
    "dtw_qk_rowcol_kernel<wdrz::Bf16>": 2 * 16 * 10 * (448 + 1500) * 64 + 16 * 10 * 448 * 8 + 16 * 10 * 3 * 1500 * 8,
    "dtw_qk_band_kernel<wdrz::Bf16, 3>": 2 * 16 * 10 * (448 + 1500) * 64 + 16 * 10 * (448 + 1500) * 8
    + 16 * 448 * 1500 * 4,
    "dense_f32_kernel<false>": 4 * 1500 * 20 * 64 * 4,
    "dense_split4_kernel<wdrz::Bf16>": 4 * 1500 * 20 * 64 * 2,
    "linear_act_kernel<wdrz::Bf16, 1, 2, 2, false>": 5120 * 1280 * 2 + 64 * 1280 * 2 + 5120 * 2 + 64 * 5120 * 2,
    "linear_act_kernel<wdrz::Bf16, 0, 2, 2, true>": 1280 * 5120 * 2 + 64 * 5120 * 2 + 4 * 64 * 1280 * 4,
    "kv_prefill_kernel<wdrz::Bf16, true>": 6 * 64 * 224 * 20 * 64 * 2,
}


def pmc_table(fetch_csv: str, write_csv: str) -> None:
    """Writes profiles/pmc_traffic.json (and prints its markdown table) from the counter CSVs of
    two `rocprofv3 --pmc FETCH_SIZE` / `--pmc WRITE_SIZE` runs of `bench.py --pmc-sample`. Both
    counters are scaled by what they read for the 1 GiB calibration copy (1 GiB read, 1 GiB
    written)."""
    import collections
    import csv
    import re

    def load(path, ctr):
        d = collections.defaultdict(list)
        with open(path) as f:
            for r in csv.DictReader(f):
                if r["Counter_Name"] == ctr:
                    d[r["Kernel_Name"]].append(float(r["Counter_Value"]))
        return d

    fe, wr = load(fetch_csv, "FETCH_SIZE"), load(write_csv, "WRITE_SIZE")
    cf, cw = max(fe["__amd_rocclr_copyBuffer"]), max(wr["__amd_rocclr_copyBuffer"])
    ff, wf = (1 << 20) / cf, (1 << 20) / cw
    out = {"calibration": {"copy_bytes_read": 1 << 30, "copy_bytes_written": 1 << 30, "fetch_size_KiB": cf,
                           "write_size_KiB": cw, "fetch_factor": round(ff, 4), "write_factor": round(wf, 4)},
           "kernels": {}}
    rows = []
    for name in fe:
        m = re.match(r"(?:void )?wdrz::\(anonymous namespace\)::(\w+(?:<[^()]*>)?)\(", name)
        if not m or name not in wr:
            continue
        k = m.group(1)
        f, w = sum(fe[name]) / len(fe[name]), sum(wr[name]) / len(wr[name])
        rb, wb = int(f * 1024 * ff), int(w * 1024 * wf)
        alg = _ALG_BYTES.get(k)
        out["kernels"][k] = {"fetch_KiB_raw": round(f, 1), "write_KiB_raw": round(w, 1), "hbm_read_bytes": rb,
                             "hbm_write_bytes": wb, "traffic_bytes": rb + wb, "algorithmic_bytes": alg,
                             "traffic_over_algorithmic": round((rb + wb) / alg, 4) if alg else None}
        ratio = f"{(rb + wb) / alg:.3f}" if alg else "n/a"
        alg_mb = f"{alg / 1e6:.1f}" if alg else "n/a"
        rows.append(f"| `{k}` | {f:.0f} | {w:.0f} | {(rb + wb) / 1e6:.1f} | {alg_mb} | {ratio} |")
    with open(_TRAFFIC_FILE, "w") as f:
        json.dump(out, f, indent=1)
    print(f"calibration fetch {cf:.0f} KiB write {cw:.0f} KiB -> factors {ff:.4f} {wf:.4f}")
    print("\n".join(sorted(rows)))


def pmc_sample(dev) -> None:
    """A short, fixed kernel sequence for hardware-counter passes (rocprofv3 --pmc):
    a calibration copy of 1 GiB (known HBM bytes), then 3 launches of the encoder kernel, of
    each decode kernel, of the DTW prep, compute_attention, the fused attention + prep, the
    cross-cache fill, the log-mel front end, the fp32 config 1 layer, one bf16 window and the
    decode step's fc1 + GELU and split-K fc2, and the 224-row prefill at the bench shapes (eager)."""
    from whisperdrz_amd import flash_attn_with_kvcache, scaled_dot_product_attention

    n = 1 << 30
    src = torch.empty(n // 2, dtype=torch.bfloat16, device=dev).normal_()
    dst = torch.empty_like(src)
    dst.copy_(src)  # calibration: reads 1 GiB, writes 1 GiB
    torch.cuda.synchronize()
    del src, dst
    B, L = 16, 1500
    for i in range(3):
        g = torch.Generator(device=dev).manual_seed(100 + i)
        qkv = torch.randn((3, B, L, H, D), generator=g, device=dev).to(torch.bfloat16)
        scaled_dot_product_attention(*(x.permute(0, 2, 1, 3) for x in qkv), scale=0.125)
        torch.cuda.synchronize()
    del qkv
    Bs = 64
    slots = torch.arange(Bs, dtype=torch.int32, device=dev)
    L3 = _lengths(3, Bs, 1, 448)
    L5 = _lengths(5, Bs, 5, 448)
    for i in range(3):
        kv_s = _head_major_cache(Bs, 448, dev, 3000 + i)
        kv_x = _head_major_cache(Bs, 1500, dev, 4000 + i)
        g = torch.Generator(device=dev).manual_seed(200 + i)
        q1, k1, v1, q5, k5, v5 = (torch.randn((Bs, s, H, D), generator=g, device=dev).to(torch.bfloat16)
                                  for s in (1, 1, 1, 5, 5, 5))
        cs3 = torch.from_numpy((L3 - 1).astype(np.int32)).to(dev)
        cs5 = torch.from_numpy((L5 - 5).astype(np.int32)).to(dev)
        flash_attn_with_kvcache(q1, kv_s[0], kv_s[1], k=k1, v=v1, cache_seqlens=cs3, cache_batch_idx=slots,
                                softmax_scale=0.125)
        flash_attn_with_kvcache(q1, kv_x[0], kv_x[1], cache_batch_idx=slots, softmax_scale=0.125)
        flash_attn_with_kvcache(q5, kv_s[0], kv_s[1], k=k5, v=v5, cache_seqlens=cs5, cache_batch_idx=slots,
                                softmax_scale=0.125)
        flash_attn_with_kvcache(q5, kv_x[0], kv_x[1], cache_batch_idx=slots, softmax_scale=0.125)
        torch.cuda.synchronize()
        del kv_s, kv_x
    from whisperdrz_amd import compute_attention, dtw_attention_prep, dtw_prep, log_mel_spectrogram

    for i in range(3):
        w, lens, caps = _dtw_inputs(dev, 5000 + i)
        dtw_prep(w, lens, caps, 7)
        torch.cuda.synchronize()
        del w
    mask = torch.zeros(32, H, dtype=torch.bool)
    for l, h in DTW_HEADS:
        mask[l, h] = True
    g = torch.Generator(device=dev).manual_seed(6000)
    q_out, k_out = [None] * 32, [None] * 32
    for l, _ in DTW_HEADS:
        q_out[l] = torch.randn((DTW_B, DTW_T, H * D), generator=g, device=dev).to(torch.bfloat16)
        k_out[l] = torch.randn((DTW_B, DTW_A, H * D), generator=g, device=dev).to(torch.bfloat16)
    for _ in range(3):
        compute_attention(q_out, k_out, mask)
        torch.cuda.synchronize()
    rng = np.random.default_rng(5000)
    lens = [int(x) for x in rng.integers(DTW_T // 2, DTW_T + 1, DTW_B)]
    for _ in range(3):
        dtw_attention_prep(q_out, k_out, mask, lens, [DTW_A] * DTW_B)
        torch.cuda.synchronize()
    from whisperdrz_amd import median_filter

    xm = torch.randn((DTW_B, DTW_H, DTW_T, DTW_A), generator=g, device=dev)
    for _ in range(3):
        median_filter(xm, 7)
        torch.cuda.synchronize()
    del xm
    del q_out, k_out
    from whisperdrz_amd.kv_cache import FlashKVCache

    fc = FlashKVCache(FILL_B, FILL_L, H, D, dtype=torch.bfloat16, device=dev)
    kv = torch.randn((FILL_B, FILL_L, 2, H, D), generator=g, device=dev).to(torch.bfloat16)
    for _ in range(3):
        fc.set_cross_attention(kv[:, :, 0], kv[:, :, 1], torch.arange(FILL_B, device=dev))
        torch.cuda.synchronize()
    del fc, kv
    audio = 0.1 * torch.randn((MEL_B, MEL_N), generator=g, device=dev)
    for _ in range(3):
        log_mel_spectrogram(audio, MEL_MELS, 3000)
        torch.cuda.synchronize()
    del audio
    # config 1 (fp32), one bf16 window (the key-split kernel), the decode step's
    # fused fc1 + GELU on three distinct (cold) weights
    from whisperdrz_amd import linear_gelu

    for dt in (torch.float32, torch.bfloat16):
        for i in range(3):
            qkv = torch.randn((3, 1, 1500, H, D), generator=g, device=dev).to(dt)
            scaled_dot_product_attention(*(x.permute(0, 2, 1, 3) for x in qkv), scale=0.125)
            torch.cuda.synchronize()
    x = torch.randn((64, 1280), generator=g, device=dev).to(torch.bfloat16)
    for i in range(3):
        lin = torch.nn.Linear(1280, 5120).to(dev, torch.bfloat16)
        linear_gelu(x, lin)
        torch.cuda.synchronize()
    # the decode step's fc2 as split-K partials (three distinct weights), and the 224-row prefill
    # into empty self caches (prefill kernel)
    from whisperdrz_amd import linear_partials

    x = torch.randn((64, 5120), generator=g, device=dev).to(torch.bfloat16)
    for i in range(3):
        lin = torch.nn.Linear(5120, 1280).to(dev, torch.bfloat16)
        linear_partials(x, lin, 4)
        torch.cuda.synchronize()
    del x
    zeros = torch.zeros(64, dtype=torch.int32, device=dev)
    for i in range(3):
        kv_s = _head_major_cache(64, 448, dev, 3100 + i)
        qkv = torch.randn((3, 64, 224, H, D), generator=g, device=dev).to(torch.bfloat16)
        flash_attn_with_kvcache(qkv[0], kv_s[0], kv_s[1], k=qkv[1], v=qkv[2], cache_seqlens=zeros,
                                cache_batch_idx=slots, softmax_scale=0.125, causal=True)
        torch.cuda.synchronize()
        del kv_s, qkv
    log("[bench] pmc sample done")


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--only", choices=["enc", "dec", "dtw", "mel", "step", "fill"], default=None)
    ap.add_argument("--pmc-sample", action="store_true",
                    help="run the short fixed kernel sequence used for rocprofv3 --pmc passes and exit")
    ap.add_argument("--pmc-table", nargs=2, metavar=("FETCH_CSV", "WRITE_CSV"),
                    help="summarise two --pmc-sample counter passes into profiles/pmc_traffic.json and exit")
    args = ap.parse_args()
    if args.pmc_table:
        pmc_table(*args.pmc_table)
        return 0
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print(
            "bench.py measures one GPU: the attention hot path shards by independent windows/slots "
            "with no collective, and this build runs on single-GPU boxes only (use --gpus 1).",
            file=sys.stderr,
        )
        return 2
    if not torch.cuda.is_available():
        print("bench.py needs a GPU (torch.cuda.is_available() is False)", file=sys.stderr)
        return 2
    from whisperdrz_amd import _lib

    _lib.load()  # fail loudly if the HIP library is missing
    dev = torch.device("cuda", 0)
    torch.cuda.set_device(dev)
    if args.pmc_sample:
        pmc_sample(dev)
        return 0

    enc = bench_encoder(dev, args.steps, args.warmup) if args.only in (None, "enc") else None
    c1 = bench_config1(dev, args.steps, args.warmup) if args.only in (None, "enc") else None
    dec = bench_decode(dev, args.steps, args.warmup) if args.only in (None, "dec") else None
    dtw = bench_dtw(dev, args.steps, args.warmup) if args.only in (None, "dtw") else None
    mel = bench_logmel(dev, args.steps, args.warmup) if args.only in (None, "mel") else None
    step = bench_decode_step(dev, args.steps, args.warmup) if args.only in (None, "step") else None
    fill = bench_cross_fill(dev, args.steps, args.warmup) if args.only in (None, "fill") else None
    cpu = None if args.no_cpu else cpu_baseline()
    if dtw is not None and not args.no_cpu:
        dtw["cpu_baseline"] = dtw_cpu_baseline()
    if mel is not None and not args.no_cpu:
        mel["cpu_baseline"] = logmel_cpu_baseline()
    if dec is not None and not args.no_cpu:
        for name, base in decode_cpu_baseline().items():
            dec[name]["cpu_baseline"] = base
    if not args.no_cpu and (step is not None or fill is not None or dtw is not None):
        extra = extra_cpu_baselines()
        if step is not None:
            step["cpu_baseline"] = extra["decode_step"]
        if fill is not None:
            fill["cpu_baseline"] = extra["cross_fill"]
        if dtw is not None:
            dtw["median_filter"]["cpu_baseline"] = extra["median_filter"]

    line = {
        "metric": METRIC,
        "value": round(enc["tflops"], 2) if enc else None,
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(enc["ms_per_step"], 4) if enc else None,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic, generated on the GPU: seeded N(0,1) Q/K/V and self K/V caches; cross K/V caches projected per layer from one seeded N(0,1) encoder output",
        "config": {
            "workload": "config2: encoder self-attention B=16 H=20 L=1500 D=64 bf16, non-causal, scale 1/8, "
            "32 sequential layers with distinct inputs; one step = 32 layers",
            "batch": 16,
            "heads": H,
            "seq_len": 1500,
            "head_dim": D,
            "layers_per_step": N_LAYERS,
            "parallelism": "single GPU",
        },
        "roofline": enc["roofline"] if enc else None,
        "encoder_single_window": enc["single_window"] if enc else None,
        "cpu_baseline": cpu,
        "config1_fp32": c1,
        "decode": dec,
        "dtw_prep": dtw,
        "log_mel": mel,
        "decode_step": step,
        "cross_fill": fill,
    }
    print(json.dumps(line), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
