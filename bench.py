#!/usr/bin/env python3
"""Benchmark of the paged-KV attention hot path on one MI355X.

Workload (N = 1): 27B-shape decode, batch 1, one full-attention layer: 24 q heads / 4 kv
heads, head_dim 256, context 32768, q8_0 KV in 256-token pages scattered by a random permutation page table, fused
sigmoid gate. A "step" is one p1a_attn_decode call (split-K kernel + merge) on inputs resident in HBM. The K timed
steps are captured once into a hipGraph (the engine replays its decode step as a graph as well) and walk over the KV of
8 full-attention layers of one sequence (the engine's pool layout: each layer its own K / V bytes, one page table per
sequence), so that consecutive steps do not find their 71 MB of KV in the 256 MB Infinity Cache.

Prints ONE JSON line: metric / value (GB/s of algorithmic KV bytes) plus `roofline` and `cpu_baseline` objects, and
secondary measurements (same-pool rate, verify, batched decode, prefill, append) under `extra`.
"""
import argparse
import ctypes
import importlib
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)
sys.path.insert(0, os.path.join(ROOT, "tests"))

HBM_PEAK_GBS = 8000.0
MFMA_F16_PEAK_TFLOPS = 2500.0


def build_layers(p1a, torch, kv_type, Hkv, D, psh, n_ctx, n_layers, seed):
    """ONE sequence of n_ctx tokens in a paged pool of n_layers full-attention layers, the engine's layout
    [page][layer][K | V][2^psh][rowb]: every layer has its own K / V bytes, all layers share the sequence's page table (a random
    permutation). Returns the per-layer descriptors; K/V are N(0,1), K RMS-normed per head, written through the library's
    own quantize-on-append."""
    ps = 1 << psh
    n_pages = (n_ctx + ps - 1) // ps
    g = torch.Generator(device="cuda").manual_seed(seed)
    tab = torch.randperm(n_pages, generator=g, device="cuda").to(torch.int32)
    rowb = p1a.kv_row_bytes(kv_type, Hkv, D)
    pool = torch.zeros(n_pages * n_layers * 2 * ps * rowb, dtype=torch.uint8, device="cuda")
    layers = [p1a.KVCache.paged(kv_type, Hkv, D, psh, n_pages, tab, n_pages, n_layers=n_layers, layer=l, pool=pool) for l in range(n_layers)]
    for c in layers:
        for a in range(0, n_ctx, 4096):
            T = min(4096, n_ctx - a)
            k = torch.randn((T, Hkv, D), generator=g, device="cuda")
            k = k * torch.rsqrt((k * k).mean(-1, keepdim=True) + 1e-6)
            v = torch.randn((T, Hkv, D), generator=g, device="cuda")
            p1a.kv_append(c, k, v, a, T)
    torch.cuda.synchronize()
    return layers, n_pages


def build_pool(p1a, torch, kv_type, Hq, Hkv, D, psh, n_ctx, n_seq, seed, lens=None):
    """n_seq sequences of n_ctx tokens (or lens[s]) in one paged pool, page tables a random permutation; K/V are
    N(0,1), K RMS-normed per head, written through the library's own quantize-on-append."""
    ps = 1 << psh
    ppseq = (n_ctx + ps - 1) // ps
    n_pages = ppseq * n_seq
    g = torch.Generator(device="cuda").manual_seed(seed)
    perm = torch.randperm(n_pages, generator=g, device="cuda").to(torch.int32)
    tabs = perm.reshape(ppseq, n_seq).t().contiguous().reshape(-1)       # pages interleaved across the slots
    kv = p1a.KVCache.paged(kv_type, Hkv, D, psh, n_pages, tabs, ppseq)
    chunk = 4096
    for s in range(n_seq):
        c = kv.slot(s, ppseq)
        n_s = n_ctx if lens is None else lens[s]
        for a in range(0, n_s, chunk):
            T = min(chunk, n_s - a)
            k = torch.randn((T, Hkv, D), generator=g, device="cuda")
            k = k * torch.rsqrt((k * k).mean(-1, keepdim=True) + 1e-6)
            v = torch.randn((T, Hkv, D), generator=g, device="cuda")
            p1a.kv_append(c, k, v, a, T)
    torch.cuda.synchronize()
    return kv, ppseq


REPLAYS = 7   # timed replays of a captured graph; the median is reported


def time_graph(torch, stream, fn_list, warmup, replays=REPLAYS, all_samples=False):
    """capture the calls of fn_list into one graph on `stream`, run `warmup` untimed calls (whole replays: at least one),
    then time `replays` replays, each bracketed by a synchronize and by events recorded on that same stream. Returns the
    MEDIAN seconds per call (and, on request, every sample)."""
    with torch.cuda.stream(stream):
        for f in fn_list[:2]:
            f()
        stream.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            for f in fn_list:
                f()
        for _ in range(max(1, -(-warmup // len(fn_list)))):
            g.replay()
        stream.synchronize()
        samples = []
        for _ in range(replays):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            e0.record(stream)
            g.replay()
            e1.record(stream)
            e1.synchronize()
            torch.cuda.synchronize()
            samples.append(e0.elapsed_time(e1) * 1e-3 / len(fn_list))
    samples.sort()
    med = samples[len(samples) // 2]
    return (med, samples) if all_samples else med


def time_eager(torch, fn, reps, warmup=2, group=1):
    """median over `reps` samples, each `group` back-to-back calls event-timed on the current stream; seconds per call"""
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    samples = []
    for _ in range(reps):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(group):
            fn()
        e1.record()
        e1.synchronize()
        samples.append(e0.elapsed_time(e1) * 1e-3 / group)
    samples.sort()
    return samples[len(samples) // 2]


def extras(p1a, torch, stream, Hq, Hkv, D, psh, scale, top, cpu):
    """secondary measurements: the other baseline configs at full size (reported, not the headline value)"""
    import math
    ex = {}
    g = torch.Generator(device="cuda").manual_seed(5)

    def normed(shape):
        x = torch.randn(shape, generator=g, device="cuda")
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6)

    # chunked prefill, T = 4096 after 28672 tokens, q8_0, append of the chunk then attention + gate
    p0, T = 28672, 4096
    kv, ppseq = build_pool(p1a, torch, p1a.KV_Q8_0, Hq, Hkv, D, psh, p0 + T, 1, seed=21)
    c = kv.slot(0, ppseq)
    q = normed((T, Hq, D)).half().float()
    gate = torch.randn((T, Hq * D), generator=g, device="cuda")
    out = torch.empty((T, Hq, D), device="cuda")
    kc = normed((T, Hkv, D))
    vc = torch.randn((T, Hkv, D), generator=g, device="cuda")
    # the caller-scratch variant (what attn_fold callers get): the cache is converted to f16 once per call
    scr = torch.empty(p1a.prefill_scratch_bytes(T, p0, Hq, Hkv, D), dtype=torch.uint8, device="cuda")
    # (eight untimed calls first: the first few calls after the pool has been built run 3 - 5 % slow, whichever variant they are)
    # (the part's clock settles over the first ten or so calls of a burst - every variant runs up to 10 % slow until then)
    sec = time_eager(torch, lambda: p1a.attn_prefill(q, c, out, T, p0, Hq, scale, gate=gate, scratch=scr), reps=9, warmup=12)
    flop = 4.0 * D * Hq * (p0 * T + T * (T + 1) / 2)
    ex["prefill_T4096_p28672_q8_0_ms"] = round(sec * 1e3, 4)
    ex["prefill_TFLOPs"] = round(flop / sec / 1e12, 1)
    ex["prefill_frac_of_f16_mfma_peak"] = round(flop / sec / 1e12 / MFMA_F16_PEAK_TFLOPS, 4)
    ex["prefill_scratch_MB"] = round(scr.numel() / 1e6, 1)
    top["roofline_prefill"] = {
        "bound": "mfma", "achieved": round(flop / sec / 1e12, 1), "peak": MFMA_F16_PEAK_TFLOPS, "unit": "TFLOP/s",
        "frac": round(flop / sec / 1e12 / MFMA_F16_PEAK_TFLOPS, 4), "traffic": prefill_traffic(), "kernel": "prefill_k<f16, 256, grouped, lds-direct>",
        "call_ms": round(sec * 1e3, 4),
        "note": "T = 4096 after 28672 tokens, q8_0, fused gate; flops = 4 D Hq (p0 T + T (T + 1) / 2); time = the "
                "whole p1a_attn_prefill call with caller scratch (the convert-once pass of about 40 us included), median of 9 "
                "after 12 untimed calls; traffic = HBM-side bytes per call read from the committed rocprofv3 counter summary "
                "(profiles/prefill_f16_staged_cfg5_traffic.json), not measured in this run"}
    # a reference point for the bound: what a plain dense f16 GEMM of the vendor library (8192^3, fp32 accumulate) reaches
    # on this part in the same run - the matrix pipe's practical ceiling under this part's power limit
    ga = torch.randn((8192, 8192), device="cuda", dtype=torch.float16)
    gb_ = torch.randn((8192, 8192), device="cuda", dtype=torch.float16)
    gsec = time_eager(torch, lambda: torch.matmul(ga, gb_), reps=9, warmup=12)
    ex["vendor_gemm_f16_8192_TFLOPs"] = round(2.0 * 8192 ** 3 / gsec / 1e12, 1)
    ex["vendor_gemm_f16_frac_of_mfma_peak"] = round(2.0 * 8192 ** 3 / gsec / 1e12 / MFMA_F16_PEAK_TFLOPS, 4)
    top["roofline_prefill"]["vendor_gemm_f16_frac"] = ex["vendor_gemm_f16_frac_of_mfma_peak"]
    del ga, gb_
    out_scr = out.clone()
    sec = time_eager(torch, lambda: p1a.attn_prefill(q, c, out, T, p0, Hq, scale, gate=gate), reps=5)
    ex["prefill_no_scratch_ms"] = round(sec * 1e3, 4)                      # (the library's own staging copy: the reference's attn_prefill call site)
    ex["prefill_no_scratch_frac_of_f16_mfma_peak"] = round(flop / sec / 1e12 / MFMA_F16_PEAK_TFLOPS, 4)
    ex["prefill_scratch_equals_no_scratch_bits"] = bool(torch.equal(out, out_scr))
    # neither the caller's scratch nor the library's staging copy: every workgroup dequantizes its own tiles
    p1a.set_prefill_staging_limit(0)
    sec = time_eager(torch, lambda: p1a.attn_prefill(q, c, out, T, p0, Hq, scale, gate=gate), reps=3)
    p1a.set_prefill_staging_limit(1 << 30)
    ex["prefill_in_kernel_dequant_ms"] = round(sec * 1e3, 4)
    ex["prefill_in_kernel_dequant_equals_bits"] = bool(torch.equal(out, out_scr))
    del scr, out_scr
    if cpu:
        top["cpu_prefill"] = cpu_prefill(torch, kv, ppseq, q, gate, out, p0, T, Hq, Hkv, D, psh, scale)
    # a short last chunk over the same context: its keys are split over several workgroups per (token block, head)
    Ts, p0s = 128, p0 + T - 128
    scr = torch.empty(p1a.prefill_scratch_bytes(Ts, p0s, Hq, Hkv, D), dtype=torch.uint8, device="cuda")
    sec = time_eager(torch, lambda: p1a.attn_prefill(q[:Ts], c, out[:Ts], Ts, p0s, Hq, scale, gate=gate[:Ts], scratch=scr), reps=5, group=10)
    ex["prefill_T128_p32640_q8_0_us"] = round(sec * 1e6, 1)
    ex["prefill_T128_key_splits"] = p1a.prefill_key_splits(Ts, p0s, Hq, Hkv)
    ex["prefill_T128_TFLOPs"] = round(4.0 * D * Hq * (p0s * Ts + Ts * (Ts + 1) / 2) / sec / 1e12, 1)
    del scr
    sec = time_eager(torch, lambda: p1a.kv_append(c, kc, vc, p0, T), reps=5, group=20)
    ab = 2 * T * Hkv * D * 4 + 2 * T * p1a.kv_row_bytes(p1a.KV_Q8_0, Hkv, D)
    ex["append_T4096_q8_0_us"] = round(sec * 1e6, 2)
    ex["append_GBs"] = round(ab / sec / 1e9, 1)
    # the input prep of a 4-row verify step (q | gate split, norm, rope, quantizing write) in front of the decode
    qg4 = torch.randn((4, Hq, 2 * D), generator=g, device="cuda")
    w_q = torch.ones(D, device="cuda")
    w_k = torch.ones(D, device="cuda")
    pos4 = torch.arange(p0, p0 + 4, dtype=torch.int32, device="cuda")
    q4 = torch.empty((4, Hq, D), device="cuda")
    g4 = torch.empty((4, Hq * D), device="cuda")
    with torch.cuda.stream(stream):
        sec = time_graph(torch, stream, [lambda: p1a.attn_prep(qg4, kc, vc, w_q, w_k, pos4, q4, g4, c, p0, 4, Hq, 64, 1e7, 1e-6)] * 20, 2)
    ex["prep_4rows_q8_0_us"] = round(sec * 1e6, 2)
    del kv, c, q, gate, out
    # q8_0 at head_dim 128 (head rows that are not whole 16-byte chunks): raw tiles fetched 4 bytes per lane and converted
    # to f16 tiles by their wave, then the f16 MFMA kernel; and head_dim 96, which the kernel
    # for any shape takes
    for Dx, tag in ((128, "staged_q8_0_D128_32K"), (96, "generic_q8_0_D96_32K")):
        kvg, ppg = build_pool(p1a, torch, p1a.KV_Q8_0, Hq, Hkv, Dx, psh, 32768, 1, seed=25)
        qg_ = normed((1, Hq, Dx))
        og_ = torch.empty((1, Hq, Dx), device="cuda")
        cg_ = kvg.slot(0, ppg)
        with torch.cuda.stream(stream):
            p1a.warmup(8, Hq, Hkv, Dx)
            sec = time_graph(torch, stream, [lambda: p1a.attn_decode(qg_, cg_, og_, 1, 32767, Hq, 1.0 / Dx ** 0.5)] * 20, 2)
        gbytes = 2 * 32768 * p1a.kv_row_bytes(p1a.KV_Q8_0, Hkv, Dx)
        ex[tag + "_us"] = round(sec * 1e6, 2)
        ex[tag + "_GBs"] = round(gbytes / sec / 1e9, 1)
        del kvg, cg_
    ex.update(verify_config(p1a, torch, stream, Hq, Hkv, D, psh, scale))
    ex.update(mtp_verify_loop(p1a, torch, Hq, Hkv, D, psh, scale))
    ex.update(mtp_verify_loop(p1a, torch, Hq, Hkv, D, psh, scale, graphed=True))
    ex.update(batched_config(p1a, torch, stream, Hq, Hkv, D, psh, scale))
    # the same kernel with enough to stream: 4 sequences of 65536 tokens, one row each, q8_0 (570 MB of KV per call)
    n4 = 65536
    kv, ppseq = build_pool(p1a, torch, p1a.KV_Q8_0, Hq, Hkv, D, psh, n4, 4, seed=24)
    pos = torch.full((4,), n4 - 1, dtype=torch.int32, device="cuda")
    rt = torch.tensor([s * ppseq for s in range(4)], dtype=torch.int32, device="cuda")
    q = normed((4, Hq, D))
    gate = torch.randn((4, Hq * D), generator=g, device="cuda")
    out = torch.empty((4, Hq, D), device="cuda")
    cr = kv.with_rows(rt)
    with torch.cuda.stream(stream):
        sec = time_graph(torch, stream, [lambda: p1a.attn_decode_rows(q, cr, out, 4, pos, Hq, scale, gate=gate)] * 10, 2)
    lb = 4 * n4 * 2 * p1a.kv_row_bytes(p1a.KV_Q8_0, Hkv, D)
    ex["decode_4x64K_q8_0_us"] = round(sec * 1e6, 2)
    ex["decode_4x64K_GBs"] = round(lb / sec / 1e9, 1)
    return ex


def prefill_traffic():
    tpath = os.path.join(ROOT, "profiles", "prefill_f16_staged_cfg5_traffic.json")
    if os.path.exists(tpath):
        with open(tpath) as f:
            return json.load(f).get("hbm_bytes_per_call")
    return None


def verify_config(p1a, torch, stream, Hq, Hkv, D, psh, scale, reps=20):
    """MTP verify, 4 sequences x 4 rows (causal inside the block), q4_0, ctx 65536, each sequence's KV read once"""
    n4 = 65536
    g = torch.Generator(device="cuda").manual_seed(6)
    kv, ppseq = build_pool(p1a, torch, p1a.KV_Q4_0, Hq, Hkv, D, psh, n4, 4, seed=22)
    pos = torch.tensor([n4 - 4 + t for _ in range(4) for t in range(4)], dtype=torch.int32, device="cuda")
    rt = torch.tensor([s * ppseq for s in range(4) for _ in range(4)], dtype=torch.int32, device="cuda")
    q = torch.randn((16, Hq, D), generator=g, device="cuda")
    q = (q * torch.rsqrt((q * q).mean(-1, keepdim=True) + 1e-6)).half().float()
    out = torch.empty((16, Hq, D), device="cuda")
    cr = kv.with_rows(rt)
    with torch.cuda.stream(stream):
        p1a.warmup(32, Hq, Hkv, D)
        # (one untimed pass first: the figures of the first graph after the pool has been built run 10 - 15 % high, whichever it is)
        time_graph(torch, stream, [lambda: p1a.attn_decode_rows(q, cr, out, 16, pos, Hq, scale, rows_per_seq=4)] * reps, 2, replays=3)
        sec = time_graph(torch, stream, [lambda: p1a.attn_decode_rows(q, cr, out, 16, pos, Hq, scale, rows_per_seq=4)] * reps, 2)
        sec_k = time_graph(torch, stream, [lambda: p1a.bench_decode_split_only(q, cr, out, 16, 0, Hq, scale, pos=pos, rows_per_seq=4)] * reps, 2)
    vb = 4 * n4 * 2 * p1a.kv_row_bytes(p1a.KV_Q4_0, Hkv, D)
    return {"verify_4x4_q4_0_64K_us": round(sec * 1e6, 2), "verify_GBs": round(vb / sec / 1e9, 1),
            "verify_kernel_us": round(sec_k * 1e6, 2), "verify_kernel_frac_of_hbm_peak": round(vb / sec_k / 1e9 / HBM_PEAK_GBS, 4),
            "roofline_verify": {"bound": "hbm", "workload": "4 sequences x 4 rows, q4_0, ctx 65536", "bytes": vb,
                                "kernel": "dec_mfma_k<q4_0, 256, 2, 8>", "kernel_us": round(sec_k * 1e6, 2),
                                "achieved": round(vb / sec_k / 1e9, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                                "frac": round(vb / sec_k / 1e9 / HBM_PEAK_GBS, 4), "call_us": round(sec * 1e6, 2),
                                "call_frac": round(vb / sec / 1e9 / HBM_PEAK_GBS, 4)}}


def batched_config(p1a, torch, stream, Hq, Hkv, D, psh, scale, reps=20):
    """8 slots, one row each, ctx log-uniform in [1024, 32768], q8_0, one shared pool"""
    import math
    g = torch.Generator(device="cuda").manual_seed(9)
    rs = torch.Generator().manual_seed(8)
    lens = [int(math.exp(float(torch.empty(1).uniform_(math.log(1024), math.log(32768), generator=rs)))) for _ in range(8)]
    kv, ppseq = build_pool(p1a, torch, p1a.KV_Q8_0, Hq, Hkv, D, psh, 32768, 8, seed=23, lens=lens)
    pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device="cuda")
    rt = torch.tensor([s * ppseq for s in range(8)], dtype=torch.int32, device="cuda")
    q = torch.randn((8, Hq, D), generator=g, device="cuda")
    q = q * torch.rsqrt((q * q).mean(-1, keepdim=True) + 1e-6)
    gate = torch.randn((8, Hq * D), generator=g, device="cuda")
    out = torch.empty((8, Hq, D), device="cuda")
    cr = kv.with_rows(rt)
    with torch.cuda.stream(stream):
        p1a.warmup(32, Hq, Hkv, D)
        sec = time_graph(torch, stream, [lambda: p1a.attn_decode_rows(q, cr, out, 8, pos, Hq, scale, gate=gate)] * reps, 2)
        sec_k = time_graph(torch, stream, [lambda: p1a.bench_decode_split_only(q, cr, out, 8, 0, Hq, scale, pos=pos)] * reps, 2)
    bb = sum(lens) * 2 * p1a.kv_row_bytes(p1a.KV_Q8_0, Hkv, D)
    res = {"batched_8slots_q8_0_us": round(sec * 1e6, 2), "batched_GBs": round(bb / sec / 1e9, 1), "batched_ctx": lens,
           "roofline_batched": {"bound": "hbm", "workload": "8 slots, 1 row each, q8_0, ctx log-uniform in [1024, 32768]",
                                "bytes": bb, "kernel": "dec_mfma_k<q8_0, 256, 1, 8, two workgroups per CU>",
                                "kernel_us": round(sec_k * 1e6, 2), "achieved": round(bb / sec_k / 1e9, 1), "peak": HBM_PEAK_GBS,
                                "unit": "GB/s", "frac": round(bb / sec_k / 1e9 / HBM_PEAK_GBS, 4), "call_us": round(sec * 1e6, 2),
                                "call_frac": round(bb / sec / 1e9 / HBM_PEAK_GBS, 4)}}
    del kv, cr
    # the widest call the library takes: 32 slots, short contexts (2 K ... 5 K) - per-workgroup set-up is most of it
    lens32 = [2048 + 100 * i for i in range(32)]
    kv, ppseq = build_pool(p1a, torch, p1a.KV_Q8_0, Hq, Hkv, D, psh, max(lens32), 32, seed=24, lens=lens32)
    pos = torch.tensor([n - 1 for n in lens32], dtype=torch.int32, device="cuda")
    rt = torch.tensor([s * ppseq for s in range(32)], dtype=torch.int32, device="cuda")
    q32 = torch.randn((32, Hq, D), generator=g, device="cuda")
    out32 = torch.empty((32, Hq, D), device="cuda")
    cr = kv.with_rows(rt)
    with torch.cuda.stream(stream):
        sec = time_graph(torch, stream, [lambda: p1a.attn_decode_rows(q32, cr, out32, 32, pos, Hq, scale)] * reps, 2)
    bb = sum(lens32) * 2 * p1a.kv_row_bytes(p1a.KV_Q8_0, Hkv, D)
    res.update({"batched_32slots_2K_5K_q8_0_us": round(sec * 1e6, 2), "batched_32slots_GBs": round(bb / sec / 1e9, 1)})
    return res


def mtp_verify_loop(p1a, torch, Hq, Hkv, D, psh, scale, n_seq=4, ctx=65000, steps=30, graphed=False):
    """The verify attention inside a step loop, as the engine's scheduler drives it (accept / rollback per sequence,
    src/sched.cpp:1053-1087 of the reference): 4 sequences of a q4_0 pool at ~64K tokens, every step 1 + 3 draft rows per
    sequence go through attn_prep (norm, rope, quantizing KV write at each row's own position) and one batched
    attn_decode_rows, the host accepts a prefix (each draft right with probability 0.7, seeded) and rolls the rest back.
    Wall time per step, host bookkeeping and the position upload included. graphed: the two launches of a step (input prep,
    batched attention) are captured once into a graph after the warm-up and replayed every step, positions and page tables
    being read on the device - the way the engine runs its decode step (src/tp_model.cu:1379-1397)."""
    import random
    import time
    gs = torch.cuda.Stream()
    with torch.cuda.stream(gs):
        res = _mtp_verify_loop(p1a, torch, gs, Hq, Hkv, D, psh, scale, n_seq, ctx, steps, graphed, random, time)
    return res


def _mtp_verify_loop(p1a, torch, gs, Hq, Hkv, D, psh, scale, n_seq, ctx, steps, graphed, random, time):
    pool = p1a.Pool(p1a.KV_Q4_0, 1, Hkv, D, psh, n_ctx=ctx + 4096, max_slots=n_seq, tokens=n_seq * (ctx + 4096), stream=gs.cuda_stream)
    g = torch.Generator(device="cuda").manual_seed(31)
    ids = [pool.seq_create() for _ in range(n_seq)]
    for i, s in enumerate(ids):
        n = ctx - 37 * i                                    # unequal depths
        for a in range(0, n, 8192):
            T = min(8192, n - a)
            k = torch.randn((T, Hkv, D), generator=g, device="cuda")
            k = k * torch.rsqrt((k * k).mean(-1, keepdim=True) + 1e-6)
            v = torch.randn((T, Hkv, D), generator=g, device="cuda")
            pool.seq_advance(s, T=T)
            p1a.kv_append(pool.cache_seq(0, s), k, v, a, T)
    torch.cuda.synchronize()
    R = 4
    rows = n_seq * R
    qg = torch.randn((rows, Hq, 2 * D), generator=g, device="cuda")
    kx = torch.randn((rows, Hkv, D), generator=g, device="cuda")
    vx = torch.randn((rows, Hkv, D), generator=g, device="cuda")
    w = torch.ones(D, device="cuda")
    q = torch.empty((rows, Hq, D), device="cuda")
    gate = torch.empty((rows, Hq * D), device="cuda")
    out = torch.empty((rows, Hq, D), device="cuda")
    pos_h = torch.empty(rows, dtype=torch.int32).pin_memory()
    pos = torch.empty(rows, dtype=torch.int32, device="cuda")
    pool.set_rows([s for s in ids for _ in range(R)])
    cr = pool.cache_rows(0)
    rnd = random.Random(7)
    emitted, t_total = 0, 0.0

    def launches():
        p1a.attn_prep(qg, kx, vx, w, w, pos, q, gate, cr, -1, rows, Hq, 64, 1e7, 1e-6)
        p1a.attn_decode_rows(q, cr, out, rows, pos, Hq, scale, gate=gate, rows_per_seq=R)

    graph = None
    if graphed:
        p1a.warmup(rows, Hq, Hkv, D)
        pos.copy_(torch.tensor([pool.seq_len(s) - 1 for s in ids for _ in range(R)], dtype=torch.int32))   # (valid rows for the capture)
        gs.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=gs):
            launches()
    for step in range(steps + 3):
        t0 = time.perf_counter()
        for i, s in enumerate(ids):
            n = pool.seq_len(s)
            for t in range(R):
                pos_h[i * R + t] = n + t
            pool.seq_advance(s, T=R)
        pos.copy_(pos_h, non_blocking=True)
        if graph is not None:
            graph.replay()
        else:
            launches()
        gs.synchronize()                                    # the engine reads the rows' logits here
        n_out = 0
        for s in ids:
            tokens = [1, 2, 3, 4]
            greedy = [2, 3, 4, 5]
            for d in range(R - 1):
                if rnd.random() > 0.7:
                    greedy[d] = 0                           # draft d + 1 was wrong
                    break
            keep, _, _ = p1a.verify_accept(tokens, greedy, 1 << 20)
            pool.rollback(s, R, keep)
            n_out += keep
        dt = time.perf_counter() - t0
        if step >= 3:
            t_total += dt
            emitted += n_out
    pool.close()
    tag = "mtp_verify_step_graphed_us" if graphed else "mtp_verify_step_us"
    return {tag: round(t_total / steps * 1e6, 1), "mtp_tokens_per_step": round(emitted / steps, 2),
            "mtp_loop": f"{n_seq} sequences x (1 + 3 drafts), q4_0, ~{ctx} tokens each, prep + decode + accept/rollback, wall clock"}


def host_cpu():
    model = "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    return model, os.cpu_count()


def host_view(torch, kv, ppseq, slot, Hkv, D, psh, kv_type):
    """the oracle's view of one sequence of a device pool: the pool's bytes and its page table copied to the host"""
    import numpy as np
    import _oracle as O
    pool = kv.pool.cpu().numpy()
    tabs = kv.pt.cpu().numpy() if hasattr(kv.pt, "cpu") else kv._keep[1].cpu().numpy()
    n_pages = pool.size // kv.pstride
    h = O.HostKV.paged(kv_type, Hkv, D, psh, n_pages, tabs, ppseq, pool=pool)
    return h.view(pt=np.ascontiguousarray(tabs[slot * ppseq:(slot + 1) * ppseq]))


def cpu_baseline(torch, kv, layer, n_layers, q, gate, out_gpu, Hq, Hkv, D, psh, n_ctx, scale):
    """The CPU oracle (fp32 restatement of the reference's attention kernel, OpenMP over heads) on a bounded sample of
    the same workload: the decode step the GPU timed last - same pool bytes, same page table, same q and gate - repeated
    for about 10 s; its result is the check of the GPU's timed output."""
    import numpy as np
    import _inputs as I
    import _oracle as O
    pool = kv.pool.cpu().numpy()
    tab = kv.pt.cpu().numpy()
    hv = O.HostKV.paged(O.KV_Q8_0, Hkv, D, psh, len(tab), tab, len(tab), n_layers=n_layers, layer=layer, pool=pool)
    hq, hg = q.cpu().numpy(), gate.cpu().numpy()
    pos = np.array([n_ctx - 1], np.int32)
    ref = O.attn_rows(hv, hq, pos, Hq, scale, gate=hg)
    reps, t0 = 0, time.perf_counter()
    while True:
        O.attn_rows(hv, hq, pos, Hq, scale, gate=hg)
        reps += 1
        dt = time.perf_counter() - t0
        if dt > 10.0:
            break
    ma, rl = I.errors(out_gpu.cpu().numpy(), ref)
    model, ncpu = host_cpu()
    bytes_ = 2 * n_ctx * O.row_bytes(O.KV_Q8_0, Hkv, D)
    return {"value": round(bytes_ * reps / dt / 1e9, 2), "unit": "GB/s", "cores": int(O.lib().orc_num_threads()), "kind": "port",
            "sample": f"{reps} full decode steps (1 row, ctx {n_ctx}, q8_0, the layer and page table of the GPU's last timed step) of "
                      f"the C oracle with OpenMP, {dt:.1f} s",
            "cpu_model": model, "nproc": ncpu,
            "gpu_output_check": {"max_abs": float(f"{ma:.3e}"), "rel_l2": float(f"{rl:.3e}"), "tol": [I.MAX_ABS_TOL, I.REL_L2_TOL],
                                 "ok": bool(ma <= I.MAX_ABS_TOL and rl <= I.REL_L2_TOL)}}


def cpu_prefill(torch, kv, ppseq, q, gate, out_gpu, p0, T, Hq, Hkv, D, psh, scale, every=32):
    """the prefill half of the metric on the host: the oracle on every 32nd row of the chunk (128 of 4096 rows, each over
    its 28673..32768 visible keys), timed once; the same rows check the GPU's output"""
    import numpy as np
    import _inputs as I
    import _oracle as O
    hv = host_view(torch, kv, ppseq, 0, Hkv, D, psh, O.KV_Q8_0)
    rows = np.arange(every - 1, T, every)
    hq, hg = q.cpu().numpy()[rows], gate.cpu().numpy()[rows]
    pos = (p0 + rows).astype(np.int32)
    t0 = time.perf_counter()
    ref = O.attn_rows(hv, hq, pos, Hq, scale, gate=hg)
    dt = time.perf_counter() - t0
    flop = float(sum(4.0 * D * Hq * (int(p) + 1) for p in pos))
    ma, rl = I.errors(out_gpu.cpu().numpy()[rows], ref)
    model, ncpu = host_cpu()
    return {"value": round(flop / dt / 1e12, 4), "unit": "TFLOP/s", "cores": int(O.lib().orc_num_threads()), "kind": "port",
            "sample": f"{len(rows)} of {T} rows (every {every}th) of the prefill chunk on the C oracle with OpenMP, {dt:.1f} s; the full "
                      f"chunk would take about {dt * T / len(rows):.0f} s",
            "cpu_model": model, "nproc": ncpu,
            "gpu_output_check": {"max_abs": float(f"{ma:.3e}"), "rel_l2": float(f"{rl:.3e}"), "tol": [I.MAX_ABS_TOL, I.REL_L2_TOL],
                                 "ok": bool(ma <= I.MAX_ABS_TOL and rl <= I.REL_L2_TOL)}}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--no-extra", action="store_true", help="only the headline workload")
    ap.add_argument("--rotating-only", action="store_true",
                    help="skip the same-pool (Infinity Cache resident) graphs, so that every launch a profiler sees is the "
                         "rotating-pool headline launch")
    ap.add_argument("--calib-copy", action="store_true",
                    help="also run a plain 256 MiB elementwise copy kernel (reference point for rocprofv3 FETCH_SIZE / WRITE_SIZE)")
    ap.add_argument("--prefill-only", action="store_true",
                    help="run only the chunked-prefill configuration (T = 4096 after 28672 tokens, q8_0) a few times and print its "
                         "time: a short program for rocprofv3 counter passes over prefill_k")
    ap.add_argument("--verify-only", action="store_true",
                    help="run only the MTP-verify configuration (4 sequences x 4 rows, q4_0, ctx 65536) a few times and print its "
                         "time: a short program for rocprofv3 counter passes over dec_mfma_k<q4_0, 256, 2, 8>")
    ap.add_argument("--batched-only", action="store_true",
                    help="run only the batched-decode configuration (8 slots of unequal depth, q8_0) a few times and print its time")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py: this path is measured on ONE GPU only (no collectives are part of it); run with --gpus 1", file=sys.stderr)
        sys.exit(2)
    import torch
    if not torch.cuda.is_available():
        print("bench.py: no GPU visible", file=sys.stderr)
        sys.exit(2)
    p1a = importlib.import_module("p100e-engine_amd")
    p1a.lib()
    Hq, Hkv, D, psh, n_ctx = 24, 4, 256, 8, 32768
    scale = 1.0 / 16.0
    if args.prefill_only:
        p0, T = 28672, 4096
        kvp, ppseq = build_pool(p1a, torch, p1a.KV_Q8_0, Hq, Hkv, D, psh, p0 + T, 1, seed=21)
        c = kvp.slot(0, ppseq)
        qp = torch.randn((T, Hq, D), device="cuda").half().float()
        gp = torch.randn((T, Hq * D), device="cuda")
        op = torch.empty((T, Hq, D), device="cuda")
        scr = torch.empty(p1a.prefill_scratch_bytes(T, p0, Hq, Hkv, D), dtype=torch.uint8, device="cuda")
        sec = time_eager(torch, lambda: p1a.attn_prefill(qp, c, op, T, p0, Hq, scale, gate=gp, scratch=scr), reps=3, warmup=1)
        flop = 4.0 * D * Hq * (p0 * T + T * (T + 1) / 2)
        print(json.dumps({"prefill_T4096_p28672_q8_0_ms": round(sec * 1e3, 4), "TFLOPs": round(flop / sec / 1e12, 1)}))
        return
    if args.verify_only:
        print(json.dumps(verify_config(p1a, torch, torch.cuda.Stream(), Hq, Hkv, D, psh, scale, reps=10)))
        return
    if args.batched_only:
        print(json.dumps(batched_config(p1a, torch, torch.cuda.Stream(), Hq, Hkv, D, psh, scale, reps=10)))
        return
    rowb = p1a.kv_row_bytes(p1a.KV_Q8_0, Hkv, D)
    step_bytes = 2 * n_ctx * rowb                                          # K + V of the visible positions
    n_pools = 8                                                            # 8 layers x 71 MB > 256 MB Infinity Cache
    slots, ppseq = build_layers(p1a, torch, p1a.KV_Q8_0, Hkv, D, psh, n_ctx, n_pools, seed=1234)
    g = torch.Generator(device="cuda").manual_seed(99)
    q = torch.randn((1, Hq, D), generator=g, device="cuda")
    q = q * torch.rsqrt((q * q).mean(-1, keepdim=True) + 1e-6)
    gate = torch.randn((1, Hq * D), generator=g, device="cuda")
    out = torch.empty((1, Hq, D), device="cuda")
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        p1a.warmup(32, Hq, Hkv, D)

    def step(i):
        return lambda: p1a.attn_decode(q, slots[i % n_pools], out, 1, n_ctx - 1, Hq, scale, gate=gate)

    def kstep(i):   # the split-K kernel alone (a benchmarks-only entry point of the library: no merge, out untouched)
        return lambda: p1a.bench_decode_split_only(q, slots[i % n_pools], out, 1, n_ctx - 1, Hq, scale)

    K, W = args.steps, args.warmup
    torch.cuda.synchronize()
    # the dominant kernel alone first, so that the LAST thing to write `out` is the timed headline graph
    sec_kernel = time_graph(torch, stream, [kstep(i) for i in range(K)], W)
    sec_kernel_same = None if args.rotating_only else time_graph(torch, stream, [kstep(0) for _ in range(K)], W)
    sec_same = None if args.rotating_only else time_graph(torch, stream, [step(0) for _ in range(K)], W)
    out.fill_(float("nan"))
    sec, samples = time_graph(torch, stream, [step(i) for i in range(K)], W, all_samples=True)
    out_timed = out.clone()                                                # the result of step K - 1 of the last timed replay
    gbs = step_bytes / sec / 1e9
    kgbs = step_bytes / sec_kernel / 1e9
    traffic = None
    tpath = os.path.join(ROOT, "profiles", "decode_q8_0_32k_traffic.json")
    if os.path.exists(tpath):
        with open(tpath) as f:
            traffic = json.load(f).get("hbm_bytes_per_launch")
    res = {
        "metric": "decode-attn HBM GB/s @27B q8_0 32K (paged, B=1, fused gate)", "value": round(gbs, 1), "unit": "GB/s",
        "n_gpus": 1, "steps": K, "warmup": W, "ms_per_step": round(sec * 1e3, 5), "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "q8_0 KV -> f16 MFMA, f32 accumulate", "data": "synthetic",
        "config": {"workload": "decode 24/4 heads, head_dim 256, ctx 32768, q8_0, 256-token pages, random page table",
                   "kv_bytes_per_step": step_bytes, "layers_rotated": n_pools,
                   "launch": f"hipGraph of K steps, replayed {REPLAYS} times, median replay"},
        "replay_ms_per_step": [round(x * 1e3, 5) for x in samples],
        "roofline": {"bound": "hbm", "achieved": round(kgbs, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": round(kgbs / HBM_PEAK_GBS, 4), "traffic": traffic, "kernel": "dec_mfma_k<q8_0, 256, 1, 8>",
                     "kernel_us": round(sec_kernel * 1e6, 2),
                     "call_us": round(sec * 1e6, 2), "call_frac": round(gbs / HBM_PEAK_GBS, 4),
                     "note": "achieved = algorithmic KV bytes of one launch (2 * ctx * 1088 B) / average duration of the "
                             "split-K kernel, event-timed on its stream over a graph of K launches walking the 8 layers (median of "
                             f"{REPLAYS} replays); traffic = HBM bytes per launch read from the committed rocprofv3 counter summary "
                             "(profiles/decode_q8_0_32k_traffic.json), not measured in this run"},
        "extra": {"same_pool_GBs": sec_same and round(step_bytes / sec_same / 1e9, 1), "same_pool_us": sec_same and round(sec_same * 1e6, 2),
                  "kernel_same_pool_us": sec_kernel_same and round(sec_kernel_same * 1e6, 2),
                  "kernel_same_pool_GBs": sec_kernel_same and round(step_bytes / sec_kernel_same / 1e9, 1),
                  "merge_kernel_us": round((sec - sec_kernel) * 1e6, 2), "nsplit": p1a.get_nsplit(Hkv)},
    }
    # a reference point for the size: a plain streaming read (nothing computed) of the same number of bytes, rotating over
    # buffers larger than the Infinity Cache - what the memory system gives a 71 MB launch
    ref_bufs = [torch.ones(step_bytes // 4, device="cuda") for _ in range(n_pools)]
    sec_ref = time_graph(torch, stream, [(lambda i=i: p1a.bench_stream_read(ref_bufs[i % n_pools])) for i in range(min(K, 64))], W)
    res["extra"]["stream_read_same_bytes_us"] = round(sec_ref * 1e6, 2)
    res["extra"]["stream_read_same_bytes_GBs"] = round(step_bytes / sec_ref / 1e9, 1)
    del ref_bufs
    if args.calib_copy:
        src = torch.ones(64 * 1024 * 1024, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(3):
            torch.mul(src, 1.0, out=dst)                                   # reads 256 MiB, writes 256 MiB
        torch.cuda.synchronize()
        del src, dst
    if not args.no_cpu:
        res["cpu_baseline"] = cpu_baseline(torch, slots[(K - 1) % n_pools], (K - 1) % n_pools, n_pools, q, gate, out_timed, Hq, Hkv, D, psh, n_ctx, scale)
    del slots
    if not args.no_extra:
        top = {}
        res["extra"].update(extras(p1a, torch, stream, Hq, Hkv, D, psh, scale, top, not args.no_cpu))
        if "roofline_prefill" in top:
            res["roofline_prefill"] = top["roofline_prefill"]
        for key in ("roofline_verify", "roofline_batched"):
            if key in res["extra"]:
                res[key] = res["extra"].pop(key)
        if "cpu_prefill" in top:
            res["cpu_baseline"]["prefill"] = top["cpu_prefill"]
    print(json.dumps(res))


if __name__ == "__main__":
    main()
