"""Benchmark of the routed sparse Pattention MLP at the Llama-3-8B shape on one MI355X.

Metric: Pattention MLP tok/s at the 8B shape (b=64 decode,
4K-token prefill) and % of roofline.

A step is one eval forward of one FovealPattentionMLP layer (d_model 4096,
14336 parameter tokens = 224 blocks of 64, 8 base + 56 remote active blocks)
over one batch of synthetic input already resident in HBM:
  decode  : x (64, 1, 4096) bf16, cached active blocks (foveal_pattention.py:278-288)   -> `value`
  prefill : x (1, 4096, 4096) bf16, same active blocks                                  -> "prefill"
Steps cycle over L distinct layers (their own weights and routed block sets) so
the active weights are not served from the 256 MB MALL of one repeated layer.
The K timed steps are captured once in a HIP graph and replayed; HIP events on
the replay stream bracket the timed region.

The default line also carries, under "workloads", one sub-object per other
config (each with its own roofline and CPU baseline, 20 graph-replayed steps):
C2 routing, C4 decode attention, C5 block-sparse GEMM, prefill attention and the
fused indexer attention (skip them with --no-workloads).  Each can also run alone as its own line:
  --workload routing      C2: fused 16-D cosine scoring + top-p selection, 8192 queries x 4096 keys
  --workload decode_attn  C4: foveal paged-KV decode attention, 32 sequences x 131072 context
  --workload prefill_attn block-sparse prefill attention, 16384 tokens, Llama-3-8B attention heads
  --workload block_sparse C5: 2-D tile-sparse matmul, 4096 x 8192 by 8192 x 8192, 128 x 128 tiles
  --workload teacher_targets dense block-energy distillation targets, Llama-3-8B MLP, 4096 tokens
  --workload hbm_stream   the HBM read ceiling (torch sum and copy over 4 GiB)
  --workload sram_attn    fused 16-D indexer + greedy selection + block attention, the reference's 3 SRAM configs

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--layers L] [--no-prefill] [--workload W]
"""
from __future__ import annotations

import argparse
import json
import math
import os
import sys
import time
from pathlib import Path

import torch

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

HBM_PEAK_GBS = 8000.0          # MI355X HBM3E, GB/s
BF16_PEAK_TFLOPS = 2516.6      # MI355X dense bf16 MFMA, TFLOP/s
FP32_PEAK_TFLOPS = 157.3       # MI355X fp32 (vector and dense matrix), TFLOP/s

D_MODEL, N_PARAM, BLOCK, BASE, REMOTE = 4096, 14336, 64, 8, 56
DECODE_BATCH, PREFILL_TOKENS = 64, 4096


# HBM bytes of one decode step measured with rocprofv3 FETCH_SIZE and WRITE_SIZE
# passes, scaled by a 512 MiB copy (profiles/pattention_decode_prefill_8b.md):
#   packed path  : (34908.2 + 18503.2) KiB x 1.99983 read + (512 + 512) KiB written
#   --no-pack    : (34872.4 + 4129.5 + 18477.7 + 4109.0) KiB x 1.9997 read + 17408 KiB written
DECODE_TRAFFIC_BYTES = int(107837.0 * 1024)
DECODE_TRAFFIC_BYTES_UNPACKED = int(140566.8 * 1024)
# Same method for the other workloads (KiB read after the x 1.99983 scale + KiB written;
# profiles/pattention_decode_prefill_8b.md, decode_attention_c4.md, indexer_routing_c2.md,
# block_sparse_gemm_c5.md).
PREFILL_TRAFFIC_BYTES = int((393537 + 33270 + 196732 + 34374) * 1024)
# C4 (decode_step_fused_kernel, one launch): FETCH 202338.9 KiB x 1.99983 + WRITE 4614.3 KiB, the read
# factor from the 512 MiB copy of the same run (profiles/decode_attention_c4.md)
C4_TRAFFIC_BYTES = int((202338.9 * 1.99983 + 4614.3) * 1024)
C2_TRAFFIC_BYTES = int((2057 + 2112) * 1024)
C5_TRAFFIC_BYTES = {0.10: (515 + 64) << 20, 0.25: (1175 + 64) << 20, 0.50: (2249 + 64) << 20}
# Prefill attention, one step (sa_vmax + sa_vt16 + sparse_attn_lds, profiles/sparse_attention_prefill_16k.md):
# (873685.9 + 16425.7 + 16507.2) KiB x 1.99983 read + (131285.4 + 32 + 32768.1) KiB written
PREFILL_ATTN_TRAFFIC_BYTES = int(906618.8 * 1.99983 * 1024 + 164085.5 * 1024)
# C2: wave-level VALU instructions of one score_route_kernel launch (rocprofv3 SQ_INSTS_VALU)
C2_VALU_INSTS = 47_169_428
VALU_PEAK_GIPS = 256 * 4 * 2.4 / 4  # G wave64 VALU instructions/s: 256 CUs x 4 SIMDs x 2.4 GHz / 4 cycles


def decode_bytes(n_active: int, batch: int) -> int:
    """Algorithmic HBM bytes of one decode forward: the active rows of k_gate,
    k_up and v (3 x 64 x 4096 x 2 B per block) plus x in and y out."""
    return n_active * 3 * BLOCK * D_MODEL * 2 + 2 * batch * D_MODEL * 2


def prefill_flops(n_active: int, tokens: int) -> int:
    """Algorithmic FLOPs of one forward: 3 GEMMs of tokens x 4096 x (64 n_active)."""
    return 2 * tokens * D_MODEL * 3 * BLOCK * n_active


def make_layers(fsi, n_layers: int, dev):
    layers = []
    g = torch.Generator(device=dev).manual_seed(0)
    for li in range(n_layers):
        m = fsi.FovealPattentionMLP(hidden_dim=D_MODEL, intermediate_dim=N_PARAM, block_size=BLOCK, base_blocks=BASE,
                                    remote_blocks=REMOTE, dtype=torch.bfloat16, use_fused_kernel=True)
        m = m.to(dev).eval()
        with torch.no_grad():
            for p in (m.k_gate, m.k_up, m.v):
                p.normal_(0.0, 0.02, generator=g)
            q = torch.linalg.qr(torch.randn(D_MODEL, 16, device=dev, generator=g, dtype=torch.float32))[0]
            m.q_proj_16d.weight.copy_(q.t())
            m.block_keys_16d.normal_(0.0, 0.25, generator=g)
        layers.append(m)
    return layers


EAGER = False  # --eager: launch every step directly (per-dispatch profiler counters), no graph


def time_graph(fn_steps, steps: int, warmup: int, dev):
    """Warm up eagerly, capture `steps` steps in one graph, replay once untimed,
    then time one replay with events on the capture stream."""
    for i in range(warmup):
        fn_steps(i)
    torch.cuda.synchronize(dev)
    if EAGER:
        start = torch.cuda.Event(enable_timing=True)
        end = torch.cuda.Event(enable_timing=True)
        s = torch.cuda.current_stream(dev)
        t0 = time.perf_counter()
        start.record(s)
        for i in range(steps):
            fn_steps(i)
        end.record(s)
        torch.cuda.synchronize(dev)
        return start.elapsed_time(end) / 1e3, time.perf_counter() - t0
    graph = torch.cuda.CUDAGraph()
    stream = torch.cuda.Stream(dev)
    stream.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            for i in range(steps):
                fn_steps(i)
    torch.cuda.synchronize(dev)
    graph.replay()
    torch.cuda.synchronize(dev)
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    replay_stream = torch.cuda.current_stream(dev)
    torch.cuda.synchronize(dev)
    t0 = time.perf_counter()
    start.record(replay_stream)
    graph.replay()
    end.record(replay_stream)
    torch.cuda.synchronize(dev)
    wall = time.perf_counter() - t0
    return start.elapsed_time(end) / 1e3, wall


def cpu_baseline(layer_cpu, x_cpu, active, reps: int):
    """The oracle's torch-CPU restatement of the reference eval forward, all host cores."""
    from oracle import pattention as opatt

    cores = len(os.sched_getaffinity(0))
    torch.set_num_threads(cores)
    kg, ku, v = layer_cpu
    for _ in range(2):
        opatt.mlp_eval_forward(x_cpu, kg, ku, v, active, BLOCK, fused=True)
    ts = []
    for _ in range(reps):
        t0 = time.perf_counter()
        opatt.mlp_eval_forward(x_cpu, kg, ku, v, active, BLOCK, fused=True)
        ts.append(time.perf_counter() - t0)
    ts.sort()
    return ts[len(ts) // 2], cores


def _result(metric, value, unit, steps, warmup, ms, dtype, data, config, higher=True):
    return {"metric": metric, "value": value, "unit": unit, "n_gpus": 1, "steps": steps, "warmup": warmup,
            "ms_per_step": ms, "higher_is_better": higher, "scaling": "weak", "vs_baseline": None, "dtype": dtype,
            "data": data, "config": config}


def c2_inputs(Q: int, N: int, dev, seed: int = 0):
    """Queries = Dirichlet(0.3)-weighted mixes of 4 random keys + N(0, 0.1) noise;
    keys N(0,1) then L2-normalised; both bf16."""
    g = torch.Generator().manual_seed(seed)
    keys = torch.nn.functional.normalize(torch.randn(N, 16, generator=g), dim=-1)
    j = torch.argsort(torch.rand(Q, N, generator=g), dim=1)[:, :4]
    w = torch.distributions.Dirichlet(torch.full((4,), 0.3)).sample((Q,))
    q = (w[..., None] * keys[j]).sum(1) + 0.1 * torch.randn(Q, 16, generator=g)
    return q.bfloat16().to(dev), keys.bfloat16().to(dev)


def bench_routing(fsi, args, dev):
    Q, N, KMIN, KMAX, CAP, TOP_P = 8192, 4096, 4, 64, 64, 0.9
    q, k = c2_inputs(Q, N, dev)
    outs = {}

    def step(i):
        outs["r"] = fsi.score_and_route(q, k, causal=False, top_p=TOP_P, min_remote_blocks=KMIN,
                                        max_remote_blocks=KMAX, remote_capacity=CAP, return_mass=True)

    t, _ = time_graph(step, args.steps, args.warmup, dev)
    per = t / args.steps
    counts = outs["r"][1].float()
    algo = Q * 16 * 2 + N * 16 * 2 + Q * CAP * 4 + Q * 4 * 2
    res = _result("indexer routing queries/s (fused 16-D cosine scoring + top-p selection)", round(Q / per, 1),
                  "queries/s", args.steps, args.warmup, round(per * 1e3, 6), "fp32",
                  "synthetic (seeded Dirichlet(0.3) mixes of 4 N(0,1)-normalised keys + N(0,0.1) noise, bf16)",
                  {"workload": "C2: 8192 queries x 4096 block keys, index_dim 16, top-p 0.9, K_min 4, K_max 64, "
                               "capacity 64, non-causal", "mean_selected": round(float(counts.mean()), 2)})
    # Algorithmic roofline: per query 4096 16-D scores (65,536 FMA = 131,072 flop) and
    # 4096 exps, counted one flop each, against the fp32 peak; the top-64 rank per
    # query has no flop count of its own, so this fraction understates the work.
    # Diagnostic beside it: the launch's wave-level VALU instruction count (rocprofv3
    # SQ_INSTS_VALU, profiles/indexer_routing_c2.md) over the issue peak of 256 CUs x
    # 4 SIMDs x 2.4 GHz / 4 cycles per wave64 instruction.
    flops = Q * N * (2 * 16 + 1)
    tfs = flops / per / 1e12
    gips = C2_VALU_INSTS / per / 1e9
    res["roofline"] = {"bound": "valu", "achieved": round(tfs, 3), "peak": FP32_PEAK_TFLOPS, "unit": "TFLOP/s",
                       "frac": round(tfs / FP32_PEAK_TFLOPS, 4), "traffic": C2_TRAFFIC_BYTES,
                       "kernel": "score_route_kernel (1 launch)", "flops_per_launch": flops,
                       "bytes_per_launch": algo, "hbm_gbs": round(algo / per / 1e9, 2),
                       "valu_issue": {"achieved": round(gips, 1), "peak": VALU_PEAK_GIPS,
                                      "unit": "G VALU wave-instructions/s", "frac": round(gips / VALU_PEAK_GIPS, 4),
                                      "valu_insts_per_launch": C2_VALU_INSTS},
                       "note": "not HBM-bound: 33.5 M scores, exps and a top-64 rank per launch; exps, "
                               "scores and the rank share the VALU issue"}
    if not args.no_cpu_baseline:
        from oracle import routing as R

        cores = len(os.sched_getaffinity(0))
        torch.set_num_threads(cores)
        qs, ks = q[:1024].cpu(), k.cpu()
        R.select_route(R.cosine_scores_f32(qs[None], ks[None]), causal=False, top_p=TOP_P, min_remote_blocks=KMIN,
                       max_remote_blocks=KMAX, remote_capacity=CAP)
        ts = []
        for _ in range(3):
            t0 = time.perf_counter()
            R.select_route(R.cosine_scores_f32(qs[None], ks[None]), causal=False, top_p=TOP_P,
                           min_remote_blocks=KMIN, max_remote_blocks=KMAX, remote_capacity=CAP)
            ts.append(time.perf_counter() - t0)
        med = sorted(ts)[1]
        res["cpu_baseline"] = {"value": round(1024 / med, 1), "unit": "queries/s", "cores": cores, "kind": "port",
                               "sample": f"oracle torch-CPU cosine scores + select_blocks on the first 1024 of the "
                                         f"8192 queries, median of 3, {med * 1e3:.1f} ms"}
    return res


C4 = dict(B=32, HQ=32, HKV=8, HD=128, CTX=131072, PAGE=64, W=1024, KMAX=32, TOP_P=0.9, N_PHYS=65536)


def c4_inputs(fsi, dev):
    """C4 decode attention inputs: a 65536-page K/V pool (N(0,1), 16 GiB), a seeded
    random page table, normalised fp32 page keys, bf16 q and rms-normed 16-D query."""
    c = C4
    B, P = c["B"], c["CTX"] // c["PAGE"]
    g = torch.Generator(device=dev).manual_seed(0)
    table = torch.randperm(c["N_PHYS"], device=dev, generator=g)[:B * P].view(B, P).to(torch.int32)
    cache = fsi.FovealKVCache(B, c["CTX"], c["HKV"], c["HD"], 16, c["PAGE"], dev, torch.bfloat16,
                              n_phys_pages=c["N_PHYS"], page_table=table)
    # pools filled in place: every page holds N(0,1) keys and values
    cache.k_cache.normal_(generator=g)
    cache.v_cache.normal_(generator=g)
    cache.kp_cache.copy_(torch.nn.functional.normalize(torch.randn(B, P, 16, device=dev, generator=g), dim=-1))
    cache.vp_cache.normal_(generator=g)
    cache.seq_len, cache.completed_pages = c["CTX"], P
    q = torch.randn(B, c["HQ"], c["HD"], device=dev, generator=g).bfloat16()
    qi = torch.nn.functional.rms_norm(torch.randn(B, 16, device=dev, generator=g), (16,)).bfloat16()
    return cache, q, qi


def bench_decode_attn(fsi, args, dev):
    B, HQ, HKV, HD, CTX, PAGE, W, KMAX, TOP_P = (C4[k] for k in ("B", "HQ", "HKV", "HD", "CTX", "PAGE", "W", "KMAX",
                                                                 "TOP_P"))
    P = CTX // PAGE
    cache, q, qi = c4_inputs(fsi, dev)
    pos = CTX - 1
    scale = 1.0 / (HD ** 0.5)
    outs = {}

    outs_pages = {}

    def step(i):
        # routing beside the local-window attention partials, then the selected pages and the merge
        outs["o"], outs_pages["p"], outs["c"], ctx = fsi.decode_step_attention(
            q, qi, cache, pos=pos, window=W, completed_pages=P, top_p=TOP_P, min_remote_blocks=0,
            max_remote_blocks=KMAX, scale=scale, return_context=True)

    t, _ = time_graph(step, args.steps, args.warmup, dev)
    per = t / args.steps
    k_sel = float(outs["c"].float().mean())
    flp = (pos + 1 - W) // PAGE
    kv_bytes = int(B * (W + PAGE * k_sel) * HKV * HD * 2 * 2)
    algo = kv_bytes + B * flp * 16 * 4 + B * P * 16 * 2 + 2 * B * HQ * HD * 2
    gbs = algo / per / 1e9
    res = _result("foveal decode attention tok/s (32 sequences x 131072 context, local 1024 + top-p pages)",
                  round(B / per, 1), "tok/s", args.steps, args.warmup, round(per * 1e3, 6), "bf16",
                  "synthetic (seeded N(0,1) K/V pool of 65536 pages, random page table, normalised page keys)",
                  {"workload": "C4: Llama-3-8B attention shape (32 q heads, 8 KV heads, head_dim 128), batch 32, "
                               "context 131072, page 64, local window 1024, top-p 0.9, K_max 32",
                   "mean_selected_pages": round(k_sel, 2)})
    res["roofline"] = {"bound": "hbm", "achieved": round(gbs, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                       "frac": round(gbs / HBM_PEAK_GBS, 4), "traffic": C4_TRAFFIC_BYTES,
                       "kernel": "decode_step_fused_kernel (1 launch: per (sequence, KV head) workgroup, 4 waves "
                                 "route while 4 stream the window, then all take selected-page chunks, in-workgroup merge)",
                       "bytes_per_launch": algo}
    # fp32 over the reference's contiguous cache layout (FovealKVCache's default dtype),
    # all 32 sequences (34.4 GB of K / V), the same pages: dec32_partial_kernel + merge
    nb = B
    c32 = fsi.FovealKVCache(nb, CTX, HKV, HD, 16, PAGE, dev, torch.float32)
    g32 = torch.Generator(device=dev).manual_seed(1)
    c32.k_cache.normal_(generator=g32)
    c32.v_cache.normal_(generator=g32)
    q32 = q[:nb].float()
    pg32, ct32 = outs_pages["p"][:nb].contiguous(), outs["c"][:nb].contiguous()
    o32 = {}

    def step32(i):
        o32["o"] = fsi.decode_attention(q32, c32, pos=pos, window=W, remote_pages=pg32, remote_counts=ct32,
                                        scale=scale)

    t32, _ = time_graph(step32, args.steps, args.warmup, dev)
    per32 = t32 / args.steps
    k32 = float(ct32.float().mean())
    b32 = int(nb * (W + PAGE * k32) * HKV * HD * 4 * 2)
    res["fp32"] = {"ms_per_step": round(per32 * 1e3, 4), "sequences": nb, "kv_bytes": b32,
                   "gbs": round(b32 / per32 / 1e9, 1), "frac": round(b32 / per32 / 1e9 / HBM_PEAK_GBS, 4),
                   "kernel": "dec32_partial_kernel<128> + dec32_merge_kernel<128> (contiguous fp32 cache)"}
    del c32
    if not args.no_cpu_baseline:
        from oracle import attention as A

        cores = len(os.sched_getaffinity(0))
        torch.set_num_threads(cores)
        # the reference's dense-layout decode attention on 4 sequences' supports, gathered on the host
        pages, counts = fsi.decode_route(qi, cache.kp_cache, None, pos=pos, page_size=PAGE, local_window=W,
                                         completed_pages=P, top_p=TOP_P, min_remote_blocks=0,
                                         max_remote_blocks=KMAX)
        nb = 4
        kd, vd = cache.to_dense(CTX, batch=slice(0, nb))
        kc, vc = kd.cpu(), vd.cpu()
        del kd, vd
        pl = [pages[b, :int(counts[b])].tolist() for b in range(nb)]
        qc = q[:nb].cpu()
        ts = []
        for _ in range(3):
            t0 = time.perf_counter()
            for b in range(nb):
                toks = torch.tensor(A.support_tokens(pos, W, pl[b], PAGE))
                kk = kc[b][:, toks].repeat_interleave(HQ // HKV, dim=0)
                vv = vc[b][:, toks].repeat_interleave(HQ // HKV, dim=0)
                torch.nn.functional.scaled_dot_product_attention(qc[b][:, None], kk, vv, scale=scale)
            ts.append(time.perf_counter() - t0)
        med = sorted(ts)[1]
        res["cpu_baseline"] = {"value": round(nb / med, 1), "unit": "tok/s", "cores": cores, "kind": "port",
                               "sample": f"gather + repeat_interleave + bf16 SDPA on the host for 4 of the 32 "
                                         f"sequences (attention.py:339-365 order), median of 3, {med * 1e3:.1f} ms"}
    return res


def prefill_attn_flops(lists, counts, T: int, W: int, page: int, hq: int, hd: int) -> int:
    """Algorithmic FLOPs of block-sparse prefill attention: for every query, its
    attended keys (the causal window of W keys plus the keys of its block's
    listed pages outside that window) x 4 hd FLOPs (QK^T and PV) x heads."""
    B, Qb, _ = lists.shape
    t = torch.arange(T, device=lists.device)
    keys = torch.clamp(t + 1, max=W).to(torch.int64).expand(B, T).clone()
    slot = torch.arange(lists.shape[2], device=lists.device)
    valid = slot[None, None] < counts[..., None]
    first = (lists.to(torch.int64) * page).masked_fill(~valid, T)       # (B, Qb, cap)
    first_t = first.repeat_interleave(page, dim=1)[:, :T]                # (B, T, cap)
    outside = torch.clamp(t[None, :, None] - W + 1 - first_t, min=0, max=page)
    keys += outside.sum(-1)
    return int(keys.sum()) * hq * hd * 4


PREFILL_ATTN = dict(B=1, HQ=32, HKV=8, HD=128, T=16384, PAGE=64, WB=16, KMAX=32, TOP_P=0.9)


def prefill_attn_inputs(fsi, dev):
    """The prefill-attention workload: seeded N(0,1) q (B, 32, 16384, 128) and
    k, v (B, 8, 16384, 128) bf16, and the pages routed as
    FovealSparseAttention.forward does: cosine/4 block scores of block-anchor
    16-D queries against normalised 16-D page keys, causal top-p with the
    16-page local window.  Returns (q, k, v, lists, counts)."""
    c = PREFILL_ATTN
    B, HQ, HKV, HD, T, PAGE = c["B"], c["HQ"], c["HKV"], c["HD"], c["T"], c["PAGE"]
    Qb = T // PAGE
    g = torch.Generator(device=dev).manual_seed(0)
    q = torch.randn(B, HQ, T, HD, device=dev, generator=g).bfloat16()
    k = torch.randn(B, HKV, T, HD, device=dev, generator=g).bfloat16()
    v = torch.randn(B, HKV, T, HD, device=dev, generator=g).bfloat16()
    qi = torch.nn.functional.normalize(torch.randn(B, Qb, 16, device=dev, generator=g), dim=-1)
    kp = torch.nn.functional.normalize(torch.randn(B, Qb, 16, device=dev, generator=g), dim=-1)
    scores = torch.bmm(qi, kp.transpose(1, 2).contiguous()) / 4.0
    route = fsi.select_blocks(scores, causal=True, block_size=PAGE, local_window_blocks=c["WB"], top_p=c["TOP_P"],
                              min_remote_blocks=0, max_remote_blocks=c["KMAX"], remote_capacity=c["KMAX"])
    return q, k, v, route.remote_indices, route.remote_counts


def bench_prefill_attn(fsi, args, dev):
    c = PREFILL_ATTN
    B, HQ, HKV, HD, T, PAGE, WB = c["B"], c["HQ"], c["HKV"], c["HD"], c["T"], c["PAGE"], c["WB"]
    W = WB * PAGE
    Qb = T // PAGE
    q, k, v, lists, counts = prefill_attn_inputs(fsi, dev)
    out = torch.empty(B, T, HQ, HD, dtype=torch.bfloat16, device=dev)
    scale = 1.0 / HD ** 0.5

    def step(i):
        fsi.sparse_attention(q, k, v, lists, counts, block=PAGE, mode=0, window=W, scale=scale,
                             out=out.transpose(1, 2))

    t, _ = time_graph(step, args.steps, args.warmup, dev)
    per = t / args.steps
    flops = prefill_attn_flops(lists, counts, T, W, PAGE, HQ, HD)
    tfs = flops / per / 1e12
    res = _result("foveal prefill attention tok/s (16384 tokens, local 1024 + top-p pages)", round(B * T / per, 1),
                  "tok/s", args.steps, args.warmup, round(per * 1e3, 6), "bf16",
                  "synthetic (seeded N(0,1) q/k/v; pages routed by select_blocks on cosine/4 scores of random "
                  "normalised 16-D anchors and page keys)",
                  {"workload": "FovealSparseAttention.forward attention core at the Llama-3-8B attention shape "
                               "(32 q heads, 8 KV heads, head_dim 128), batch 1 x 16384 tokens, page 64, local "
                               "window 1024, top-p 0.9, K_max 32",
                   "mean_remote_pages": round(float(counts.float().mean()), 2)})
    # the backward (fsi_sparse_attn_bwd, training through FovealSparseAttention.forward)
    # on the same pattern, timed eagerly: 2.5 x the forward's products (Q K^T and dP
    # recomputed, dV, dQ, dK)
    from foveal_sparse_indexer_amd import attention as fatt

    out4 = out.transpose(1, 2)
    g = torch.Generator(device=dev).manual_seed(5)
    dout = torch.randn(B, HQ, T, HD, device=dev, generator=g).bfloat16()
    for _ in range(2):
        fatt._sparse_attention_bwd(q, k, v, out4, dout, lists, counts, c["KMAX"], PAGE, 0, W, scale)
    torch.cuda.synchronize(dev)
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    n_bwd = 3
    ev0.record()
    for _ in range(n_bwd):
        fatt._sparse_attention_bwd(q, k, v, out4, dout, lists, counts, c["KMAX"], PAGE, 0, W, scale)
    ev1.record()
    torch.cuda.synchronize(dev)
    bwd_ms = ev0.elapsed_time(ev1) / n_bwd
    bwd_tf = 2.5 * flops / (bwd_ms * 1e-3) / 1e12
    # the same forward in fp32 (FovealSparseAttention's default dtype): the fp32
    # MFMA kernel (sparse_attn_f32_kernel), graded against the fp32 matrix peak
    q32, k32, v32 = q.float(), k.float(), v.float()
    out32 = torch.empty(B, T, HQ, HD, dtype=torch.float32, device=dev)

    def step32(i):
        fsi.sparse_attention(q32, k32, v32, lists, counts, block=PAGE, mode=0, window=W, scale=scale,
                             out=out32.transpose(1, 2))

    n32s = max(1, args.steps // 2)
    t32, _ = time_graph(step32, n32s, args.warmup, dev)
    tf32 = flops / (t32 / n32s) / 1e12
    res["fp32"] = {"ms_per_step": round(t32 / n32s * 1e3, 4), "tflops": round(tf32, 1), "peak": FP32_PEAK_TFLOPS,
                   "frac": round(tf32 / FP32_PEAK_TFLOPS, 4),
                   "kernel": "vt32_kernel + sparse_attn_f32_kernel<128> (v_mfma_f32_16x16x4_f32)"}
    del q32, k32, v32, out32
    res["backward"] = {"ms": round(bwd_ms, 3), "tflops": round(bwd_tf, 1), "peak": BF16_PEAK_TFLOPS,
                       "frac": round(bwd_tf / BF16_PEAK_TFLOPS, 4),
                       "flops": int(2.5 * flops), "kernel": "sab_map + sab_q_bf (statistics, dQ) + sab_kv_bf (dK, dV)",
                       "note": "every product on v_mfma_f32_16x16x32_bf16 over bf16 LDS tiles (direct-to-LDS; "
                               "transposed operands by ds_read_b64_tr_b16); P and dS enter dV / dK / dQ as bf16 hi + lo pairs (~2^-17 relative), "
                               "fp32 accumulation; memory O(T hd), no (T, T) tensor"}
    res["roofline"] = {"bound": "mfma", "achieved": round(tfs, 1), "peak": BF16_PEAK_TFLOPS, "unit": "TFLOP/s",
                       "frac": round(tfs / BF16_PEAK_TFLOPS, 4), "traffic": PREFILL_ATTN_TRAFFIC_BYTES,
                       "kernel": "sa_vmax_kernel + sa_vt16_kernel + sparse_attn_lds_kernel (3 launches)", "flops_per_launch": flops}
    if not args.no_cpu_baseline:
        cores = len(os.sched_getaffinity(0))
        torch.set_num_threads(cores)
        # the reference's dense masked SDPA (attention.py:199-216) for the last query block only
        nq = PAGE
        qc = q[:, :, T - nq:].cpu()
        kc = k.cpu().repeat_interleave(HQ // HKV, dim=1)
        vc = v.cpu().repeat_interleave(HQ // HKV, dim=1)
        tq = torch.arange(T - nq, T)
        ks = torch.arange(T)
        mask = (ks[None] <= tq[:, None]) & (ks[None] > tq[:, None] - W)
        for p in lists[0, Qb - 1, :int(counts[0, Qb - 1])].tolist():
            mask[:, p * PAGE:(p + 1) * PAGE] = True
        ts = []
        for _ in range(3):
            t0 = time.perf_counter()
            torch.nn.functional.scaled_dot_product_attention(qc, kc, vc, attn_mask=mask[None, None], scale=scale)
            ts.append(time.perf_counter() - t0)
        med = sorted(ts)[1]
        res["cpu_baseline"] = {"value": round(nq / med, 1), "unit": "tok/s", "cores": cores, "kind": "port",
                               "sample": f"the reference's dense bool-masked bf16 SDPA over all 16384 keys for the "
                                         f"last 64-query block (32 heads), median of 3, {med * 1e3:.1f} ms"}
    return res


C5 = dict(M=4096, K=8192, N=8192, T=128, DENSITIES=(0.10, 0.25, 0.50))


def c5_inputs(dev):
    """C5 inputs: X N(0,1) (4096, 8192) and W N(0, 0.01^2) (8192, 8192) bf16, plus
    seeded uniform tile scores per 128-row group (32 x 4096 tiles)."""
    M, K, N, T = C5["M"], C5["K"], C5["N"], C5["T"]
    g = torch.Generator(device=dev).manual_seed(0)
    x = torch.randn(M, K, device=dev, generator=g).bfloat16()
    w = (torch.randn(N, K, device=dev, generator=g) * 0.01).bfloat16()
    scores = torch.rand(M // T, (K // T) * (N // T), device=dev, generator=g)
    return x, w, scores


def c5_mask(scores, density: float):
    """Per-row-group tile masks: the top ceil(density x tiles) tiles of each group's scores."""
    groups, tiles = scores.shape
    n_tiles = int(-(-density * tiles // 1))
    mask = torch.zeros(groups, tiles, dtype=torch.bool, device=scores.device)
    mask.scatter_(1, scores.topk(n_tiles, dim=1).indices, True)
    return mask, n_tiles


def bench_block_sparse(fsi, args, dev):
    M, K, N, T = C5["M"], C5["K"], C5["N"], C5["T"]
    groups, nkb, nnb = M // T, K // T, N // T
    x, w, scores = c5_inputs(dev)
    lines = {}
    for d in C5["DENSITIES"]:
        mask, n_tiles = c5_mask(scores, d)
        outs = {}

        def step(i):
            outs["o"] = fsi.blockwise_matmul(x, w, mask, T, T, rows_per_group=T)

        t, _ = time_graph(step, args.steps, args.warmup, dev)
        per = t / args.steps
        flops = groups * n_tiles * 2 * T * T * T
        # HBM floor: X and Y once plus every weight tile some group uses
        hbm = 2 * M * K * 2 + int(mask.any(dim=0).sum()) * T * T * 2
        lines[d] = (per, flops, n_tiles, hbm)
    per, flops, n_tiles, _ = lines[0.25]
    tf = flops / per / 1e12

    def grade(v):
        per_d, fl, nt, hbm = v
        tfs, gbs = fl / per_d / 1e12, hbm / per_d / 1e9
        # the bound is whichever floor is longer: MFMA time or HBM time
        bound = "mfma" if fl / (BF16_PEAK_TFLOPS * 1e12) >= hbm / (HBM_PEAK_GBS * 1e9) else "hbm"
        return {"ms_per_step": round(per_d * 1e3, 4), "tiles_per_group": nt, "tflops": round(tfs, 2),
                "hbm_bytes": hbm, "gbs": round(gbs, 1), "bound": bound,
                "frac": round(tfs / BF16_PEAK_TFLOPS if bound == "mfma" else gbs / HBM_PEAK_GBS, 4)}

    res = _result("2-D tile-sparse matmul TFLOP/s (per-row-group 128x128 tile masks)", round(tf, 2), "TFLOP/s",
                  args.steps, args.warmup, round(per * 1e3, 6), "bf16",
                  "synthetic (seeded N(0,1) X, N(0,0.01) W, per-row-group top-d tiles of seeded uniform scores)",
                  {"workload": "C5: X 4096 x 8192, W 8192 x 8192 in 128 x 128 tiles (4096), one mask per 128-row "
                               "group (32 groups), density 25% (1024 tiles per group)",
                   "densities": {f"{d:.2f}": dict(grade(v), traffic=C5_TRAFFIC_BYTES.get(d))
                                 for d, v in lines.items()}})
    res["roofline"] = {"bound": "mfma", "achieved": round(tf, 2), "peak": BF16_PEAK_TFLOPS, "unit": "TFLOP/s",
                       "frac": round(tf / BF16_PEAK_TFLOPS, 4), "traffic": C5_TRAFFIC_BYTES[0.25],
                       "kernel": "tile_list_gemm_kernel (k-block lists built in its prologue)",
                       "flops_per_launch": flops}
    # the same 25% product in fp32 (the reference modules' default dtype):
    # tile_list_gemm_kernel<float> on v_mfma_f32_16x16x4_f32, graded against the
    # fp32 matrix peak
    x32, w32 = x.float(), w.float()
    mask, n_tiles = c5_mask(scores, 0.25)
    outs32 = {}

    def step32(i):
        outs32["o"] = fsi.blockwise_matmul(x32, w32, mask, T, T, rows_per_group=T)

    t32, _ = time_graph(step32, max(1, args.steps // 2), args.warmup, dev)
    per32 = t32 / max(1, args.steps // 2)
    tf32 = flops / per32 / 1e12
    res["fp32"] = {"ms_per_step": round(per32 * 1e3, 4), "tflops": round(tf32, 2), "peak": FP32_PEAK_TFLOPS,
                   "frac": round(tf32 / FP32_PEAK_TFLOPS, 4), "density": 0.25,
                   "kernel": "tile_list_gemm_kernel<float> (v_mfma_f32_16x16x4_f32)"}
    del x32, w32, outs32
    if not args.no_cpu_baseline:
        cores = len(os.sched_getaffinity(0))
        torch.set_num_threads(cores)
        from oracle import blocksparse as BS

        # masked dense matmul on the host for one 128-row group at 25% density
        mask, n_tiles = c5_mask(scores, 0.25)
        xc, wc = x[:T].cpu(), w.cpu()
        em = BS.expand_tile_mask(mask[0].cpu(), N, K, T, T)
        ts = []
        for _ in range(3):
            t0 = time.perf_counter()
            torch.nn.functional.linear(xc, wc * em)
            ts.append(time.perf_counter() - t0)
        med = sorted(ts)[1]
        gflop = n_tiles * 2 * T ** 3
        res["cpu_baseline"] = {"value": round(gflop / med / 1e12, 4), "unit": "TFLOP/s", "cores": cores,
                               "kind": "port", "sample": f"masked dense F.linear on the host for one 128-row group "
                                                         f"at 25% density (bf16), median of 3, {med * 1e3:.1f} ms"}
    return res


def bench_teacher_targets(fsi, args, dev):
    """Dense block-energy teacher targets (compute_teacher_dense_block_targets) for
    one Llama-3-8B MLP over 4096 tokens: the fused gate/up GEMM with the |act|
    block-sum epilogue plus the column-norm and softmax kernels."""
    M, D, I, BS, T = 4096, D_MODEL, N_PARAM, 64, 1.0
    g = torch.Generator(device=dev).manual_seed(0)
    h = torch.randn(M, D, device=dev, generator=g).bfloat16()
    gw = (torch.randn(I, D, device=dev, generator=g) * 0.02).bfloat16()
    uw = (torch.randn(I, D, device=dev, generator=g) * 0.02).bfloat16()
    dw = (torch.randn(D, I, device=dev, generator=g) * 0.02).bfloat16()
    out = {}

    def step(i):
        out["p"] = fsi.dense_block_targets(h, gw, uw, dw, BS, T)

    t, _ = time_graph(step, args.steps, args.warmup, dev)
    per = t / args.steps
    flops = 2 * M * D * 2 * I
    tfs = flops / per / 1e12
    res = _result("dense teacher block targets tok/s (Llama-3-8B MLP, 4096 tokens)", round(M / per, 1), "tok/s",
                  args.steps, args.warmup, round(per * 1e3, 6), "bf16",
                  "synthetic (seeded N(0,1) hidden states, N(0,0.02) gate/up/down weights)",
                  {"workload": "compute_teacher_dense_block_targets per layer: h (4096, 4096), gate/up (14336, 4096), "
                               "down (4096, 14336), block 64 (224 blocks), T = 1"})
    res["roofline"] = {"bound": "mfma", "achieved": round(tfs, 1), "peak": BF16_PEAK_TFLOPS, "unit": "TFLOP/s",
                       "frac": round(tfs / BF16_PEAK_TFLOPS, 4), "traffic": None,
                       "kernel": "bsgemm_dma_kernel<N_DUAL, K_DENSE, EPI_ENERGY> (+ column_sumsq_kernel, "
                                 "column_norms_kernel, block_mean_kernel, block_softmax_kernel: 5 launches)",
                       "flops_per_launch": flops}
    if not args.no_cpu_baseline:
        cores = len(os.sched_getaffinity(0))
        torch.set_num_threads(cores)
        from oracle import pattention as OP

        n = 64
        hc, gc, uc, dc = h[:n].cpu(), gw.cpu(), uw.cpu(), dw.cpu()
        ts = []
        for _ in range(3):
            t0 = time.perf_counter()
            OP.dense_block_targets(hc, gc, uc, dc, BS, T)
            ts.append(time.perf_counter() - t0)
        med = sorted(ts)[1]
        res["cpu_baseline"] = {"value": round(n / med, 1), "unit": "tok/s", "cores": cores, "kind": "port",
                               "sample": f"the reference's torch ops (bf16, train_foveal_pattention_speedrun.py:"
                                         f"176-185) on the host for 64 of the 4096 tokens, median of 3, "
                                         f"{med * 1e3:.1f} ms"}
    return res


SRAM_CONFIGS = [(64, 64, 16), (32, 256, 16), (16, 1024, 32)]  # (batch, seq_len, block_size)
SRAM_REF_A10G_MS = [0.0566, 0.0515, 0.0619]  # the reference's fused kernel on A10G, BENCHMARKS.md:308-314


def bench_sram_attn(fsi, args, dev):
    """The reference's SRAM-fused indexer benchmark (benchmark_a10g_full.py:314-376):
    fp16, 4 heads, head_dim 32, max_remote 2, top_p 0.8, three (batch, seq_len,
    block) configs; one call of each per step.  HBM bytes per call: q and the
    output once, k and v of the self block plus every attended pick per query
    block and head, q16 / k16 once."""
    H, D, R = 4, 32, 2
    g = torch.Generator(device=dev).manual_seed(0)
    cases, bytes_call, per_cfg = [], 0, []
    for B, N, bs in SRAM_CONFIGS:
        M = N // bs
        q, k, v = (torch.randn(B, H, N, D, device=dev, generator=g).half() for _ in range(3))
        q16, k16 = (torch.randn(B, M, 16, device=dev, generator=g).half() for _ in range(2))
        _, sel = fsi.sram_indexer_attention(q, k, v, q16, k16, max_remote_blocks=R, block_size=bs,
                                            return_selection=True)
        attended = int((sel >= 0).sum())
        b = 2 * (2 * B * H * N * D) + 2 * H * (B * M + attended) * bs * D * 2 + 2 * 2 * B * M * 16
        bytes_call += b
        cases.append((q, k, v, q16, k16, bs))
        per_cfg.append(b)
    out = {}

    def step(i):
        for j, (q, k, v, q16, k16, bs) in enumerate(cases):
            out[j] = fsi.sram_indexer_attention(q, k, v, q16, k16, max_remote_blocks=R, block_size=bs)

    t, _ = time_graph(step, args.steps, args.warmup, dev)
    per = t / args.steps
    ms_each = []
    for j, (q, k, v, q16, k16, bs) in enumerate(cases):
        def one(i, j=j):
            q_, k_, v_, a_, b_, bs_ = cases[j]
            out[j] = fsi.sram_indexer_attention(q_, k_, v_, a_, b_, max_remote_blocks=R, block_size=bs_)

        tj, _ = time_graph(one, args.steps, 1, dev)
        ms_each.append(round(tj / args.steps * 1e3, 5))
    gbs = bytes_call / per / 1e9
    res = _result("fused indexer attention: ms per call of the reference's 3 SRAM configs (sum)",
                  round(per * 1e3, 5), "ms", args.steps, args.warmup, round(per * 1e3, 5), "fp16",
                  "synthetic (seeded N(0,1) q, k, v, q16, k16)",
                  {"workload": "triton_fused_sram_indexer_attention: (B, N, block) in "
                               f"{SRAM_CONFIGS}, 4 heads, head_dim 32, max_remote 2, top_p 0.8",
                   "ms_per_config": ms_each, "reference_a10g_ms_per_config": SRAM_REF_A10G_MS},
                  higher=False)
    res["roofline"] = {"bound": "hbm", "achieved": round(gbs, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                       "frac": round(gbs / HBM_PEAK_GBS, 5), "traffic": None,
                       "kernel": "sram_attn_mfma_kernel (fp16: 16x16x16 MFMA tiles; one launch per config, latency bound at these sizes)",
                       "bytes_per_launch": per_cfg}
    if not args.no_cpu_baseline:
        from oracle import attention as OA

        cores = len(os.sched_getaffinity(0))
        torch.set_num_threads(cores)
        q, k, v, q16, k16, bs = cases[1]
        qc, kc, vc, ac, bc = (t.cpu() for t in (q, k, v, q16, k16))
        ts = []
        for _ in range(3):
            t0 = time.perf_counter()
            picks, _ = OA.sram_select(ac, bc, 0.8, R)
            OA.sram_attention_f64(qc, kc, vc, picks, bs, 1.0 / math.sqrt(D))
            ts.append(time.perf_counter() - t0)
        med = sorted(ts)[1]
        res["cpu_baseline"] = {"value": round(med * 1e3, 3), "unit": "ms", "cores": cores, "kind": "port",
                               "sample": "oracle sram_select (fp32) + sram_attention_f64 on the second config "
                                         "(B 32, N 256, block 16), median of 3"}
    return res


def library_gemm_ceiling(dev, n_active: int, steps: int) -> dict:
    """hipBLASLt (torch F.linear, bf16) on dense GEMMs of the prefill shapes: x (4096
    tokens x 4096) times the active gate+up rows (2 x 64 n_active x 4096) and H
    (4096 x 64 n_active) times the active V^T, timed like the prefill step.  The
    same FLOPs on the vendor library on this box: the practical MFMA ceiling."""
    n_ch = 64 * n_active
    g = torch.Generator(device=dev).manual_seed(7)
    x = torch.randn(PREFILL_TOKENS, D_MODEL, device=dev, generator=g).bfloat16()
    wgu = (torch.randn(2 * n_ch, D_MODEL, device=dev, generator=g) * 0.02).bfloat16()
    h = torch.randn(PREFILL_TOKENS, n_ch, device=dev, generator=g).bfloat16()
    wd = (torch.randn(D_MODEL, n_ch, device=dev, generator=g) * 0.02).bfloat16()
    outs = {}

    def gu(i):
        outs["g"] = torch.nn.functional.linear(x, wgu)

    def dn(i):
        outs["d"] = torch.nn.functional.linear(h, wd)

    res = {}
    for name, fn, fl in (("gateup", gu, 2 * PREFILL_TOKENS * D_MODEL * 2 * n_ch),
                         ("down", dn, 2 * PREFILL_TOKENS * n_ch * D_MODEL)):
        t, _ = time_graph(fn, steps, 2, dev)
        tf = fl / (t / steps) / 1e12
        res[name] = {"ms": round(t / steps * 1e3, 4), "tflops": round(tf, 1), "frac": round(tf / BF16_PEAK_TFLOPS, 4)}
    total = res["gateup"]["ms"] + res["down"]["ms"]
    tf = prefill_flops(n_active, PREFILL_TOKENS) / (total * 1e-3) / 1e12
    res["both"] = {"ms": round(total, 4), "tflops": round(tf, 1), "frac": round(tf / BF16_PEAK_TFLOPS, 4)}
    res["note"] = "torch F.linear (hipBLASLt) on dense operands of the same shapes; context, not this library"
    del x, wgu, h, wd, outs
    return res


def bench_hbm_stream(fsi, args, dev):
    """The practical HBM ceiling the HBM-bound kernels are measured against: a
    plain device copy (read + write) and a read-only sum, 4 GiB each, timed with
    events over graph replays like every other workload."""
    n = 4 << 30
    a = torch.empty(n, dtype=torch.uint8, device=dev).fill_(1)
    b = torch.empty_like(a)
    av = a.view(torch.float32)
    outs = {}

    def copy_step(i):
        b.copy_(a)

    def read_step(i):
        outs["s"] = av.sum()

    t_c, _ = time_graph(copy_step, args.steps, args.warmup, dev)
    t_r, _ = time_graph(read_step, args.steps, args.warmup, dev)
    copy_gbs = 2 * n / (t_c / args.steps) / 1e9
    read_gbs = n / (t_r / args.steps) / 1e9
    res = _result("HBM stream bandwidth GB/s (torch sum over 4 GiB)", round(read_gbs, 1), "GB/s", args.steps,
                  args.warmup, round(t_r / args.steps * 1e3, 6), "u8", "synthetic (4 GiB buffers)",
                  {"workload": "torch sum over 4 GiB of fp32 (read); torch copy_ of 4 GiB (read + write)",
                   "torch_copy_gbs": round(copy_gbs, 1), "torch_sum_gbs": round(read_gbs, 1)})
    res["roofline"] = {"bound": "hbm", "achieved": round(read_gbs, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                       "frac": round(read_gbs / HBM_PEAK_GBS, 4), "traffic": None}
    return res


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    # defaults: 1000 timed / 100 warm-up steps for the C3 decode line (a 30 ms timed
    # window; 200 / 10 measured ~3 % slower per step), 100 / 10 for a workload line
    ap.add_argument("--steps", type=int, default=None)
    ap.add_argument("--warmup", type=int, default=None)
    ap.add_argument("--layers", type=int, default=8)
    ap.add_argument("--prefill-steps", type=int, default=64)
    ap.add_argument("--no-prefill", action="store_true")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-workloads", action="store_true",
                    help="only the C3 line (skip the C2 / C4 / C5 / prefill-attention sub-objects)")
    ap.add_argument("--workload", default="pattention",
                    choices=["pattention", "routing", "decode_attn", "prefill_attn", "block_sparse",
                             "teacher_targets", "hbm_stream", "sram_attn"])
    ap.add_argument("--eager", action="store_true", help="no graph capture (for per-dispatch counter runs)")
    ap.add_argument("--no-pack", action="store_true",
                    help="decode from the parameters in place (4-kernel split-K path) instead of packed weights")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="also run one plain 512 MiB device copy (reference kernel for HBM counters)")
    args = ap.parse_args()
    direct = args.workload != "pattention"
    if args.steps is None:
        args.steps = 100 if direct else 1000
    if args.warmup is None:
        args.warmup = 10 if direct else 100
    global EAGER
    EAGER = args.eager
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU; --gpus {args.gpus} is not supported "
              "(the multi-GPU sharding of this path is described, not run)", file=sys.stderr)
        sys.exit(2)

    import __graft_entry__

    fsi = __graft_entry__.load_package()
    dev = torch.device("cuda:0")
    torch.manual_seed(0)
    if args.copy_calibration:
        # reference dispatch for the HBM counters: one plain 512 MiB device copy
        a = torch.empty(512 << 20, dtype=torch.uint8, device=dev)
        b = torch.empty_like(a)
        b.copy_(a)
        torch.cuda.synchronize(dev)
        del a, b
    if args.workload != "pattention":
        fn = {"routing": bench_routing, "decode_attn": bench_decode_attn, "prefill_attn": bench_prefill_attn,
              "block_sparse": bench_block_sparse, "teacher_targets": bench_teacher_targets,
              "hbm_stream": bench_hbm_stream, "sram_attn": bench_sram_attn}[args.workload]
        with torch.no_grad():
            print(json.dumps(fn(fsi, args, dev)), flush=True)
        return
    layers = make_layers(fsi, args.layers, dev)

    gx = torch.Generator(device=dev).manual_seed(1)
    x_dec = torch.randn(DECODE_BATCH, 1, D_MODEL, device=dev, generator=gx).bfloat16()
    x_pre = torch.randn(1, PREFILL_TOKENS, D_MODEL, device=dev, generator=gx).bfloat16()
    # Routing once per layer (the eval cache fill), then cached blocks for every step.
    # One decode call per layer packs its weights into the MFMA operand layout (a
    # once-per-weight-version transform, outside the timed region).
    with torch.no_grad():
        for m in layers:
            m.pack_decode_weights = not args.no_pack
            m.clear_cache()
            m(x_pre)
            m(x_dec)
    n_active = int(layers[0]._cached_active_blocks.numel())

    outs = {}

    def dec_step(i):
        outs["d"] = layers[i % len(layers)](x_dec)

    with torch.no_grad():
        t_dec, wall_dec = time_graph(dec_step, args.steps, args.warmup, dev)
    ms_dec = t_dec / args.steps * 1e3
    tok_s = DECODE_BATCH * args.steps / t_dec
    bytes_step = decode_bytes(n_active, DECODE_BATCH)
    achieved = bytes_step / (t_dec / args.steps) / 1e9

    result = {
        "metric": "Pattention MLP tok/s at 8B shape (b64 decode, 4K prefill); % roofline",
        "value": round(tok_s, 1),
        "unit": "tok/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_dec, 6),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic (seeded N(0,0.02) weights, orthonormal 4096->16 router, N(0,1) inputs)",
        "config": {
            "workload": "C3a: Llama-3-8B-shaped FovealPattentionMLP decode, batch 64 x 1 token, d_model 4096, "
                        "14336 parameter tokens (224 blocks of 64), 8 base + 56 remote active blocks",
            "global_batch": DECODE_BATCH,
            "seq_len": 1,
            "parallelism": "single GPU",
            "layers_cycled": args.layers,
            "n_active_blocks": n_active,
        },
        "roofline": {
            "bound": "hbm",
            "achieved": round(achieved, 1),
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": round(achieved / HBM_PEAK_GBS, 4),
            "traffic": (DECODE_TRAFFIC_BYTES_UNPACKED if args.no_pack else DECODE_TRAFFIC_BYTES)
                       if n_active == BASE + REMOTE else None,
            "kernel": ("decode forward = dec_gateup + dec_act + dec_down + dec_reduce (4 launches" if args.no_pack else
                       "decode forward = ws_gateup_kernel + ws_down_kernel over packed weights (2 launches")
                      + ", graph-replayed); achieved = algorithmic bytes of the forward / forward duration",
            "bytes_per_launch": bytes_step,
        },
    }

    if not args.no_prefill:
        def pre_step(i):
            outs["p"] = layers[i % len(layers)](x_pre)

        with torch.no_grad():
            t_pre, _ = time_graph(pre_step, args.prefill_steps, 2, dev)
        flops = prefill_flops(n_active, PREFILL_TOKENS)
        tflops = flops / (t_pre / args.prefill_steps) / 1e12
        result["prefill"] = {
            "value": round(PREFILL_TOKENS * args.prefill_steps / t_pre, 1),
            "unit": "tok/s",
            "steps": args.prefill_steps,
            "ms_per_step": round(t_pre / args.prefill_steps * 1e3, 4),
            "config": "C3b: 1 x 4096 tokens, same layers and active blocks",
            "roofline": {"bound": "mfma", "achieved": round(tflops, 2), "peak": BF16_PEAK_TFLOPS, "unit": "TFLOP/s",
                         "frac": round(tflops / BF16_PEAK_TFLOPS, 4),
                         "traffic": PREFILL_TRAFFIC_BYTES if n_active == BASE + REMOTE else None,
                         "flops_per_launch": flops},
            "library_gemm": library_gemm_ceiling(dev, n_active, args.prefill_steps),
        }

    if not args.no_cpu_baseline:
        m0 = layers[0]
        layer_cpu = (m0.k_gate.detach().cpu(), m0.k_up.detach().cpu(), m0.v.detach().cpu())
        act = m0._cached_active_blocks.cpu()
        med, cores = cpu_baseline(layer_cpu, x_dec.reshape(-1, D_MODEL).cpu(), act, reps=7)
        result["cpu_baseline"] = {
            "value": round(DECODE_BATCH / med, 1),
            "unit": "tok/s",
            "cores": cores,
            "kind": "port",
            "sample": f"oracle torch-CPU restatement of the eval forward (gather + 3 F.linear + fused SwiGLU), "
                      f"decode batch 64 on layer 0, median of 7 after 2 warm-ups, {med * 1e3:.1f} ms/step",
        }
        if "prefill" in result:
            med_p, _ = cpu_baseline(layer_cpu, x_pre.reshape(-1, D_MODEL).cpu(), act, reps=3)
            result["prefill"]["cpu_baseline"] = {
                "value": round(PREFILL_TOKENS / med_p, 1), "unit": "tok/s", "cores": cores, "kind": "port",
                "sample": f"oracle torch-CPU restatement of the eval forward on the full 4096-token prefill of layer "
                          f"0, median of 3 after 2 warm-ups, {med_p * 1e3:.1f} ms/step"}
    del layers, outs
    torch.cuda.empty_cache()

    if not args.no_workloads:
        # The other workloads, each one JSON sub-object with its own roofline and CPU baseline.
        sub_args = argparse.Namespace(**vars(args))
        # 100 graph-replayed steps (20 measured 5-10 % slower per step than 200: the
        # shorter timed window starts on a GPU that idled through the CPU baselines)
        sub_args.steps, sub_args.warmup = max(1, min(args.steps, 100)), max(1, min(args.warmup, 10))
        result["workloads"] = {}
        for name, fn in (("C2_routing", bench_routing), ("C4_decode_attention", bench_decode_attn),
                         ("C5_block_sparse", bench_block_sparse), ("prefill_attention", bench_prefill_attn),
                         ("sram_indexer_attention", bench_sram_attn)):
            with torch.no_grad():
                r = fn(fsi, sub_args, dev)
            result["workloads"][name] = {k: r[k] for k in ("metric", "value", "unit", "steps", "ms_per_step",
                                                           "dtype", "config", "roofline", "cpu_baseline", "fp32",
                                                           "backward") if k in r}
            torch.cuda.empty_cache()
            print(f"bench: {name} {r['value']} {r['unit']}", file=sys.stderr, flush=True)
    print(json.dumps(result), flush=True)


if __name__ == "__main__":
    main()
