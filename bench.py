#!/usr/bin/env python3
"""Benchmark of the DeepSeek-V3.2 quantized decode-attention hot path on one MI355X.

One step = one decode step of the path for a batch: lightning indexer (int8 index scores + top-2048) over
the paged index-K cache, then sparse flash attention over the selected rows of the int8 paged MLA cache,
chained (the indexer's output is the attention's top-k list).  Workload: batch 32, one query token per
sequence, every context 65536 tokens, 64 index heads x 128, 128 absorbed heads, 512 nope + 64 rope, pages
of 128 tokens.  Inputs are synthetic, resident in HBM before the timed region; three copies of the caches
are rotated so that no step finds its cache lines in the 256 MB last-level cache from the step before.

Prints ONE JSON line: whole-job decode tokens/s, the roofline object of the dominant kernel (duration from
HIP events recorded on the launch stream inside the library, second pass over the same steps), and the
CPU oracle timed on the host cores on a bounded sample of the same workload.
"""
import argparse
import ctypes
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
MFMA_BF16_PEAK_TFLOPS = 2500.0

def profile_traffic(name):
    """HBM bytes per launch (read + written) of every kernel in the table of profiles/<name>: rocprofv3 FETCH_SIZE and
    WRITE_SIZE per dispatch, each scaled by what the same counter reads for a plain elementwise kernel of known size
    (the file says how it was made; --calibrate-copy puts that kernel into a counter run).  The figures belong to the
    exact workload the file names and are reported for that workload only.  {} when the file is not there."""
    path = os.path.join(ROOT, "profiles", name)
    out, in_table = {}, False
    if not os.path.exists(path):
        return out
    for line in open(path):
        cols = line.split()
        if cols[:2] == ["kernel", "FETCH_SIZE"]:
            in_table = True
        elif in_table:
            if len(cols) < 5 or not cols[1].isdigit():
                break
            # columns: kernel, FETCH_SIZE KiB, read MB, WRITE_SIZE KiB, written MB; the kernel as bench.py names it
            out[cols[0].split("<")[0].replace("_paged", "")] = (float(cols[2]) + float(cols[4])) * 1e6
    return out


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    # (the first hundred or so steps after an idle period run 8-10 % slower than the steady state - clocks and caches
    # come up - so the defaults warm up for 100 steps and time 500; the whole default run still takes well under a minute
    # of GPU time)
    ap.add_argument("--steps", type=int, default=500)
    ap.add_argument("--warmup", type=int, default=100)
    ap.add_argument("--batch", type=int, default=32)
    ap.add_argument("--ctx", type=int, default=65536)
    ap.add_argument("--s1", type=int, default=1)
    ap.add_argument("--ctx-min", type=int, default=0,
                    help="v32 workload: draw every context length from U{ctx-min..ctx} (seeded) instead of ctx for all")
    ap.add_argument("--cpu-seqs", type=int, default=8, help="sequences of the workload timed on the CPU oracle")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--packed", action="store_true", help="use the packed 656-byte-row attention entry point")
    ap.add_argument("--fp32-scales", action="store_true",
                    help="indexer query / key scales as fp32 tensors (the default is fp16, the reference operator's signature)")
    ap.add_argument("--workload", choices=["v32", "gqa", "select_experts", "indexer_prolog", "mla_prolog", "mla_indexer_prolog", "decode_layer", "attention_pre_quant", "sfa_prefill", "paged_gather"], default="v32",
                    help="v32 (default): the headline DeepSeek-V3.2 indexer + sparse attention decode step; gqa: GLM-4.5 "
                         "paged GQA decode (batch 64, 96/8 heads, contexts U[4096, 32768]); select_experts: GLM-4.5 "
                         "router (8192 tokens x 160 experts); attention_pre_quant: GLM-4.5 fused attention prolog")
    ap.add_argument("--q-heads", type=int, default=12,
                    help="attention_pre_quant: query heads on this device (12 = the reference test's share of GLM-4.5's "
                         "96, with 1 key / value head; 96 = the whole model, 8 key / value heads)")
    ap.add_argument("--warm-weights", action="store_true",
                    help="prolog workloads: one copy of the weights, re-read every step (they then partly come out of "
                         "the 256 MB last-level cache); default: rotate enough copies to exceed it")
    ap.add_argument("--streams", type=int, default=1,
                    help="v32 workload: launch consecutive steps on this many HIP streams in turn (each with its own "
                         "outputs), the way a server keeps several micro-batches in flight; the default, 1, is the "
                         "headline measurement")
    ap.add_argument("--graph", action="store_true",
                    help="replay the step from HIP graphs (one per cache copy) instead of launching it eagerly")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="also launch one plain elementwise kernel that reads 256 MiB and writes 256 MiB, so that a "
                         "counter run of this command holds a dispatch of known HBM traffic to scale FETCH_SIZE / "
                         "WRITE_SIZE by")
    return ap.parse_args()


def make_workload(torch, dev, b, ctx, s1, nbuf, seed=0, ctx_min=0, idx_scale_dtype=None):
    g = torch.Generator(device=dev).manual_seed(seed)
    bs = 128
    sdt = idx_scale_dtype or torch.float16  # fp16: the reference operator's signature; fp32: --fp32-scales
    pages_per_seq = (ctx + bs - 1) // bs
    n_pages = b * pages_per_seq
    n_rows = n_pages * bs
    table = torch.randperm(n_pages, generator=g, device=dev).to(torch.int32).reshape(b, pages_per_seq).contiguous()
    t = b * s1
    sets = []
    for _ in range(nbuf):
        sets.append({
            "idx_k": torch.randint(-127, 128, (n_pages, bs, 1, 128), generator=g, device=dev, dtype=torch.int8),
            "idx_ks": (0.005 + 0.015 * torch.rand((n_pages, bs, 1), generator=g, device=dev)).to(sdt),
            "kn": torch.randint(-127, 128, (n_rows, 512), generator=g, device=dev, dtype=torch.int8),
            "kr": torch.randn((n_rows, 64), generator=g, device=dev).to(torch.bfloat16),
            "ks": (0.005 + 0.015 * torch.rand((n_rows, 4), generator=g, device=dev)).float(),
        })
    w = {
        "b": b, "s1": s1, "ctx": ctx, "bs": bs, "pages_per_seq": pages_per_seq, "table": table, "sets": sets,
        "idx_q": torch.randint(-127, 128, (t, 64, 128), generator=g, device=dev, dtype=torch.int8),
        "idx_qs": (0.005 + 0.015 * torch.rand((t, 64), generator=g, device=dev)).to(sdt),
        "idx_w": (torch.randn((t, 64), generator=g, device=dev) / 8).to(torch.float16),
        "q_nope": torch.randn((t * 128, 512), generator=g, device=dev).to(torch.bfloat16),
        "q_rope": torch.randn((t * 128, 64), generator=g, device=dev).to(torch.bfloat16),
        "act": (torch.randint(ctx_min, ctx + 1, (b,), generator=g, device=dev).to(torch.int32) if ctx_min
                else torch.full((b,), ctx, dtype=torch.int32, device=dev)),
        "topk_res": torch.zeros((t, 1, 2048), dtype=torch.int32, device=dev),
        "out": torch.zeros((b, s1, 128, 512), dtype=torch.bfloat16, device=dev),
    }
    return w


def read_kernel_times(lib):
    """us per launch of every library kernel timed since timing was enabled, less the offset of the event pairs (what
    a pair around an empty kernel reads beyond that kernel's own duration)."""
    import torch
    lib.pto_kernel_name.restype = ctypes.c_char_p
    off = ctypes.c_double(0)
    lib.pto_kernel_timing_overhead(ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), ctypes.byref(off))
    kernels, raw = {}, {}
    for kid in range(64):
        if not lib.pto_kernel_name(kid):
            break
        ms, n = ctypes.c_double(0), ctypes.c_uint64(0)
        lib.pto_kernel_timing_read(kid, ctypes.byref(ms), ctypes.byref(n))
        if n.value:
            name = lib.pto_kernel_name(kid).decode()
            raw[name] = ms.value * 1e3 / n.value
            kernels[name] = max(raw[name] - off.value * 1e3, 0.05)
    read_kernel_times.offset_us = off.value * 1e3
    read_kernel_times.raw_us = raw
    return kernels


def rotated(torch, tensors, weight_idx, args):
    """Copies of an operator's tensor list that differ in their weight tensors (the entries at weight_idx): enough of
    them to exceed the 256 MB last-level cache, so that a step finds none of its weights there - the case a layer stack
    is in.  One list when --warm-weights."""
    nbytes = sum(tensors[i].numel() * tensors[i].element_size() for i in weight_idx)
    copies = 1 if args.warm_weights else max(2, min(32, -(-320 * 2 ** 20 // max(nbytes, 1))))
    sets = [tensors]
    for _ in range(copies - 1):
        t = list(tensors)
        for i in weight_idx:
            t[i] = tensors[i].clone()
        sets.append(t)
    return sets


def timed(torch, lib, step, args, nsets=1):
    """ms per step over args.steps steps after args.warmup (eager launches, or - with --graph - replays of the step
    captured into HIP graphs, one per input set, which leaves the host's per-call work out), then a second eager pass
    with an event pair around every kernel."""
    eager = step
    if args.graph:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            eager(0)
        torch.cuda.current_stream().wait_stream(side)
        graphs = []
        for i in range(nsets):
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                eager(i)
            graphs.append(graph)

        def step(i):  # noqa: F811
            graphs[i % nsets].replay()
    for i in range(args.warmup):
        step(i)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i in range(args.steps):
        step(i)
    torch.cuda.synchronize()
    ms_per_step = (time.perf_counter() - t0) * 1e3 / args.steps
    lib.pto_kernel_timing_enable(1)
    for i in range(args.steps):
        eager(i)
    torch.cuda.synchronize()
    lib.pto_kernel_timing_enable(0)
    return ms_per_step, read_kernel_times(lib)


def bench_gqa(args, torch, lib, dev):
    """GLM-4.5 GQA decode: batch 64, 96 query heads over 8 KV heads, head dim 128, bf16, pages of 128 tokens, context
    lengths U[4096, 32768] (seed 0); q/k/v ~ N(0,1) (the rotary embedding is applied upstream of this operator and does
    not change its cost)."""
    from pypto_amd.glm_v4_5.glm_attention import IfaTileShapeConfig, attention
    b, nq, nkv, d, bs = 64, 96, 8, 128, 128
    g = torch.Generator(device=dev).manual_seed(0)
    act = torch.randint(4096, 32769, (b,), generator=g, device=dev, dtype=torch.int32)
    pages = ((act + bs - 1) // bs).tolist()
    n_pages = sum(pages)
    perm = torch.randperm(n_pages, generator=g, device=dev).to(torch.int32)
    table = torch.full((b, max(pages)), -1, dtype=torch.int32, device=dev)
    pos = 0
    for i, n in enumerate(pages):
        table[i, :n] = perm[pos:pos + n]
        pos += n
    k = torch.randn((n_pages, bs, nkv, d), generator=g, device=dev, dtype=torch.bfloat16)
    v = torch.randn((n_pages, bs, nkv, d), generator=g, device=dev, dtype=torch.bfloat16)
    q = torch.randn((b, nq, d), generator=g, device=dev, dtype=torch.bfloat16)
    out = torch.zeros_like(q)
    cfg = IfaTileShapeConfig()

    def step(i):
        attention(q, k, v, table, act, out, d ** -0.5, cfg)

    ms, kernels = timed(torch, lib, step, args)
    tokens = int(act.sum())
    work = tokens * nkv * d * 2 * 2 + 2 * b * nq * d * 2
    us = kernels["gqa_decode_kernel"]
    achieved = work / us / 1e3
    print(json.dumps({
        "metric": "decode tokens/sec + achieved HBM GB/s (% of peak), GLM-4.5 GQA decode b=64 ctx U[4K,32K]",
        "value": round(b / (ms * 1e-3), 1), "unit": "tokens/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(ms, 4), "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "bf16",
        "data": "synthetic",
        "config": {"workload": f"paged GQA decode attention, batch {b}, {nq}/{nkv} heads x {d}, bf16 KV, block {bs}, "
                               f"{tokens} cached tokens in total"},
        "roofline": {"kernel": "gqa_decode_kernel", "bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS,
                     "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": profile_traffic("bench_gqa_b64_hbm_traffic.txt").get("gqa_decode_kernel"),
                     "traffic_unit": "bytes per launch (rocprofv3 FETCH_SIZE + WRITE_SIZE, calibrated)",
                     "work_per_launch": work, "us_per_launch": round(us, 2)},
        "kernels": [{"kernel": n, "us": round(u, 2)} for n, u in kernels.items()], "cpu_baseline": None,
    }))


def bench_select_experts(args, torch, lib, dev):
    """GLM-4.5 router: 8192 tokens x 160 experts, bf16 logits ~ N(0,1), fp32 bias ~ N(0,0.1), 8 groups, top-4 groups,
    top-8 experts, renormalised, x 2.5."""
    from pypto_amd.glm_v4_5.glm_select_experts import select_experts
    t, ne, k = 8192, 160, 8
    g = torch.Generator(device=dev).manual_seed(0)
    logits = torch.randn((t, ne), generator=g, device=dev).to(torch.bfloat16)
    bias = 0.1 * torch.randn((ne,), generator=g, device=dev)
    w = torch.zeros((t, k), dtype=torch.float32, device=dev)
    ids = torch.zeros((t, k), dtype=torch.int32, device=dev)

    def step(i):
        select_experts(logits, k, True, 4, 8, bias, w, ids, routed_scaling_factor=2.5, fill_neg_inf=True)

    ms, kernels = timed(torch, lib, step, args)
    work = t * ne * 2 + ne * 4 + t * k * 8
    us = kernels["select_experts_kernel"]
    achieved = work / us / 1e3
    print(json.dumps({
        "metric": "routed tokens/sec, GLM-4.5 select_experts 8192 x 160", "value": round(t / (ms * 1e-3), 1),
        "unit": "tokens/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms, 4),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": f"grouped expert selection, {t} tokens x {ne} experts, 8 groups / top-4, top-{k}"},
        "roofline": {"kernel": "select_experts_kernel", "bound": "hbm", "achieved": round(achieved, 1),
                     "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": None,
                     "work_per_launch": work, "us_per_launch": round(us, 2),
                     "note": "3 MB of traffic: bound by launch and memory latency, not by a roofline"},
        "kernels": [{"kernel": n, "us": round(u, 2)} for n, u in kernels.items()], "cpu_baseline": None,
    }))


def _paged_rows(torch, dev, g, b, s2, bs):
    """A random page table for b sequences of s2 tokens and the flat cache row of each sequence's last token."""
    pages_per_seq = (s2 + bs - 1) // bs
    n_pages = b * pages_per_seq
    table = torch.randperm(n_pages, generator=g, device=dev).reshape(b, pages_per_seq)
    pos = s2 - 1
    rows = (table[:, pos // bs] * bs + pos % bs).to(torch.int64).contiguous()
    return n_pages, rows


def bench_indexer_prolog(args, torch, lib, dev):
    """DeepSeek-V3.2 lightning-indexer prolog at decode size: one new token for each of `batch` sequences, h 7168,
    q_lora_rank 1536, 64 index heads x 128, a 4K-token paged index cache per sequence; the reference generator's
    distributions (U[-1,1), int8 tensors uniform over their range)."""
    from pypto_amd.deepseek_v32_exp import lightning_indexer_prolog_quant_impl as impl
    t, n, h, r, d, bs = args.batch, 64, 7168, 1536, 128, 128
    g = torch.Generator(device=dev).manual_seed(0)
    bf = torch.bfloat16

    def uni(*shape):
        return torch.rand(shape, generator=g, device=dev) * 2 - 1

    def i8(*shape):
        return torch.randint(-128, 128, shape, generator=g, device=dev, dtype=torch.int8)

    # t == 8 is the configuration the reference quotes a latency for (batch 4, one extra MTP token each, 64K cache:
    # docs/zh/tutorials/debug/performance_case_quantindexerprolog.md:37,47 - 49 us on an Ascend NPU)
    published = t == 8
    n_pages, rows = _paged_rows(torch, dev, g, t, 65536 if published else 4096, bs)
    ang = torch.rand((t, 64), generator=g, device=dev) * 6.2831853
    k_cache, k_scale_cache = i8(n_pages, bs, 1, d), uni(n_pages, bs, 1, 1).to(torch.float16)
    tensors = [uni(t, h).to(bf), i8(t, r), uni(t, 1), i8(r, n * d), uni(n * d, 1), uni(h, d).to(bf), uni(h, n).to(bf),
               torch.ones(d, dtype=bf, device=dev), torch.zeros(d, dtype=bf, device=dev), torch.cos(ang).to(bf),
               torch.sin(ang).to(bf), uni(d, d).to(bf), uni(d, d).to(bf), k_cache, k_scale_cache, rows,
               torch.zeros((t, n, d), dtype=torch.int8, device=dev), torch.zeros((t, n, 1), dtype=torch.float16, device=dev),
               k_cache, k_scale_cache, torch.zeros((t, n), dtype=torch.float16, device=dev)]
    cfg, attrs = impl.IndexerPrologQuantConfigs(), impl.IndexerPrologQuantAttr()

    sets = rotated(torch, tensors, (3, 5, 6), args)

    def step(i):
        impl.lightning_indexer_prolog_quant(*sets[i % len(sets)], cfg, attrs)

    ms, kernels = timed(torch, lib, step, args, len(sets))
    work = r * n * d + h * (d + n) * 2 + t * (h * 2 + r + n * 130 + n * 2 + 130)
    total_us = sum(kernels.values())
    print(json.dumps({
        "metric": "prolog tokens/sec, DeepSeek-V3.2 lightning_indexer_prolog_quant decode", "value": round(t / (ms * 1e-3), 1),
        "unit": "tokens/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms, 4),
        "higher_is_better": True, "scaling": "weak",
        # published: 49 us per call of 8 tokens (other hardware) = 163265 tokens/s
        "vs_baseline": round((t / (ms * 1e-3)) / (8 / 49e-6), 3) if published else None,
        "dtype": "int8+bf16", "data": "synthetic", "launch": "hip graph replay" if args.graph else "eager",
        "config": {"workload": f"lightning indexer prolog, {t} tokens, h 7168, q_lora_rank 1536, 64 x 128 index heads"
                               + (", batch 4 x 2 tokens over a 64K-token paged cache (the reference's quoted case)" if published else "")
                               + f", weights rotated over {len(sets)} copies"},
        "roofline": {"kernel": f"prolog ({len(kernels)} kernels)", "bound": "hbm", "achieved": round(work / total_us / 1e3, 1),
                     "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": round(work / total_us / 1e3 / HBM_PEAK_GBS, 4),
                     "traffic": None, "work_per_launch": work, "us_per_launch": round(total_us, 2),
                     "note": "15 MB of weights read once: bound by launch and memory latency at decode sizes"},
        "kernels": [{"kernel": k, "us": round(u, 2)} for k, u in kernels.items()], "cpu_baseline": None,
    }))


def bench_mla_prolog(args, torch, lib, dev):
    """DeepSeek-V3.2 MLA prolog (int8 form) at decode size: one new token for each of `batch` sequences, h 7168,
    q_lora_rank 1536, 128 heads x (128 + 64), kv_lora_rank 512, a 4K-token paged cache per sequence; the reference
    generator's distributions (x U[-1,1), weights U[-0.1,0.1), w_uq_qr quantised per output channel, cos/sin
    U[-0.1,0.1))."""
    from pypto_amd.deepseek_v32_exp import mla_prolog_quant_impl as impl
    t, n, h, r, c, bs = args.batch, 128, 7168, 1536, 512, 128
    g = torch.Generator(device=dev).manual_seed(0)
    bf = torch.bfloat16

    def uni(lo, hi, *shape):
        return torch.rand(shape, generator=g, device=dev) * (hi - lo) + lo

    w = uni(-0.1, 0.1, r, n * 192)
    w_scale = (w.abs().amax(0, keepdim=True) / 127)
    w_uq_qr = torch.round(w / w_scale).to(torch.int8)
    n_pages, rows = _paged_rows(torch, dev, g, t, 4096, bs)
    kv = torch.randint(-127, 128, (n_pages, bs, 1, c), generator=g, device=dev, dtype=torch.int8)
    kr = uni(-1, 1, n_pages, bs, 1, 64).to(bf)
    ks = uni(0.001, 0.01, n_pages, bs, 1, 4)
    tensors = [uni(-1, 1, t, h).to(bf), uni(-0.1, 0.1, h, r).to(bf), w_uq_qr, w_scale.reshape(-1, 1).contiguous(),
               uni(-0.1, 0.1, n, 128, c).to(bf), uni(-0.1, 0.1, h, c + 64).to(bf), uni(-1, 1, r).to(bf), uni(-1, 1, c).to(bf),
               uni(-0.1, 0.1, t, 64).to(bf), uni(-0.1, 0.1, t, 64).to(bf), rows, kv, kr, ks,
               torch.zeros((t, r), dtype=torch.int8, device=dev), torch.zeros((t, 1), dtype=torch.float32, device=dev),
               torch.zeros((t, n, c), dtype=bf, device=dev), torch.zeros((t, n, 64), dtype=bf, device=dev), kv, kr, ks]
    cfg, rope = impl.MlaTileConfig(), impl.RopeTileShapeConfig([32, 64], [32, 32, 128], [16, 128, 128, 128])

    sets = rotated(torch, tensors, (1, 2, 4, 5), args)

    def step(i):
        impl.mla_prolog_quant_d(*sets[i % len(sets)], 1e-5, 1e-5, "PA_BSND", cfg, rope)

    ms, kernels = timed(torch, lib, step, args, len(sets))
    # weights once, plus per token: x, q_norm + scale, q_nope, q_rope, the cache row
    work = h * r * 2 + r * n * 192 + n * 192 * 4 + n * 128 * c * 2 + h * (c + 64) * 2 + \
        t * (h * 2 + r + 4 + n * c * 2 + n * 64 * 2 + c + 16 + 128)
    total_us = sum(kernels.values())
    print(json.dumps({
        "metric": "prolog tokens/sec, DeepSeek-V3.2 mla_prolog_quant decode", "value": round(t / (ms * 1e-3), 1),
        "unit": "tokens/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms, 4),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "int8+bf16", "data": "synthetic", "launch": "hip graph replay" if args.graph else "eager",
        "config": {"workload": f"MLA prolog (int8 form), {t} tokens, h 7168, q_lora_rank 1536, 128 heads x 192, "
                               f"kv_lora_rank 512, weights rotated over {len(sets)} copies"},
        "roofline": {"kernel": f"mla prolog ({len(kernels)} kernels)", "bound": "hbm", "achieved": round(work / total_us / 1e3, 1),
                     "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": round(work / total_us / 1e3 / HBM_PEAK_GBS, 4),
                     "traffic": None, "work_per_launch": work, "us_per_launch": round(total_us, 2),
                     "note": "85 MB of weights read once per call"},
        "kernels": [{"kernel": k, "us": round(u, 2)} for k, u in kernels.items()], "cpu_baseline": None,
    }))


def bench_mla_indexer_prolog(args, torch, lib, dev):
    """DeepSeek-V3.2 fused MLA + lightning-indexer prolog at decode size: the two workloads above in one call (shared
    token_x, cos, sin, cache_index; q_norm handed over inside the workspace)."""
    from pypto_amd.deepseek_v32_exp import mla_indexer_prolog_quant_impl as impl
    t, n, ni, h, r, c, d, bs = args.batch, 128, 64, 7168, 1536, 512, 128, 128
    g = torch.Generator(device=dev).manual_seed(0)
    bf = torch.bfloat16

    def uni(lo, hi, *shape):
        return torch.rand(shape, generator=g, device=dev) * (hi - lo) + lo

    def i8(*shape):
        return torch.randint(-128, 128, shape, generator=g, device=dev, dtype=torch.int8)

    w = uni(-0.1, 0.1, r, n * 192)
    w_scale = (w.abs().amax(0, keepdim=True) / 127)
    n_pages, rows = _paged_rows(torch, dev, g, t, 4096, bs)
    kv = torch.randint(-127, 128, (n_pages, bs, 1, c), generator=g, device=dev, dtype=torch.int8)
    kr, ks = uni(-1, 1, n_pages, bs, 1, 64).to(bf), uni(0.001, 0.01, n_pages, bs, 1, 4)
    ik, iks = i8(n_pages, bs, 1, d), uni(-1, 1, n_pages, bs, 1, 1).to(torch.float16)
    tensors = [uni(-1, 1, t, h).to(bf), uni(-0.1, 0.1, h, r).to(bf), torch.round(w / w_scale).to(torch.int8),
               w_scale.reshape(-1, 1).contiguous(), uni(-0.1, 0.1, n, 128, c).to(bf), uni(-0.1, 0.1, h, c + 64).to(bf),
               uni(-1, 1, r).to(bf), uni(-1, 1, c).to(bf), uni(-0.1, 0.1, t, 64).to(bf), uni(-0.1, 0.1, t, 64).to(bf), rows,
               kv, kr, ks,
               i8(r, ni * d), uni(-1, 1, ni * d, 1), uni(-1, 1, h, d).to(bf), uni(-1, 1, h, ni).to(bf),
               torch.ones(d, dtype=bf, device=dev), torch.zeros(d, dtype=bf, device=dev), uni(-1, 1, d, d).to(bf),
               uni(-1, 1, d, d).to(bf), ik, iks,
               torch.zeros((t, n, c), dtype=bf, device=dev), torch.zeros((t, n, 64), dtype=bf, device=dev), kv, kr, ks,
               torch.zeros((t, ni, d), dtype=torch.int8, device=dev), torch.zeros((t, ni, 1), dtype=torch.float16, device=dev),
               ik, iks, torch.zeros((t, ni), dtype=torch.float16, device=dev)]
    scal = (1e-5, 1e-5, "PA_BSND", impl.MlaTileConfig(), impl.IndexerPrologQuantAttr(), impl.IndexerPrologQuantConfigs(),
            impl.RopeTileShapeConfig([32, 64], [32, 32, 128], [16, 128, 128, 128]))

    sets = rotated(torch, tensors, (1, 2, 4, 5, 14, 16, 17), args)

    def step(i):
        impl.mla_indexer_prolog_quant_d(*sets[i % len(sets)], *scal)

    ms, kernels = timed(torch, lib, step, args, len(sets))
    work = h * r * 2 + r * n * 192 + n * 192 * 4 + n * 128 * c * 2 + h * (c + 64) * 2 + r * ni * d + h * (d + ni) * 2 + \
        t * (h * 2 + n * c * 2 + n * 64 * 2 + c + 16 + 128 + ni * 130 + ni * 2 + 130)
    total_us = sum(kernels.values())
    print(json.dumps({
        "metric": "prolog tokens/sec, DeepSeek-V3.2 mla_indexer_prolog_quant decode", "value": round(t / (ms * 1e-3), 1),
        "unit": "tokens/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms, 4),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "int8+bf16", "data": "synthetic", "launch": "hip graph replay" if args.graph else "eager",
        "config": {"workload": f"fused MLA + lightning-indexer prolog, {t} tokens, h 7168, q_lora_rank 1536, 128 heads x 192, "
                               f"kv_lora_rank 512, 64 x 128 index heads, weights rotated over {len(sets)} copies"},
        "roofline": {"kernel": f"fused prolog ({len(kernels)} kernels)", "bound": "hbm", "achieved": round(work / total_us / 1e3, 1),
                     "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": round(work / total_us / 1e3 / HBM_PEAK_GBS, 4),
                     "traffic": None, "work_per_launch": work, "us_per_launch": round(total_us, 2),
                     "note": "100 MB of weights read once per call"},
        "kernels": [{"kernel": k, "us": round(u, 2)} for k, u in kernels.items()], "cpu_baseline": None,
    }))


def bench_attention_pre_quant(args, torch, lib, dev):
    """GLM-4.5 attention_pre_quant at decode size: `batch` tokens, hidden 5120, `q-heads` query heads and q-heads / 12
    key / value heads of 128, rotary on 64 dims (the reference test's shape at 8 tokens and 12 heads:
    models/glm_v4_5/glm_attention_pre_quant.py:510-519); zero-mean activations, a quantisation scale that spreads the
    normalised row over the int8 range, weights uniform over int8."""
    from pypto_amd.glm_v4_5 import glm_attention_pre_quant as impl
    t, h, d, half = args.batch, 5120, 128, 32
    qh = args.q_heads
    kvh = max(qh // 12, 1)
    n_out = (qh + 2 * kvh) * d
    g = torch.Generator(device=dev).manual_seed(0)
    bf = torch.bfloat16

    def randn(*shape):
        return torch.randn(shape, generator=g, device=dev)

    def rand(*shape):
        return torch.rand(shape, generator=g, device=dev)

    ang = rand(t, 1, half) * 6.2831853
    tensors = [randn(t, h).to(bf), randn(t, h).to(bf), (1 + 0.1 * randn(h)).to(bf), (0.05 * randn(h)).to(bf),
               (30 + 10 * rand(h)).to(bf), torch.round(4 * randn(h)).to(bf),
               torch.randint(-128, 128, (h, n_out), generator=g, device=dev, dtype=torch.int8),
               torch.randint(-128, 128, (n_out,), generator=g, device=dev, dtype=torch.int32),
               1e-4 * (0.5 + rand(n_out)), (1 + 0.1 * randn(d)).to(bf), (0.05 * randn(d)).to(bf),
               (1 + 0.1 * randn(d)).to(bf), (0.05 * randn(d)).to(bf), torch.cos(ang).to(bf), torch.sin(ang).to(bf),
               torch.zeros((t, qh * d), dtype=bf, device=dev), torch.zeros((t, kvh * d), dtype=bf, device=dev),
               torch.zeros((t, kvh * d), dtype=bf, device=dev), torch.zeros((t, h), dtype=bf, device=dev)]
    sets = rotated(torch, tensors, (6,), args)

    def step(i):
        impl.attention_pre_quant(*sets[i % len(sets)])

    ms, kernels = timed(torch, lib, step, args, len(sets))
    # read once: the weight, the two activation rows, the per-channel vectors; written: the four outputs
    work = h * n_out + n_out * 8 + h * 8 + t * (h * 2 * 3 + n_out * 2 + half * 4)
    total_us = sum(kernels.values())
    print(json.dumps({
        "metric": "prolog tokens/sec, GLM-4.5 attention_pre_quant decode", "value": round(t / (ms * 1e-3), 1),
        "unit": "tokens/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms, 4),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "int8+bf16", "data": "synthetic", "launch": "hip graph replay" if args.graph else "eager",
        "config": {"workload": f"GLM-4.5 attention_pre_quant, {t} tokens, hidden 5120, {qh} + {kvh} + {kvh} heads of 128, "
                               f"rotary 64, weights rotated over {len(sets)} copies"},
        "roofline": {"kernel": f"attention_pre_quant ({len(kernels)} kernels)", "bound": "hbm", "achieved": round(work / total_us / 1e3, 1),
                     "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": round(work / total_us / 1e3 / HBM_PEAK_GBS, 4),
                     "traffic": None, "work_per_launch": work, "us_per_launch": round(total_us, 2),
                     "note": f"{h * n_out / 1e6:.1f} MB of weights read once: bound by launch and memory latency at decode sizes"},
        "kernels": [{"kernel": k, "us": round(u, 2)} for k, u in kernels.items()], "cpu_baseline": None,
    }))


def bench_sfa_prefill(args, torch, lib, dev):
    """The prefill entry of sparse flash attention at the reference's prefill case (sfa_bf16_b1_s256_seq64K_int8_p,
    models/deepseek_v32_exp/deepseekv32_sparse_flash_attention_quant.py:498): one sequence of `ctx` cached tokens, 256
    query tokens (`--s1`), 128 heads, every query token with its own 2048 selected rows (random, distinct)."""
    from pypto_amd.deepseek_v32_exp.sparse_flash_attention_quant_impl import SaTileShapeConfig, sparse_flash_attention_quant_p
    s1 = args.s1 if args.s1 > 1 else 256
    w = make_workload(torch, dev, 1, args.ctx, s1, 1)
    g = torch.Generator(device=dev).manual_seed(1)
    topk = torch.stack([torch.randperm(args.ctx, generator=g, device=dev)[:2048] for _ in range(s1)]).to(torch.int32).contiguous()
    c = w["sets"][0]
    cfg = SaTileShapeConfig()
    scale = 192 ** -0.5

    def step(i):
        sparse_flash_attention_quant_p(w["q_nope"], w["q_rope"], c["kn"], c["kr"], c["ks"], topk, w["table"], w["act"],
                                       w["out"], 128, 1, scale, 2048, 128, w["pages_per_seq"], cfg)

    ms, kernels = timed(torch, lib, step, args)
    flops = s1 * 2048 * 128 * (2 * 576 + 2 * 512)
    us = kernels.get("sfa_decode_kernel", 0.0)
    print(json.dumps({
        "metric": "prefill query tokens/sec, V3.2 sparse flash attention", "value": round(s1 / (ms * 1e-3), 1), "unit": "tokens/s",
        "n_gpus": 1, "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms, 4), "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "int8+bf16", "data": "synthetic",
        "launch": "hip graph replay" if args.graph else "eager",
        "config": {"workload": f"sparse flash attention, prefill entry, 1 sequence of {args.ctx} cached tokens, {s1} query tokens, "
                               f"128 heads, top-2048 per query token, int8 paged MLA cache"},
        "roofline": {"kernel": "sfa_decode_kernel", "bound": "mfma", "achieved": round(flops / us / 1e6, 1) if us else None,
                     "peak": 2500.0, "unit": "TFLOP/s", "frac": round(flops / us / 1e6 / 2500.0, 4) if us else None,
                     "traffic": None, "work_per_launch": flops, "us_per_launch": round(us, 2)},
        "kernels": [{"kernel": k, "us": round(u, 2)} for k, u in kernels.items()], "cpu_baseline": None,
    }))


def bench_paged_gather(args, torch, lib, dev):
    """Standalone paged gather at the attention's own gather shape: batch 32 sequences of --ctx cached tokens in pages
    of 128, packed 656-byte cache rows (512 int8 + 64 bf16 + 4 fp32), 2048 random distinct logical indices per sequence
    -> 65536 rows of 656 bytes.  Three caches are rotated so that no step finds its rows in the last-level cache."""
    from pypto_amd.experimental import paged_gather
    b, k, bs, hidden = args.batch, 2048, 128, 656
    g = torch.Generator(device=dev).manual_seed(0)
    per = -(-args.ctx // bs)
    table = torch.randperm(b * per, generator=g, device=dev).to(torch.int32).reshape(b, per)
    idx = torch.stack([torch.randperm(args.ctx, generator=g, device=dev)[:k] for _ in range(b)]).to(torch.int32)
    caches = [torch.randint(-127, 128, (b * per * bs, hidden), generator=g, device=dev, dtype=torch.int8)
              for _ in range(3)]
    out = torch.empty((b * k, hidden), dtype=torch.int8, device=dev)

    def step(i):
        paged_gather(caches[i % len(caches)], idx, table, bs, out=out)

    ms, kernels = timed(torch, lib, step, args, nsets=len(caches))
    rows = b * k
    work = rows * (2 * hidden + 4)
    us = kernels["paged_gather_kernel"]
    achieved = work / us / 1e3
    cpu = None
    if not args.no_cpu:
        from oracle import paged
        src, ix, tb = caches[0][:per * bs * 4].cpu(), idx[:4].cpu(), (table[:4] % (per * 4)).cpu()
        paged.paged_gather(src, ix[0], tb[0], bs)
        t0, n = time.perf_counter(), 0
        while time.perf_counter() - t0 < 10.0:
            for i in range(4):
                paged.paged_gather(src, ix[i], tb[i], bs)
            n += 4 * k
        cpu = {"value": round(n / (time.perf_counter() - t0), 1), "unit": "rows/s", "cores": torch.get_num_threads(),
               "kind": "port", "sample": "4 sequences' 2048-row gathers out of a 4-sequence cache of the same row "
                                         "width, repeated for ten seconds after an untimed pass"}
    print(json.dumps({
        "metric": "gathered cache rows/sec + achieved HBM GB/s (% of peak), paged gather of 656-byte rows",
        "value": round(rows / (ms * 1e-3), 1), "unit": "rows/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(ms, 4), "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "u8",
        "data": "synthetic",
        "config": {"workload": f"paged gather, batch {b} x {k} logical indices over {args.ctx} cached tokens each, "
                               f"pages of {bs}, rows of {hidden} bytes"},
        "roofline": {"kernel": "paged_gather_kernel", "bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS,
                     "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBS, 4),
                     "traffic": profile_traffic("bench_paged_gather_b32_k2048_hbm_traffic.txt").get("paged_gather_kernel") if (b, args.ctx) == (32, 65536) else None,
                     "traffic_unit": "bytes per launch (rocprofv3 FETCH_SIZE + WRITE_SIZE, calibrated)",
                     "work_per_launch": work, "us_per_launch": round(us, 2)},
        "kernels": [{"kernel": n, "us": round(u, 2)} for n, u in kernels.items()], "cpu_baseline": cpu,
    }))


def bench_decode_layer(args, torch, lib, dev):
    """The attention front end of one DeepSeek-V3.2 decode layer as three chained calls on shared buffers: the fused MLA +
    indexer prolog writes the query tensors and the new cache rows (the last position of every sequence), the lightning
    indexer selects 2048 rows per token, sparse flash attention reads them.  Shapes of the default workload (batch 32, one
    token each, every context 65536) and of the prolog workloads."""
    from pypto_amd.deepseek_v32_exp import mla_indexer_prolog_quant_impl as pimpl
    from pypto_amd.deepseek_v32_exp.lightning_indexer_quant_impl import LightningIndexerConfigs, lightning_indexer_decode
    from pypto_amd.deepseek_v32_exp.sparse_flash_attention_quant_impl import (SaTileShapeConfig,
                                                                              sparse_flash_attention_quant_d)
    b, ctx, s1 = args.batch, args.ctx, 1
    t, n, ni, h, r, c, d, bs = b, 128, 64, 7168, 1536, 512, 128, 128
    w = make_workload(torch, dev, b, ctx, s1, 1)
    cs = w["sets"][0]
    g = torch.Generator(device=dev).manual_seed(1)
    bf = torch.bfloat16

    def uni(lo, hi, *shape):
        return torch.rand(shape, generator=g, device=dev) * (hi - lo) + lo

    wq = uni(-0.1, 0.1, r, n * 192)
    wq_scale = (wq.abs().amax(0, keepdim=True) / 127)
    pos = ctx - 1
    rows = (w["table"][:, pos // bs].to(torch.int64) * bs + pos % bs).contiguous()
    n_pages = w["table"].numel()
    kv, kr, ks = cs["kn"].view(n_pages, bs, 1, c), cs["kr"].view(n_pages, bs, 1, 64), cs["ks"].view(n_pages, bs, 1, 4)
    ik, iks = cs["idx_k"], cs["idx_ks"].view(n_pages, bs, 1, 1)
    q_nope, q_rope = w["q_nope"].view(t, n, c), w["q_rope"].view(t, n, 64)
    idx_q, idx_qs, idx_w = w["idx_q"], w["idx_qs"].view(t, ni, 1), w["idx_w"]
    ang = torch.rand((t, 64), generator=g, device=dev) * 6.2831853
    prolog = [uni(-1, 1, t, h).to(bf), uni(-0.1, 0.1, h, r).to(bf), torch.round(wq / wq_scale).to(torch.int8),
              wq_scale.reshape(-1, 1).contiguous(), uni(-0.1, 0.1, n, 128, c).to(bf), uni(-0.1, 0.1, h, c + 64).to(bf),
              uni(-1, 1, r).to(bf), uni(-1, 1, c).to(bf), torch.cos(ang).to(bf), torch.sin(ang).to(bf), rows, kv, kr, ks,
              torch.randint(-128, 128, (r, ni * d), generator=g, device=dev, dtype=torch.int8), uni(0.001, 0.01, ni * d, 1),
              uni(-0.1, 0.1, h, d).to(bf), uni(-0.1, 0.1, h, ni).to(bf), torch.ones(d, dtype=bf, device=dev),
              torch.zeros(d, dtype=bf, device=dev), uni(-1, 1, d, d).to(bf) / 11.3, uni(-1, 1, d, d).to(bf) / 11.3, ik, iks,
              q_nope, q_rope, kv, kr, ks, idx_q, idx_qs, ik, iks, idx_w]
    scal = (1e-5, 1e-5, "PA_BSND", pimpl.MlaTileConfig(), pimpl.IndexerPrologQuantAttr(), pimpl.IndexerPrologQuantConfigs(),
            pimpl.RopeTileShapeConfig([32, 64], [32, 32, 128], [16, 128, 128, 128]))
    cfg, tile, unroll = LightningIndexerConfigs(), SaTileShapeConfig(), [128, 64, 32, 16, 8, 4, 1]
    scale = 192 ** -0.5

    def step(i):
        pimpl.mla_indexer_prolog_quant_d(*prolog, *scal)
        lightning_indexer_decode(idx_q, w["idx_qs"], ik, cs["idx_ks"], idx_w, w["act"], w["table"], w["topk_res"], unroll,
                                 cfg, 2048)
        sparse_flash_attention_quant_d(w["q_nope"], w["q_rope"], cs["kn"], cs["kr"], cs["ks"], w["topk_res"].view(t, 2048),
                                       w["table"], w["act"], w["out"], 128, 1, scale, 2048, 128, w["pages_per_seq"], tile)

    ms, kernels = timed(torch, lib, step, args)
    assert torch.isfinite(w["out"].float()).all()
    print(json.dumps({
        "metric": "decode tokens/sec, DeepSeek-V3.2 attention front end (fused prolog + indexer + SFA) b=32 ctx=64K",
        "value": round(t / (ms * 1e-3), 1), "unit": "tokens/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(ms, 4), "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "int8+bf16", "data": "synthetic", "launch": "hip graph replay" if args.graph else "eager",
        "config": {"workload": f"fused MLA + indexer prolog -> lightning indexer top-2048 -> sparse flash attention, batch {b}, "
                               f"1 query token per sequence, context {ctx}, model sizes"},
        "roofline": None, "kernels": [{"kernel": k, "us": round(u, 2)} for k, u in kernels.items()], "cpu_baseline": None,
    }))


def main():
    args = parse()
    if args.gpus != 1:
        print(f"bench.py measures one GPU only (this build has no multi-GPU path); got --gpus {args.gpus}",
              file=sys.stderr)
        sys.exit(2)
    import torch
    from pypto_amd import _runtime
    from pypto_amd.deepseek_v32_exp.lightning_indexer_quant_impl import (LightningIndexerConfigs,
                                                                         lightning_indexer_decode)
    from pypto_amd.deepseek_v32_exp.sparse_attention_antiquant_impl import sparse_attention_antiquant_d
    from pypto_amd.deepseek_v32_exp.sparse_flash_attention_quant_impl import (SaTileShapeConfig,
                                                                              sparse_flash_attention_quant_d)
    if not torch.cuda.is_available():
        print("bench.py needs a GPU", file=sys.stderr)
        sys.exit(2)
    lib = _runtime.load_library()
    dev = torch.device("cuda:0")
    if args.workload == "gqa":
        return bench_gqa(args, torch, lib, dev)
    if args.workload == "select_experts":
        return bench_select_experts(args, torch, lib, dev)
    if args.workload == "indexer_prolog":
        return bench_indexer_prolog(args, torch, lib, dev)
    if args.workload == "mla_prolog":
        return bench_mla_prolog(args, torch, lib, dev)
    if args.workload == "mla_indexer_prolog":
        return bench_mla_indexer_prolog(args, torch, lib, dev)
    if args.workload == "decode_layer":
        return bench_decode_layer(args, torch, lib, dev)
    if args.workload == "attention_pre_quant":
        return bench_attention_pre_quant(args, torch, lib, dev)
    if args.workload == "paged_gather":
        return bench_paged_gather(args, torch, lib, dev)
    if args.workload == "sfa_prefill":
        return bench_sfa_prefill(args, torch, lib, dev)
    b, ctx, s1 = args.batch, args.ctx, args.s1
    scale = 192 ** -0.5
    nbuf = 3
    w = make_workload(torch, dev, b, ctx, s1, nbuf, ctx_min=args.ctx_min,
                      idx_scale_dtype=torch.float32 if args.fp32_scales else None)
    ks_bytes = 4 if args.fp32_scales else 2
    lengths = w["act"].tolist()
    if args.packed:
        for s in w["sets"]:
            rows = torch.empty((s["kn"].shape[0], 656), dtype=torch.int8, device=dev)
            rows[:, :512] = s["kn"]
            rows[:, 512:640] = s["kr"].view(torch.int8)
            rows[:, 640:] = s["ks"].view(torch.int8)
            s["rows"] = rows
    cfg, tile = LightningIndexerConfigs(), SaTileShapeConfig()
    unroll = [128, 64, 32, 16, 8, 4, 1]

    def one_step(i, topk_res, out):
        s = w["sets"][i % nbuf]
        lightning_indexer_decode(w["idx_q"], w["idx_qs"], s["idx_k"], s["idx_ks"], w["idx_w"], w["act"], w["table"],
                                 topk_res, unroll, cfg, 2048)
        tk = topk_res.view(b * s1, 2048)
        if args.packed:
            sparse_attention_antiquant_d(w["q_nope"], w["q_rope"], s["rows"], tk, w["table"], w["act"],
                                         out.view(b * s1 * 128, 512), 128, 1, scale, 2048, 128,
                                         w["pages_per_seq"], tile)
        else:
            sparse_flash_attention_quant_d(w["q_nope"], w["q_rope"], s["kn"], s["kr"], s["ks"], tk, w["table"],
                                           w["act"], out, 128, 1, scale, 2048, 128, w["pages_per_seq"], tile)

    def step(i):
        one_step(i, w["topk_res"], w["out"])

    eager_step = step
    if args.streams > 1:
        if args.graph:
            print("--streams and --graph do not combine", file=sys.stderr)
            sys.exit(2)
        # consecutive steps on different streams, each stream with outputs of its own (the inputs are only read)
        lanes = [(torch.cuda.Stream(), torch.empty_like(w["topk_res"]), torch.empty_like(w["out"])) for _ in range(args.streams)]
        torch.cuda.synchronize()

        def step(i):  # noqa: F811
            st, topk_res, out = lanes[i % args.streams]
            with torch.cuda.stream(st):
                one_step(i, topk_res, out)
    if args.graph:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for i in range(nbuf):
                eager_step(i)
        torch.cuda.current_stream().wait_stream(side)
        graphs = []
        for i in range(nbuf):
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                eager_step(i)
            graphs.append(g)

        def step(i):  # noqa: F811 - the timed loop below replays the captured steps
            graphs[i % nbuf].replay()

    if args.calibrate_copy:
        src = torch.ones(64 << 20, dtype=torch.int32, device=dev)
        dst = torch.empty_like(src)
        torch.add(src, 1, out=dst)
        torch.cuda.synchronize()
        del src, dst

    for i in range(args.warmup):
        step(i)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i in range(args.steps):
        step(i)
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    ms_per_step = (t1 - t0) * 1e3 / args.steps
    tokens_per_s = b * s1 / (ms_per_step * 1e-3)

    # the same steps once more, one event pair per step on the launch stream (torch's current stream is the stream the
    # operators launch on): the spread of a single step, next to the mean above
    n_single = max(args.steps, 100)
    evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(n_single)]
    for i, (e0, e1) in enumerate(evs):
        e0.record()
        eager_step(i)
        e1.record()
    torch.cuda.synchronize()
    single = sorted(e0.elapsed_time(e1) * 1e3 for e0, e1 in evs)
    step_us = {"median": round(single[len(single) // 2], 1), "p10": round(single[len(single) // 10], 1),
               "p90": round(single[len(single) * 9 // 10], 1), "n": n_single,
               "note": "one event pair per step; includes about 4 us of the pair's own offset"}

    # second pass over the same steps with an event pair around every kernel launch
    lib.pto_kernel_timing_enable(1)
    for i in range(args.steps):
        eager_step(i)
    torch.cuda.synchronize()
    lib.pto_kernel_timing_enable(0)
    kernels = read_kernel_times(lib)

    t = b * s1
    # algorithmic traffic / work per launch, summed over the sequences' lengths
    score_bytes = sum(L * 128 + L * ks_bytes + (L + 127) // 128 * 4 for L in lengths) + t * (64 * 128 + 64 * ks_bytes + 64 * 2)
    topk_bytes = t * 2048 * 4
    curs = [min(max(L - s1 + 1 + i, 0), 2048) for L in lengths for i in range(s1)]
    sfa_bytes = sum(cur * 656 for cur in curs) + t * (128 * 576 * 2 + 128 * 512 * 2 + 2048 * 4)
    sfa_flops = sum(278528 * cur for cur in curs)
    select_bytes = s1 * sum(lengths) * 4
    info = {
        "indexer_score_kernel": {"bound": "hbm", "work": score_bytes, "peak": HBM_PEAK_GBS, "unit": "GB/s"},
        "indexer_topk_kernel": {"bound": "hbm", "work": topk_bytes, "peak": HBM_PEAK_GBS, "unit": "GB/s"},
        "sfa_decode_kernel": {"bound": "mfma", "work": sfa_flops, "peak": MFMA_BF16_PEAK_TFLOPS, "unit": "TFLOP/s"},
        "sfa_combine_kernel": {"bound": "hbm", "work": t * 128 * 512 * 2, "peak": HBM_PEAK_GBS, "unit": "GB/s"},
        "indexer_select_kernel": {"bound": "hbm", "work": select_bytes, "peak": HBM_PEAK_GBS, "unit": "GB/s"},
        "indexer_zero_kernel": {"bound": "hbm", "work": t * 2052 * 4, "peak": HBM_PEAK_GBS, "unit": "GB/s"},
    }
    per_kernel = []
    for name, us in kernels.items():
        k = info[name]
        div = 1e3 if k["unit"] == "GB/s" else 1e6  # bytes/us -> GB/s is /1e3 ; flop/us -> TFLOP/s is /1e6
        achieved = k["work"] / us / div
        per_kernel.append({"kernel": name, "us": round(us, 2), "us_event_pair": round(read_kernel_times.raw_us[name], 2),
                           "bound": k["bound"], "achieved": round(achieved, 2), "peak": k["peak"], "unit": k["unit"],
                           "frac": round(achieved / k["peak"], 4)})
    per_kernel.sort(key=lambda r: -r["us"])
    dom = per_kernel[0]
    default_workload = (b, ctx, s1, args.packed, args.ctx_min) == (32, 65536, 1, False, 0)
    roofline = {"kernel": dom["kernel"], "bound": dom["bound"], "achieved": dom["achieved"], "peak": dom["peak"],
                "unit": dom["unit"], "frac": dom["frac"],
                "traffic": profile_traffic("bench_b32_ctx64k_hbm_traffic.txt").get(dom["kernel"]) if default_workload else None,
                "traffic_unit": "bytes per launch (rocprofv3 FETCH_SIZE + WRITE_SIZE, calibrated)",
                "work_per_launch": info[dom["kernel"]]["work"], "us_per_launch": dom["us"]}
    sfa_row = next((r for r in per_kernel if r["kernel"] == "sfa_decode_kernel"), None)
    if sfa_row:
        sfa_row["hbm_gbs"] = round(sfa_bytes / sfa_row["us"] / 1e3, 1)
    score_row = next((r for r in per_kernel if r["kernel"] == "indexer_score_kernel"), None)
    if score_row:
        # the score kernel is bound by the cache stream; its int8 MFMA rate (2 x 64 heads x 128 dims per key and query
        # token) is reported beside it
        int8_ops = s1 * sum(lengths) * 2 * 64 * 128
        score_row["int8_mfma_tops"] = round(int8_ops / score_row["us"] / 1e6, 1)
        score_row["int8_mfma_frac"] = round(int8_ops / score_row["us"] / 1e6 / 5000.0, 4)

    # the two stages of the step against their rooflines: the indexer (all of its kernels) streams the index cache
    # once; attention (decode + split merge) is the bf16 contraction.  The reference labels four sub-stages of its
    # attention tile loop (Sa_V0 gather and dequantisation, Sa_C1 scores, Sa_V1 softmax, Sa_C2 values:
    # sparse_flash_attention_quant_impl.py:147,179,261,271); here all four run inside sfa_decode_kernel.
    idx_us = sum(us for n, us in kernels.items() if n.startswith("indexer_"))
    sfa_us = sum(us for n, us in kernels.items() if n.startswith("sfa_"))
    stages = [
        {"name": "indexer", "kernels": [n for n in kernels if n.startswith("indexer_")], "us": round(idx_us, 2),
         "bound": "hbm", "achieved": round((score_bytes + topk_bytes) / idx_us / 1e3, 1), "peak": HBM_PEAK_GBS,
         "unit": "GB/s", "frac": round((score_bytes + topk_bytes) / idx_us / 1e3 / HBM_PEAK_GBS, 4)},
        {"name": "sparse flash attention (Sa_V0 + Sa_C1 + Sa_V1 + Sa_C2, split merge)",
         "kernels": [n for n in kernels if n.startswith("sfa_")], "us": round(sfa_us, 2), "bound": "mfma",
         "achieved": round(sfa_flops / sfa_us / 1e6, 1), "peak": MFMA_BF16_PEAK_TFLOPS, "unit": "TFLOP/s",
         "frac": round(sfa_flops / sfa_us / 1e6 / MFMA_BF16_PEAK_TFLOPS, 4)},
    ]

    cpu_baseline, cpu_as_written = None, None
    if not args.no_cpu:
        cpu_baseline = time_cpu_oracle(torch, w, min(args.cpu_seqs, b), scale)
        cpu_as_written = time_cpu_as_written(torch, w, scale)

    print(json.dumps({
        "metric": "decode tokens/sec + achieved HBM GB/s (% of peak), V3.2 SFA b=32 ctx=64K",
        "value": round(tokens_per_s, 1), "unit": "tokens/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(ms_per_step, 4), "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "int8+bf16",
        "data": "synthetic", "launch": "hip graph replay" if args.graph else "eager" if args.streams == 1 else f"eager, steps in turn on {args.streams} streams",
        "config": {"workload": f"lightning indexer top-2048 + sparse flash attention decode, batch {b}, "
                               f"s1 {s1}, ctx {f'U[{args.ctx_min}, {ctx}]' if args.ctx_min else ctx}, 64x128 int8 index heads, 128 heads x (512 nope + 64 rope), "
                               f"int8 paged MLA cache, block 128, {'packed 656 B rows' if args.packed else 'three cache tensors'}"},
        "roofline": roofline, "kernels": per_kernel, "event_pair_offset_us": round(read_kernel_times.offset_us, 2),
        "step_us": step_us, "stages": stages, "cpu_baseline": cpu_baseline, "cpu_baseline_as_written": cpu_as_written,
    }))


def time_cpu_oracle(torch, w, n_seq, scale):
    """Oracle (vectorised torch restatement of the reference's CPU golden) timed on the first n_seq sequences
    of the same inputs (cache copy 0)."""
    from oracle import indexer as oi
    from oracle import sfa as osfa
    s1, ctx = w["s1"], w["ctx"]
    s = w["sets"][0]
    host = {k: v.cpu() for k, v in s.items() if k != "rows"}
    table = w["table"][:n_seq].cpu()
    act = w["act"][:n_seq].tolist()
    t = n_seq * s1
    idx_q, idx_qs, idx_w = w["idx_q"][:t].cpu(), w["idx_qs"][:t].cpu(), w["idx_w"][:t].cpu()
    q = torch.cat([w["q_nope"][:t * 128].cpu().reshape(n_seq, s1, 128, 512),
                   w["q_rope"][:t * 128].cpu().reshape(n_seq, s1, 128, 64)], dim=-1)
    def one_pass():
        tk = oi.lightning_indexer(idx_q, idx_qs, host["idx_k"], host["idx_ks"], idx_w, act, table, s1, 2048)
        return osfa.attention_no_flash(q, host["kn"], host["kr"], host["ks"], tk.reshape(t, 2048), table, act, 128, scale,
                                       2048)

    one_pass()  # untimed: first touch of the host copies, thread pool start-up
    passes, t0 = 0, time.perf_counter()
    while passes < 3 or time.perf_counter() - t0 < 10.0:
        one_pass()
        passes += 1
    dt = time.perf_counter() - t0
    return {"value": round(passes * t / dt, 2), "unit": "tokens/s", "cores": torch.get_num_threads(), "kind": "port",
            "sample": f"first {n_seq} of the {w['b']} sequences of the same workload, {passes} passes after an untimed one "
                      f"({dt:.1f} s): oracle.indexer.lightning_indexer + oracle.sfa.attention_no_flash",
            "host_cpus": os.cpu_count()}


def time_cpu_as_written(torch, w, scale):
    """The reference's goldens the way it writes them - a Python loop over pages for the indexer, Python loops over
    batch, query token and selected token for attention - timed once each at the tiny attention configuration (batch 1,
    16 heads, 4096-token cache, top-256) and on the first two sequences of this workload."""
    from oracle import indexer as oi
    from oracle import sfa as osfa
    out = {"kind": "as-written", "unit": "us per query token", "cores": torch.get_num_threads(), "host_cpus": os.cpu_count()}
    c1 = osfa.make_case(1, 16, 1, [4096], topk=256, seed=7, dist="bench", softmax_scale=scale)
    args1 = (c1["q"], c1["kn"], c1["kr"], c1["kn_scales"], c1["topk_indices"], c1["block_table"], c1["act_seq"],
             c1["block_size"], c1["softmax_scale"], c1["topk"])
    osfa.attention_no_flash_token_loop(*args1)
    t0 = time.perf_counter()
    osfa.attention_no_flash_token_loop(*args1)
    out["attention_tiny"] = round((time.perf_counter() - t0) * 1e6, 1)
    n_seq, s1 = min(2, w["b"]), w["s1"]
    t = n_seq * s1
    s = w["sets"][0]
    host = {k: v.cpu() for k, v in s.items() if k != "rows"}
    table, act = w["table"][:n_seq].cpu(), w["act"][:n_seq].tolist()
    q = torch.cat([w["q_nope"][:t * 128].cpu().reshape(n_seq, s1, 128, 512),
                   w["q_rope"][:t * 128].cpu().reshape(n_seq, s1, 128, 64)], dim=-1)
    t0 = time.perf_counter()
    tk = oi.lightning_indexer(w["idx_q"][:t].cpu(), w["idx_qs"][:t].cpu(), host["idx_k"], host["idx_ks"],
                              w["idx_w"][:t].cpu(), act, table, s1, 2048)
    t1 = time.perf_counter()
    osfa.attention_no_flash_token_loop(q, host["kn"], host["kr"], host["ks"], tk.reshape(t, 2048), table, act, 128, scale, 2048)
    t2 = time.perf_counter()
    out["indexer_first_2_sequences"] = round((t1 - t0) * 1e6 / t, 1)
    out["attention_first_2_sequences"] = round((t2 - t1) * 1e6 / t, 1)
    out["sample"] = ("one pass each: oracle.sfa.attention_no_flash_token_loop at batch 1 / 16 heads / top-256, then "
                     "oracle.indexer.lightning_indexer (page loop) + the token loop on the first 2 sequences of this workload")
    return out


if __name__ == "__main__":
    main()
