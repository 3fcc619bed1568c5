"""Benchmark of the LCSA layer call on one MI355X.

A step is one LCSA layer call of the DiT self-attention block on the 1920x1152 workload (bf16, 12 heads x 128,
Lq 17280 = 2 latent frames, Lk 43200 = 5 latent frames incl. cache, local range 11, 30% of the in-window block pairs
kept; Q/K a smooth low-frequency field plus noise, per-head RMS-normed, with 3-D RoPE): block selection (pool Q and K,
block scores, softmax, exact per-(head, slice) top-k, key lists) followed by the block-sparse attention over the kept
128x128 blocks. Inputs are resident in HBM before the timed region. Throughput counts kept-block FLOPs only
(4 * 128 * valid q tokens * valid k tokens per kept (head, q-block, k-block)).

Printed: one JSON line (rank 0) with the layer-call rate, the attention kernel's MFMA roofline fraction (kernel time
from HIP events on the launch stream), the same kernel's dense fallback (every key block of every row listed), the
top-k threshold margin of the workload, and the CPU oracle timed on a bounded sample on the host.
"""
from __future__ import annotations

import argparse
import json
import math
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(ROOT, "mlx-flashvsr-swift_amd")
for p in (PKG, ROOT):
    if p not in sys.path:
        sys.path.insert(0, p)

METRIC = "block-sparse attn ms/layer-call + effective TFLOP/s (% MFMA peak), 1920×1152"
HEADLINE = "sparse_1920x1152_bf16"   # the workload METRIC is quoted on; its PMC summary holds the traffic figure
PEAK_BF16_TFLOPS = 2500.0            # MI355X dense bf16 MFMA
PEAK_FP32_TFLOPS = 157.3             # MI355X dense fp32 MFMA (the fp32 lane, split on the bf16 matrix cores, can pass it)
PROFILE_PMC = os.path.join(ROOT, "profiles", "lcsa_attn_bf16_1920x1152_pmc.txt")


def warmup_of(args, default):
    return default if args.warmup is None else args.warmup


def parse_args():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=None,
                    help="untimed steps first (default: 300 layer calls, ~0.2 s, so the part's clock has settled "
                         "before timing; 20 for the other modes, whose warm-up already runs that long)")
    ap.add_argument("--workload", default=HEADLINE)
    ap.add_argument("--seed", type=int, default=None, help="generator seed (default: the workload's own)")
    ap.add_argument("--cpu-seconds", type=float, default=15.0, help="budget of the CPU oracle sample")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-stream", action="store_true",
                    help="leave out the streaming-stack figures (30 layers from the projections) of the default line")
    ap.add_argument("--attn-only", action="store_true",
                    help="profiling: run only the sparse attention launches (one selection up front) and print a "
                         "summary line instead of the benchmark line")
    ap.add_argument("--stream", action="store_true",
                    help="the streaming attention stack at 1920x1152 instead: 30 layers (KV ring per layer) over a "
                         "6-latent-frame first chunk and 4 chunks of 2 latent frames; append + select + attention + "
                         "evict per layer call; prints its own JSON line")
    ap.add_argument("--layers", type=int, default=30)
    ap.add_argument("--iid", action="store_true", help="with --stream: i.i.d. N(0,1) Q/K instead of a smooth field")
    ap.add_argument("--from-projections", action="store_true",
                    help="with --stream: feed each layer the q/k/v projections in natural token order "
                         "(normQ/normK + RoPE + window partition + ring append fused, output window-reversed)")
    ap.add_argument("--full-blocks", action="store_true",
                    help="with --stream: run whole DiT blocks (norms, modulation, projections, LCSA layer call, "
                         "cross-attention over 512 context tokens, FFN) with random-init weights, 30 of them")
    ap.add_argument("--epilogue", action="store_true",
                    help="time the fused QKV epilogue into the KV ring on one 1920x1152 streaming chunk (HBM-bound)")
    ap.add_argument("--block", action="store_true",
                    help="time one whole DiT block (blockForward: norms, modulation, q/k/v/o, LCSA layer call, "
                         "cross-attention over 512 context tokens, FFN 1536->8960->1536) on a steady 1920x1152 "
                         "streaming chunk; prints its own JSON line")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="run only a plain copy of known size (the window-partition kernel over 16x72x120 bf16 "
                         "tokens of 1536 channels: 424.7 MB read + 424.7 MB written per launch), the reference "
                         "point that scales the FETCH_SIZE / WRITE_SIZE counters")
    ap.add_argument("--gemm-ceiling", action="store_true",
                    help="time only a plain bf16 GEMM (torch.matmul on hipBLASLt, 8192^3 and 16384^3, N(0,1) data): "
                         "the practical MFMA rate of these parts, beside which the attention's rate is read")
    return ap.parse_args()


def read_traffic():
    """HBM bytes per attention launch from the committed rocprofv3 --pmc summary (null if absent)."""
    try:
        with open(PROFILE_PMC) as f:
            for line in f:
                if line.startswith("traffic_bytes_per_launch:"):
                    return float(line.split(":", 1)[1].split()[0])
    except OSError:
        pass
    return None


def threshold_margin(probs, q_slices: int, topk: int) -> float:
    """Smallest relative gap, over the (head, query slice) rows, between the top-k threshold (the (k+1)-th largest
    probability) and the k-th largest, from the selection's own probabilities: the mask is reproducible by any fp32
    implementation of the same formula when this is far above fp32 rounding."""
    import torch

    h, nq, nk = probs.shape
    flat = probs.reshape(h * q_slices, -1)
    kk = min(flat.shape[1] - 1, topk)
    top = torch.topk(flat, kk + 1, dim=1).values            # descending
    thr = top[:, kk]
    if kk == 0:
        return float("inf")
    above = top[:, kk - 1]
    return float(((above - thr) / above.clamp_min(1e-38)).min().item())


def cpu_baseline(wl, q, k, v, mask, kept_flops_total, budget_s):
    """The oracle on the host: selection over the whole workload plus attention over a sample of (head, query
    block) rows, scaled to one layer call. The oracle's attention is a per-row masked softmax over the selected key
    blocks only (a sparse CPU path; the reference's own CPU path, MLX-CPU blockMaskedAttention, computes every
    block pair and would be slower). Also reports whether the oracle's block mask equals the GPU's bit for bit."""
    import numpy as np
    from threadpoolctl import threadpool_info

    from fvsr_lcsa import synth
    from oracle import lcsa as O

    qn, kn, vn = (t.float().cpu().numpy() for t in (q, k, v))
    local = synth.local_mask(wl).numpy()
    topk = synth.workload_topk(wl)
    t0 = time.perf_counter()
    ref_mask, _ = O.draft_block_mask_and_probs(qn, kn, wl.heads, wl.q_slices, wl.s, local, topk, lk=wl.lk)
    t_sel = time.perf_counter() - t0
    m = mask.cpu().numpy()
    mask_equal = bool(np.array_equal(m, ref_mask))
    rows = [(h, i) for h in range(wl.heads) for i in range(wl.nq)]
    rng = np.random.default_rng(0)
    order = rng.permutation(len(rows))
    done, t_att = [], 0.0
    for idx in order:
        h, i = rows[idx]
        t0 = time.perf_counter()
        O.block_masked_attention(qn, kn, vn, m, wl.heads, dtype=np.float32, heads_subset=[h], qblocks_subset=[i])
        t_att += time.perf_counter() - t0
        done.append((h, i))
        if t_att + t_sel >= budget_s and len(done) >= 4:
            break
    # kept FLOPs of the sampled rows vs all rows
    def row_flops(h, i):
        sel = np.nonzero(m[h, i] > 0.5)[0]
        keys = sum(min(128, wl.lk - j * 128) for j in sel)
        return 4.0 * 128 * min(128, wl.lq - i * 128) * keys
    sample_flops = sum(row_flops(h, i) for h, i in done)
    t_layer = t_sel + t_att * kept_flops_total / max(sample_flops, 1.0)
    # the reference's own CPU path (blockMaskedAttention, DiT.swift:279-313): SDPA of a query block over EVERY key
    # under the expanded boolean mask, so its cost does not depend on the selection; a few rows, scaled to all rows
    d = 128
    t_dense, n_dense = 0.0, 0
    for idx in order[:96]:
        h, i = rows[idx]
        t0 = time.perf_counter()
        qh = qn[i * 128:(i + 1) * 128, h * d:(h + 1) * d]
        sc = (qh @ kn[:, h * d:(h + 1) * d].T) * np.float32(1.0 / math.sqrt(d))
        keep = np.repeat(m[h, i] > 0.5, 128)[: wl.lk]
        sc[:, ~keep] = -np.inf
        if keep.any():
            sc = np.exp(sc - sc.max(axis=1, keepdims=True))
            o_row = (sc / sc.sum(axis=1, keepdims=True)) @ vn[:, h * d:(h + 1) * d]
        t_dense += time.perf_counter() - t0
        n_dense += 1
        if t_dense >= 3.0:
            break
    t_dense_layer = t_sel + t_dense * len(rows) / max(n_dense, 1)
    threads = max([p.get("num_threads", 1) for p in threadpool_info() if p.get("user_api") == "blas"] or [1])
    return {
        "value": kept_flops_total / t_layer / 1e12,
        "unit": "TFLOP/s (effective, kept blocks)",
        "ms_per_layer_call": t_layer * 1e3,
        "cores": int(threads),
        "host_cpus": os.cpu_count(),
        "host_cpus_usable": len(os.sched_getaffinity(0)),
        "kind": "port",
        "sample": f"oracle (numpy fp32, {threads} BLAS threads) selection over the full workload ({t_sel:.2f} s) + "
                  f"per-row masked attention over the selected key blocks of {len(done)} of {len(rows)} (head, "
                  f"query block) rows ({t_att:.2f} s), scaled by kept FLOPs",
        "mask_equals_gpu": mask_equal,
        "reference_dense_path": {
            "ms_per_layer_call": round(t_dense_layer * 1e3, 1),
            "tflops_effective_kept": round(kept_flops_total / t_dense_layer / 1e12, 4),
            "sample": f"the selection as above + masked SDPA of a query block over all {wl.lk} keys (the "
                      f"reference's blockMaskedAttention CPU path) on {n_dense} rows ({t_dense:.2f} s), scaled by "
                      f"row count",
        },
    }


def copy_calibration(steps: int):
    """A plain copy of known size: window_partition reads and writes every byte exactly once."""
    import torch

    import fvsr_lcsa

    f, h, w, ch = 16, 72, 120, 1536
    x = torch.randn((f * h * w, ch), device="cuda:0").to(torch.bfloat16)
    nbytes = x.numel() * 2
    for _ in range(2):
        fvsr_lcsa.window_partition(x, f, h, w)
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(steps):
        fvsr_lcsa.window_partition(x, f, h, w)
    e1.record()
    torch.cuda.synchronize()
    ms = e0.elapsed_time(e1) / steps
    print(json.dumps({"copy_calibration": {"bytes_read": nbytes, "bytes_written": nbytes, "ms": round(ms, 4),
                                           "GB/s": round(2 * nbytes / ms / 1e6, 1)}}), flush=True)


def gemm_ceiling(steps: int):
    """The best plain bf16 GEMM the library stack reaches on this part (torch.matmul -> hipBLASLt)."""
    import torch

    out = {}
    for n in (8192, 16384):
        a = torch.randn((n, n), device="cuda:0", dtype=torch.bfloat16)
        b = torch.randn((n, n), device="cuda:0", dtype=torch.bfloat16)
        for _ in range(3):
            c = a @ b
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        reps = max(1, steps)
        e0.record()
        for _ in range(reps):
            c = a @ b
        e1.record()
        torch.cuda.synchronize()
        ms = e0.elapsed_time(e1) / reps
        out[f"{n}^3"] = {"ms": round(ms, 4), "TFLOP/s": round(2 * n ** 3 / (ms * 1e-3) / 1e12, 1)}
        del a, b, c
    print(json.dumps({"gemm_ceiling": out}), flush=True)


def stream_measure(layers: int, reps: int, warm_runs: int, seed: int, iid: bool, proj: bool, split: bool):
    """The attention stack of the streaming DiT at 1920x1152 (the reference's geometry: s = 135 blocks per slice, a
    first chunk of 6 latent frames = 3 slices, then chunks of 2 latent frames = 1 slice; KV window 3 slices;
    default top-k 16199, local range 11; Pipeline.swift:22-23,68,95-102; DiT.swift:478-538). Each layer call runs
    append + select + block-sparse attention + evict through fvsr_lcsa_layer (fvsr_lcsa_layer_qkv with `proj`).
    Q/K/V of each chunk are synthetic, resident in HBM and shared by the layers: by default Q/K are a smooth field
    over the 14 latent frames plus noise (with `proj`: WanRMSNorm weights of about 2, so the pooled scores of a row
    span a wide range, as for real features); `iid` draws them N(0,1). Without `proj` Q/K are per-head RMS-normed
    with 3-D RoPE at the chunk's latent frames. With `split`, the selection and the attention of one steady layer
    call are also timed apart (on the last layer's ring, the new slice appended, back to back). Returns a dict."""
    import torch

    import fvsr_lcsa
    from fvsr_lcsa import synth

    dev = torch.device("cuda:0")
    H, bh, bw = 12, 9, 15
    s = bh * bw
    lat_h, lat_w, C = 8 * bh, 8 * bw, H * 128
    local = fvsr_lcsa.local_block_mask(bh, bw, 11)
    topk = synth.step_topk(s, synth.default_topk_ratio(1152, 1920))
    chunks = [(3, 0), (1, 6), (1, 8), (1, 10), (1, 12)]   # (slices, first latent frame)
    gen = torch.Generator(device=dev).manual_seed(seed)
    data = []
    smooth = not iid
    if smooth:
        cgen = torch.Generator().manual_seed(seed)
        field = synth.smooth_field(14, lat_h, lat_w, C, cgen)
        wscale = 2.0
    else:
        wscale = 1.0
    wq = (wscale * (0.5 + torch.rand(C, generator=gen, device=dev))).to(torch.bfloat16)
    wk = (wscale * (0.5 + torch.rand(C, generator=gen, device=dev))).to(torch.bfloat16)
    for n, t0 in chunks:
        f = 2 * n
        L = f * lat_h * lat_w
        if smooth:
            sl = slice(t0 * lat_h * lat_w, (t0 + f) * lat_h * lat_w)
            q = (field[sl] + 0.5 * torch.randn((L, C), generator=cgen)).to(dev)
            k = (field[sl] + 0.5 * torch.randn((L, C), generator=cgen)).to(dev)
            v = torch.randn((L, C), generator=gen, device=dev)
        else:
            q, k, v = (torch.randn((L, C), generator=gen, device=dev) for _ in range(3))
        if proj:   # the projections themselves, natural token order; the layer call normalises and rotates
            data.append(tuple(x.to(torch.bfloat16).contiguous() for x in (q, k, v)))
            continue
        cos, sin = synth.rope_grid(f, lat_h, lat_w, t0, device=dev)
        q = synth.rope_apply(synth.rms_norm(q, H), H, cos, sin)
        k = synth.rope_apply(synth.rms_norm(k, H), H, cos, sin)
        data.append(tuple(synth.window_partition(x, f, lat_h, lat_w).to(torch.bfloat16).contiguous()
                          for x in (q, k, v)))
    if smooth:
        del field
    ring = fvsr_lcsa.KVRing(layers, H, bh, bw, capacity=4, kv_len=3, dtype=torch.bfloat16)
    outs = [torch.empty_like(d[0]) for d in data]
    qwork = [torch.empty_like(d[0]) for d in data]

    def call(layer, c, want_mask=False):
        (n, t0), (q, k, v), o = chunks[c], data[c], outs[c]
        if proj:
            return ring.layer_call_qkv(layer, q, k, v, n, t0, wq, wk, local, topk, out=o, q_work=qwork[c],
                                       want_mask=want_mask)
        return ring.layer_call(layer, q, k, v, n, n, local, topk, out=o, want_mask=want_mask)

    # kept block pairs per chunk (untimed; the same data feeds every layer)
    kept_pairs = []
    for c in range(len(chunks)):
        _, m, _ = call(0, c, want_mask=True)
        kept_pairs.append(float(m.sum().item()))
    ring.reset()

    def run_stream(events=None):
        ring.reset()
        for c in range(len(chunks)):
            if events is not None:
                events[c][0].record()
            for layer in range(layers):
                call(layer, c)
            if events is not None:
                events[c][1].record()

    for _ in range(warm_runs):
        run_stream()
    torch.cuda.synchronize()
    tot = [0.0] * len(chunks)
    for _ in range(reps):
        ev = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in chunks]
        run_stream(ev)
        torch.cuda.synchronize()
        for c, (a0, a1) in enumerate(ev):
            tot[c] += a0.elapsed_time(a1) / reps
    flops = [4.0 * 128 ** 3 * p * layers for p in kept_pairs]
    steady = tot[1:]
    out = {
        "chunk_ms": [round(t, 3) for t in tot],
        "per_layer_call_ms": [round(t / layers, 4) for t in tot],
        "steady_ms_per_layer_call": round(sum(steady) / len(steady) / layers, 4),
        "chunk0_ms_per_layer_call": round(tot[0] / layers, 4),
        "kept_block_fraction": [round(p / (H * n * s * min(n + (3 if c else 0), 4) * s), 4)
                                for c, ((n, _), p) in enumerate(zip(chunks, kept_pairs))],
        "effective_tflops_kept": [round(f / (t * 1e-3) / 1e12, 1) for f, t in zip(flops, tot)],
        "steady_ms_per_chunk": round(sum(steady) / len(steady), 3),
        "topk": topk, "layers": layers, "reps": reps,
        "_meta": {"H": H, "s": s, "chunks": chunks, "smooth": smooth, "proj": proj},
    }
    if split:
        # one steady layer call taken apart on the last layer's ring (3 slices held): the new slice appended, then
        # the selection and the attention timed back to back, n calls each; then the slice is evicted again
        layer, c = layers - 1, len(chunks) - 1
        (n, t0), (q, k, v) = chunks[c], data[c]
        qw = qwork[c]
        if proj:
            ring.append_qkv(layer, q, k, v, n, t0, wq, wk, q_out=qw)
        else:
            qw = q
            ring.append(layer, k, v, n)
        _, _, kidx, kcnt = ring.select(layer, qw, n, local, topk, want_mask=False, want_probs=False)
        o = outs[c]
        nrep = 20
        for _ in range(3):
            ring.select(layer, qw, n, local, topk, want_mask=False, want_probs=False)
            ring.attention(layer, qw, kidx, kcnt, out=o)
        torch.cuda.synchronize()
        e = [torch.cuda.Event(enable_timing=True) for _ in range(3)]
        e[0].record()
        for _ in range(nrep):
            ring.select(layer, qw, n, local, topk, want_mask=False, want_probs=False)
        e[1].record()
        for _ in range(nrep):
            ring.attention(layer, qw, kidx, kcnt, out=o)
        e[2].record()
        torch.cuda.synchronize()
        ring.evict(layer)
        out["steady_selection_ms"] = round(e[0].elapsed_time(e[1]) / nrep, 4)
        out["steady_attention_ms"] = round(e[1].elapsed_time(e[2]) / nrep, 4)
        steady_flops = 4.0 * 128 ** 3 * kept_pairs[c]
        out["steady_attention_tflops"] = round(steady_flops / (out["steady_attention_ms"] * 1e-3) / 1e12, 1)
    ring.close()
    return out


def stream_bench(args):
    """`--stream`: the streaming attention stack on its own JSON line (see stream_measure)."""
    proj = args.from_projections
    smooth = not args.iid
    r = stream_measure(args.layers, max(1, args.steps // 10), max(1, warmup_of(args, 20) // 5), args.seed or 0,
                       args.iid, proj, split=True)
    meta = r.pop("_meta")
    H, s, chunks = meta["H"], meta["s"], meta["chunks"]
    line = {
        "metric": ("LCSA attention stack per streaming chunk, 1920x1152 (q/k/v projections -> norm + RoPE + window "
                   "partition + append + select + attention + evict + window reverse)" if proj else
                   "LCSA attention stack per streaming chunk, 1920x1152 (append + select + attention + evict)"),
        "unit": "ms per chunk (all layers)",
        "value": r["steady_ms_per_chunk"],
        "higher_is_better": False,
        "n_gpus": 1,
        "dtype": "bf16",
        "data": ("synthetic, seeded: " + ("Q/K a smooth field + N(0, 0.25) noise" if smooth else "Q/K N(0,1)") +
                 ("; WanRMSNorm weights " + ("~2" if smooth else "~1") if proj else "; per-head RMS norm") +
                 " + 3-D RoPE; no checkpoint"),
        "config": {"workload": "stream_1920x1152_bf16" + ("_from_projections" if proj else "") + ("_iid" if not smooth else ""), "layers": args.layers, "heads": H, "head_dim": 128,
                   "spatial_blocks_per_slice": s, "local_range": 11, "topk": r["topk"], "kv_window_slices": 3,
                   "chunks": [{"query_blocks": n * s, "key_blocks": min(n + (3 if c else 0), 4) * s}
                              for c, (n, _) in enumerate(chunks)]},
    }
    line.update(r)
    print(json.dumps(line), flush=True)


def epilogue_bench(args):
    """The projection epilogue of one streaming chunk at 1920x1152 (2 latent frames, 17280 tokens, 12 x 128 heads,
    bf16): WanRMSNorm of q and k, 3-D RoPE, window partition, K/V appended to the ring with pooled keys
    (DiT.swift:34-47,100-118,496-511), one kernel plus the pooled-key finish. HBM-bound: reports GB/s of the
    algorithmic bytes (q, k, v read once; Q, K, V written once; the pooled-key runs written and read once)."""
    import torch

    import fvsr_lcsa

    dev = torch.device("cuda:0")
    H, bh, bw = 12, 9, 15
    s, C = bh * bw, H * 128
    f, h, w = 2, 8 * bh, 8 * bw
    L = f * h * w
    gen = torch.Generator(device=dev).manual_seed(args.seed or 0)
    q, k, v = (torch.randn((L, C), generator=gen, device=dev).to(torch.bfloat16) for _ in range(3))
    wq = (0.5 + torch.rand(C, generator=gen, device=dev)).to(torch.bfloat16)
    wk = (0.5 + torch.rand(C, generator=gen, device=dev)).to(torch.bfloat16)
    ring = fvsr_lcsa.KVRing(1, H, bh, bw, capacity=4, kv_len=3, dtype=torch.bfloat16)
    qo = torch.empty_like(q)

    def once():
        ring.append_qkv(0, q, k, v, 1, 6, wq, wk, q_out=qo)
        ring.evict(0)
        if ring.slices(0) >= 3:
            ring.reset()

    for _ in range(max(3, warmup_of(args, 20))):
        once()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    n = max(10, args.steps)
    e0.record()
    for _ in range(n):
        once()
    e1.record()
    torch.cuda.synchronize()
    ms = e0.elapsed_time(e1) / n
    nbytes = 6 * L * C * 2 + 2 * (L // 128) * 4 * C * 4 + (L // 128) * C * 4
    gbs = nbytes / (ms * 1e-3) / 1e9
    print(json.dumps({
        "metric": "fused QKV epilogue into the KV ring, one 1920x1152 streaming chunk",
        "value": round(gbs, 1), "unit": "GB/s (algorithmic bytes)", "ms_per_call": round(ms, 4),
        "higher_is_better": True, "n_gpus": 1, "dtype": "bf16", "data": "synthetic (seeded N(0,1))",
        "config": {"workload": "epilogue_1920x1152_bf16", "tokens": L, "channels": C, "heads": H},
        "roofline": {"bound": "hbm", "achieved": round(gbs, 1), "peak": 8000.0, "unit": "GB/s",
                     "frac": round(gbs / 8000.0, 4), "traffic": None},
        "algorithmic_bytes": nbytes}), flush=True)


def _random_block(torch, dev, gen, C, F, H, n_ctx, fvsr_lcsa):
    def rnd(*shape, scale=1.0):
        return (torch.randn(shape, generator=gen, device=dev) * scale).to(torch.bfloat16)

    W = {"modulation": rnd(6, C, scale=0.1)}
    for p in ("q", "k", "v", "o", "cross_q", "cross_k", "cross_v", "cross_o"):
        W[p + "_weight"] = rnd(C, C, scale=C ** -0.5)
        W[p + "_bias"] = rnd(C, scale=0.05)
    for p in ("norm_q", "norm_k", "cross_norm_q", "cross_norm_k", "norm3"):
        W[p + "_weight"] = (1 + 0.1 * torch.randn(C, generator=gen, device=dev)).to(torch.bfloat16)
    W["norm3_bias"] = rnd(C, scale=0.05)
    W["ffn1_weight"], W["ffn1_bias"] = rnd(F, C, scale=C ** -0.5), rnd(F, scale=0.05)
    W["ffn2_weight"], W["ffn2_bias"] = rnd(C, F, scale=F ** -0.5), rnd(C, scale=0.05)
    blk = fvsr_lcsa.DiTBlock(W, H)
    blk.set_context(rnd(n_ctx, C))
    return blk


def stream_blocks_bench(args):
    """The streaming DiT's blocks end to end at 1920x1152 (DiT.swift:556-578 without the patch embedding and head):
    30 random-init Wan2.1-1.3B-shaped blocks (dim 1536, 12 heads, FFN 8960, 512 context tokens), a first chunk of
    3 slices then 4 chunks of 1 slice (Pipeline.swift:95-102), each chunk's tokens through every block in turn
    (blockForward: norms, modulation, projections, LCSA layer call on the block's ring layer, cross-attention, FFN).
    FLOPs of a steady chunk: 30 x (1.4405 GEMM + 0.0544 cross-attention + 1.6306 LCSA kept) = 93.77 TFLOP."""
    import torch

    import fvsr_lcsa
    from fvsr_lcsa import synth

    dev = torch.device("cuda:0")
    H, bh, bw, F, n_ctx = 12, 9, 15, 8960, 512
    C, s = H * 128, bh * bw
    lat_h, lat_w = 8 * bh, 8 * bw
    local = fvsr_lcsa.local_block_mask(bh, bw, 11)
    topk = synth.step_topk(s, synth.default_topk_ratio(1152, 1920))
    gen = torch.Generator(device=dev).manual_seed(args.seed or 0)
    blocks = [_random_block(torch, dev, gen, C, F, H, n_ctx, fvsr_lcsa) for _ in range(args.layers)]
    t_mod = (torch.randn((6, C), generator=gen, device=dev) * 0.1).to(torch.bfloat16)
    ring = fvsr_lcsa.KVRing(args.layers, H, bh, bw, capacity=4, kv_len=3, dtype=torch.bfloat16)
    chunks = [(3, 0), (1, 6), (1, 8), (1, 10), (1, 12)]
    xs = [(torch.randn((2 * n * lat_h * lat_w, C), generator=gen, device=dev)).to(torch.bfloat16) for n, _ in chunks]

    def run(events=None):
        ring.reset()
        for c, (n, t0) in enumerate(chunks):
            x = xs[c].clone()
            if events is not None:
                events[c][0].record()
            for layer, blk in enumerate(blocks):
                blk.forward(ring, layer, x, t_mod, n, t0, local, topk)
            if events is not None:
                events[c][1].record()
            if not torch.isfinite(x.float()).all():
                raise RuntimeError("DiT blocks produced non-finite tokens")

    run()   # warm-up: workspaces, GEMM algorithms
    torch.cuda.synchronize()
    reps = max(1, args.steps // 10)
    tot = [0.0] * len(chunks)
    for _ in range(reps):
        ev = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in chunks]
        run(ev)
        torch.cuda.synchronize()
        for c, (a0, a1) in enumerate(ev):
            tot[c] += a0.elapsed_time(a1) / reps
    steady = tot[1:]
    L = s * 128   # tokens of a steady chunk: one slice = 2 latent frames
    per_block = 2.0 * L * (6 * C * C + 2 * C * F) + 4.0 * L * n_ctx * C + 4.0 * 128 ** 3 * H * topk
    print(json.dumps({
        "metric": "streaming DiT blocks per chunk, 1920x1152 (30 blocks: norms, modulation, projections, LCSA, "
                  "cross-attention, FFN)",
        "unit": "ms per chunk (all blocks)", "value": round(sum(steady) / len(steady), 3), "higher_is_better": False,
        "n_gpus": 1, "dtype": "bf16", "data": "synthetic tokens, random-init weights (no checkpoint)",
        "config": {"workload": "stream_blocks_1920x1152_bf16", "blocks": args.layers, "heads": H, "dim": C,
                   "ffn_dim": F, "context_tokens": n_ctx, "topk": topk, "local_range": 11, "kv_window_slices": 3},
        "chunk_ms": [round(t, 3) for t in tot],
        "per_block_ms": [round(t / args.layers, 4) for t in tot],
        "steady_effective_tflops": round(args.layers * per_block / (sum(steady) / len(steady) * 1e-3) / 1e12, 1),
        "reps": reps}), flush=True)


def block_bench(args):
    """One streaming `blockForward` (DiT.swift:491-551) of the Wan2.1-1.3B-shaped DiT (dim 1536, 12 heads, FFN 8960,
    512 context tokens) on a steady 1920x1152 chunk: 2 latent frames = 17280 tokens, KV window of 3 slices + the new
    one (135 x 540 key blocks, top-k 16199, local range 11). Random-init weights (no checkpoint), synthetic tokens;
    the ring is filled by a first chunk of 3 slices before timing. FLOPs per call: GEMMs 17280 x (12 C^2 + 4 C F)
    = 1.4405 TFLOP, cross-attention 4 x 17280 x 512 x C = 0.0544 TFLOP, LCSA kept blocks 12 x 16199 x 128^3 x 4 =
    1.6306 TFLOP (top-k keeps exactly 16199 pairs per (head, slice) without ties)."""
    import torch

    import fvsr_lcsa
    from fvsr_lcsa import synth

    dev = torch.device("cuda:0")
    H, bh, bw, F, n_ctx = 12, 9, 15, 8960, 512
    C, s = H * 128, bh * bw
    lat_h, lat_w = 8 * bh, 8 * bw
    local = fvsr_lcsa.local_block_mask(bh, bw, 11)
    topk = synth.step_topk(s, synth.default_topk_ratio(1152, 1920))
    gen = torch.Generator(device=dev).manual_seed(args.seed or 0)

    def rnd(*shape, scale=1.0):
        return (torch.randn(shape, generator=gen, device=dev) * scale).to(torch.bfloat16)

    blk = _random_block(torch, dev, gen, C, F, H, n_ctx, fvsr_lcsa)
    t_mod = rnd(6, C, scale=0.1)
    ring = fvsr_lcsa.KVRing(1, H, bh, bw, capacity=4, kv_len=3, dtype=torch.bfloat16)
    x0 = rnd(6 * lat_h * lat_w, C)
    blk.forward(ring, 0, x0, t_mod, 3, 0, local, topk)   # chunk 0: 3 slices fill the window
    L = 2 * lat_h * lat_w
    x = rnd(L, C)
    t0 = 6
    for _ in range(max(2, warmup_of(args, 20))):
        blk.forward(ring, 0, x, t_mod, 1, t0, local, topk)
    torch.cuda.synchronize()
    n = max(5, args.steps)
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(n):
        blk.forward(ring, 0, x, t_mod, 1, t0, local, topk)
    e1.record()
    torch.cuda.synchronize()
    ms = e0.elapsed_time(e1) / n
    if not torch.isfinite(x.float()).all():
        raise RuntimeError("DiT block produced non-finite tokens")
    gemm = 2.0 * L * (6 * C * C + 2 * C * F)   # q, k, v, o, cross q, cross o; FFN up and down
    cross = 4.0 * L * n_ctx * C
    lcsa = 4.0 * 128 ** 3 * H * topk
    total = gemm + cross + lcsa
    print(json.dumps({
        "metric": "DiT block (blockForward) per steady streaming chunk, 1920x1152",
        "value": round(ms, 4), "unit": "ms per block call", "higher_is_better": False, "n_gpus": 1, "dtype": "bf16",
        "data": "synthetic tokens, random-init weights (no checkpoint)",
        "config": {"workload": "dit_block_1920x1152_bf16", "tokens": L, "dim": C, "heads": H, "ffn_dim": F,
                   "context_tokens": n_ctx, "key_blocks": 4 * s, "topk": topk, "local_range": 11},
        "tflop_per_call": {"gemm": round(gemm / 1e12, 4), "cross_attention": round(cross / 1e12, 4),
                           "lcsa_kept": round(lcsa / 1e12, 4)},
        "effective_tflops": round(total / (ms * 1e-3) / 1e12, 1),
        "per_chunk_ms_30_blocks": round(30 * ms, 2),
        "steps": n}), flush=True)


def main():
    args = parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU: this build has no multi-GPU path (asked for --gpus {args.gpus}). "
              "Run with --gpus 1.", file=sys.stderr)
        sys.exit(2)
    import torch

    import fvsr_lcsa
    from fvsr_lcsa import synth

    assert torch.cuda.is_available(), "bench.py needs a HIP device"
    if args.copy_calibration:
        copy_calibration(args.steps)
        return
    if args.gemm_ceiling:
        gemm_ceiling(args.steps)
        return
    if args.stream and args.full_blocks:
        stream_blocks_bench(args)
        return
    if args.stream:
        stream_bench(args)
        return
    if args.epilogue:
        epilogue_bench(args)
        return
    if args.block:
        block_bench(args)
        return
    dev = torch.device("cuda:0")
    wl = synth.WORKLOADS[args.workload]
    seed = wl.seed if args.seed is None else args.seed
    q, k, v = synth.make_qkv(wl, seed=seed, device=dev)
    local = synth.local_mask(wl).numpy()
    topk = synth.workload_topk(wl)
    ctx = fvsr_lcsa.Context.get(dev)
    ctx.reserve(fvsr_lcsa.workspace_size(wl.heads, wl.lq, wl.lk, wl.channels))
    stream = torch.cuda.current_stream()
    o = torch.empty_like(q)

    def select():
        return fvsr_lcsa.draft_block_mask_and_probs(q, k, wl.heads, wl.q_slices, wl.s, local, topk,
                                                    want_mask=False, want_probs=False)

    def attend(kidx, kcnt, out=o):
        fvsr_lcsa.block_sparse_attention(q, k, v, kidx, kcnt, wl.heads, out=out)

    # one selection up front (untimed) for FLOP counting, the threshold margin and the dense fallbacks
    mask, probs, kidx, kcnt = fvsr_lcsa.draft_block_mask_and_probs(q, k, wl.heads, wl.q_slices, wl.s, local, topk)
    torch.cuda.synchronize()
    kept = synth.kept_flops(kcnt, kidx, wl.lq, wl.lk)
    kept_fraction = float(kcnt.sum().item()) / (wl.heads * wl.nq * wl.nk)
    margin = threshold_margin(probs, wl.q_slices, topk)
    empty_rows = int((kcnt == 0).sum().item())
    del probs

    for _ in range(warmup_of(args, 300)):
        _, _, ki, kc = select()
        attend(ki, kc)
    torch.cuda.synchronize()

    # the layer call: K back to back (events only around the loop: an event between two kernels stalls the queue for
    # several microseconds)
    t_start = torch.cuda.Event(enable_timing=True)
    t_end = torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    wall0 = time.perf_counter()
    t_start.record(stream)
    for _ in range(args.steps):
        if args.attn_only:
            attend(kidx, kcnt)
            continue
        _, _, ki, kc = select()
        attend(ki, kc)
    t_end.record(stream)
    torch.cuda.synchronize()
    wall = time.perf_counter() - wall0
    ms_step = t_start.elapsed_time(t_end) / args.steps
    if args.attn_only:   # profiling runs: the sparse attention launches only, then one summary line
        print(json.dumps({"profiling": "attention only", "workload": wl.name, "steps": args.steps,
                          "ms_per_attention_call": round(ms_step, 4),
                          "attention_tflops": round(kept / (ms_step * 1e-3) / 1e12, 2)}), flush=True)
        return
    # the attention alone (row order + sparse walk, the roofline kernel) and the selection alone, K back to back each,
    # on the launch stream
    a0, a1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    a0.record(stream)
    for _ in range(args.steps):
        attend(kidx, kcnt)
    a1.record(stream)
    s0, s1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    s0.record(stream)
    for _ in range(args.steps):
        select()
    s1.record(stream)
    # the layer call timed once more, after the two loops above: the first loop runs while the part's clock is still
    # rising from idle (it settles over roughly 0.1 s of load), this one on a settled clock; `value` stays the first
    r0, r1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    r0.record(stream)
    for _ in range(args.steps):
        _, _, ki, kc = select()
        attend(ki, kc)
    r1.record(stream)
    torch.cuda.synchronize()
    ms_attn = a0.elapsed_time(a1) / args.steps
    ms_select = s0.elapsed_time(s1) / args.steps
    ms_again = r0.elapsed_time(r1) / args.steps

    def timed(fn, n):
        for _ in range(2):
            fn()
        torch.cuda.synchronize()
        d0, d1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        d0.record(stream)
        for _ in range(n):
            fn()
        d1.record(stream)
        torch.cuda.synchronize()
        return d0.elapsed_time(d1) / n

    nd = max(3, args.steps // 4)
    od = torch.empty_like(q)
    # dense fallback as the reference's blockMaskedAttention costs it (DiT.swift:279-313): every key block of every
    # query block listed (kcnt = Nk), the same kernel walking all H x Nq x Nk block pairs
    kidx_all = torch.arange(wl.nk, dtype=torch.int32, device=dev).repeat(wl.heads, wl.nq, 1).contiguous()
    kcnt_all = torch.full((wl.heads, wl.nq), wl.nk, dtype=torch.int32, device=dev)
    ms_dense = timed(lambda: attend(kidx_all, kcnt_all, od), nd)
    del kidx_all, kcnt_all
    # the call from the selected mask (either mode): the mask -> list build (a few us) and the same walk
    ms_masked = timed(lambda: fvsr_lcsa.block_masked_attention(q, k, v, mask, wl.heads, out=od), nd)
    dense_flops = 4.0 * 128 * wl.heads * wl.lq * wl.lk
    cpu_inputs = None
    if not args.no_cpu and not args.no_stream and wl.name == HEADLINE:
        cpu_inputs = tuple(t.cpu() for t in (q, k, v, mask))

    achieved = kept / (ms_attn * 1e-3) / 1e12
    value = kept / (ms_step * 1e-3) / 1e12
    fp32 = wl.dtype == torch.float32
    peak = PEAK_FP32_TFLOPS if fp32 else PEAK_BF16_TFLOPS
    # the committed PMC summary covers the headline workload's kernel only
    traffic = read_traffic() if wl.name == HEADLINE else None
    res = f"{wl.width}×{wl.height}"
    line = {
        "metric": METRIC if wl.name == HEADLINE else METRIC.replace("1920×1152", res),
        "value": round(value, 2),
        "unit": "TFLOP/s (effective, kept blocks; whole layer call = selection + attention)",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": warmup_of(args, 300),
        "ms_per_step": round(ms_step, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp32" if fp32 else "bf16",
        "data": (f"synthetic, seed {seed} ({'smooth field + noise, ' if wl.smooth else 'i.i.d. N(0,1), '}"
                 "per-head RMS norm + 3-D RoPE on Q/K; no checkpoint)"),
        "config": {
            "workload": wl.name,
            "description": wl.description,
            "heads": wl.heads, "head_dim": 128, "lq": wl.lq, "lk": wl.lk, "q_blocks": wl.nq, "k_blocks": wl.nk,
            "spatial_blocks_per_slice": wl.s, "local_range": wl.local_range, "topk": topk,
            "kept_block_fraction": round(kept_fraction, 4), "kept_tflop": round(kept / 1e12, 4),
            "empty_rows": empty_rows, "rows": wl.heads * wl.nq,
            "threshold_margin": float(f"{margin:.4g}"),
        },
        "breakdown_ms": {
            "layer_call": round(ms_step, 4),
            "attention_kernel": round(ms_attn, 4),
            "selection": round(ms_select, 4),
            "selection_plus_attention": round(ms_select + ms_attn, 4),
            "layer_call_timed_again": round(ms_again, 4),
            "dense_fallback_all_blocks": round(ms_dense, 4),
            "attention_from_mask": round(ms_masked, 4),
        },
        "attention_tflops": round(achieved, 2),
        "layer_call_frac": round(value / peak, 4),
        "sparse_vs_dense_speedup": round(ms_dense / ms_attn, 3),
        "layer_call_vs_dense_speedup": round(ms_dense / ms_step, 3),
        "dense_fallback_tflops": round(dense_flops / (ms_dense * 1e-3) / 1e12, 1),
        "roofline": {
            "bound": "mfma",
            "achieved": round(achieved, 2),
            "peak": peak,
            "unit": "TFLOP/s",
            "frac": round(achieved / peak, 4),
            "traffic": traffic,
            "traffic_source": (f"{os.path.relpath(PROFILE_PMC, ROOT)}: rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE of "
                               "the sparse attention kernel, copy-calibrated (not measured in this run)"
                               if traffic is not None else None),
        },
        "host_wall_s": round(wall, 3),
    }
    if not args.no_stream and wl.name == HEADLINE:
        # the streaming stack of the same resolution (30 layers, chunks of 3, 1, 1, 1, 1 slices from the q/k/v
        # projections: epilogue + append + select + attention + evict per layer call), one timed pass
        del q, k, v, o, od, mask, kidx, kcnt
        torch.cuda.empty_cache()
        r = stream_measure(30, 1, 1, 0, iid=False, proj=True, split=True)
        r.pop("_meta")
        line["stream_1920x1152"] = {
            "workload": "stream_1920x1152_bf16_from_projections",
            "steady_ms_per_layer_call": r["steady_ms_per_layer_call"],
            "chunk0_ms_per_layer_call": r["chunk0_ms_per_layer_call"],
            "steady_selection_ms": r["steady_selection_ms"],
            "steady_attention_ms": r["steady_attention_ms"],
            "steady_attention_tflops": r["steady_attention_tflops"],
            "chunk_ms_30_layers": r["chunk_ms"],
            "kept_block_fraction": r["kept_block_fraction"],
        }
        if cpu_inputs is not None:
            q, k, v, mask = cpu_inputs
    if not args.no_cpu and not args.attn_only:
        line["cpu_baseline"] = cpu_baseline(wl, q, k, v, mask, kept, args.cpu_seconds)
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
