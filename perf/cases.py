"""The calls whose speed this framework is measured by: what a FlashVSR pipeline has it do, from one 256 x 256 block call
to the 1920 x 1152 streaming stack, through the package's public entry points.

A case is a dict of plain values with a `kind`:

  layer     one LCSA layer call over plain buffers: block selection, then block-sparse attention, from the lists
            (`api` "lists") or from the block mask (`api` "mask": the reference's own sequence of calls)
  masked    attention under a given block mask (FlashVSRAttentionOps.kernel / .dense), any token counts
  clip      a streaming clip on one layer from the q/k/v projections: a first chunk of 3 temporal slices, then chunks of
            one (epilogue into the KV ring, selection, attention in the `auto` mode, evict)
  windows   the same clip from normed and rotated tokens in natural order: window partition of the queries, ring append
            from grid order, selection, attention, window reverse
  block     a streaming clip through one whole DiT block (projections, clip attention, cross-attention, FFN)
  epilogue  RMSNorm + RoPE + window partition of one chunk's projections

Sizes are given in 128 x 128 pixel blocks (bh x bw; s = bh * bw windows of 128 tokens per temporal slice of two latent
frames). Inputs are made on the GPU from the seed alone: smooth low-frequency fields plus noise where a path meets
features of a video (their pooled scores are what a selection is made from), N(0, 1) elsewhere.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "mlx-flashvsr-swift_amd"))

import fvsr_lcsa  # noqa: E402

D = 128             # head dim, and tokens per window
EPS = 1e-6


def listed():
    return [
        # the headline workload: one layer call at 1920 x 1152, 2 latent frames of queries over 5 of keys (a ragged end)
        dict(name="layer 1920x1152", kind="layer", api="lists", dtype="bf16", bh=9, bw=15, heads=12, q_frames=2,
             k_frames=5, local=11, keep=0.3, rope=True, noise=1.0),
        # an ordinary sparse layer call: 1280 x 768, a locality window of 3 blocks
        dict(name="layer 1280x768", kind="layer", api="lists", dtype="bf16", bh=6, bw=10, heads=12, q_frames=2,
             k_frames=5, local=3, keep=0.6, rope=False, noise=0.35),
        # the fp32 lane at 512 x 512: draft mask, then the kernel under that mask
        dict(name="layer 512x512 fp32", kind="layer", api="mask", dtype="fp32", bh=4, bw=4, heads=12, q_frames=2,
             k_frames=6, local=3, keep=0.5, rope=False, noise=0.0),
        # the dense fallback of a steady 1280 x 768 chunk (60 x 240 blocks, half of them kept)
        dict(name="dense fallback 60x240", kind="masked", mode="dense", dtype="bf16", heads=12, lq=7680, lk=30720,
             density=0.5),
        # a small kernel call with ragged ends on both sides
        dict(name="kernel ragged small", kind="masked", mode="kernel", dtype="bf16", heads=12, lq=1100, lk=2330,
             density=0.5),
        # the largest call: a first chunk and a steady one at 1920 x 1152 (default top-k, window 11)
        dict(name="clip 1920x1152", kind="clip", dtype="bf16", bh=9, bw=15, heads=12, chunks=2, local=11, ratio=0.888889),
        # the same at the default 1280 x 768, where `auto` takes the dense fallback
        dict(name="clip 1280x768", kind="clip", dtype="bf16", bh=6, bw=10, heads=12, chunks=2, local=11, ratio=2.0),
        # a small preview clip, five chunks: launches and latency
        dict(name="clip 384x256", kind="clip", dtype="bf16", bh=2, bw=3, heads=12, chunks=5, local=3, ratio=2.0),
        # the fp32 lane streaming at 512 x 512
        dict(name="windows 512x512 fp32", kind="windows", dtype="fp32", bh=4, bw=4, heads=12, chunks=2, local=11,
             ratio=2.0),
        # one DiT block of the 1.3B-shaped model at 1280 x 768, first chunk and a steady one
        dict(name="block 1280x768", kind="block", dtype="bf16", bh=6, bw=10, heads=12, chunks=2, local=11, ratio=2.0,
             ffn=8960, context=512),
        # and at 256 x 256: small GEMMs, launches
        dict(name="block 256x256", kind="block", dtype="bf16", bh=2, bw=2, heads=12, chunks=3, local=11, ratio=2.0,
             ffn=8960, context=512),
        # the projections' epilogue of a steady 1920 x 1152 chunk
        dict(name="epilogue 1920x1152", kind="epilogue", dtype="bf16", bh=9, bw=15, heads=12, slices=1),
    ]


def draw(rng):
    biggest = max(_cost(c) for c in listed())
    while True:
        c = _draw(rng)
        if _cost(c) <= 0.8 * biggest:
            return c


def _draw(rng):
    kind = rng.choice(["layer", "layer", "masked", "masked", "clip", "clip", "windows", "block", "epilogue"])
    dtype = "fp32" if kind not in ("clip", "block") and rng.random() < 0.35 else "bf16"
    bh, bw = rng.randint(1, 9), rng.randint(2, 15)
    heads = rng.choice([2, 3, 4, 8, 12, 12, 12])
    local = rng.choice([3, 5, 9, 11, 11])
    c = dict(kind=kind, dtype=dtype, bh=bh, bw=bw, heads=heads)
    if kind == "layer":
        c.update(api=rng.choice(["lists", "mask"]), q_frames=rng.choice([2, 2, 2, 4, 6]), k_frames=rng.randint(2, 8),
                 local=local, keep=round(rng.uniform(0.15, 0.95), 3), rope=rng.random() < 0.5,
                 noise=rng.choice([0.35, 0.5, 1.0]))
        c["k_frames"] = max(c["k_frames"], c["q_frames"])
    elif kind == "masked":
        lq = int(math.exp(rng.uniform(math.log(130), math.log(24000))))
        lk = int(math.exp(rng.uniform(math.log(130), math.log(60000))))
        c = dict(kind=kind, mode=rng.choice(["dense", "kernel"]), dtype=dtype, heads=heads, lq=lq, lk=lk,
                 density=round(rng.uniform(0.15, 0.95), 3))
    elif kind in ("clip", "windows"):
        c.update(chunks=rng.randint(1, 4), local=local, ratio=round(rng.uniform(0.4, 2.5), 3))
    elif kind == "block":
        c.update(chunks=rng.randint(1, 3), local=local, ratio=round(rng.uniform(0.4, 2.5), 3),
                 ffn=8 * rng.randint(32 * heads, 94 * heads), context=rng.choice([100, 257, 512]))
    else:
        c.update(slices=rng.randint(1, 3))
    return c


# ---------------------------------------------------------------------------------------------------------------
# geometry
# ---------------------------------------------------------------------------------------------------------------
def _dtype(c):
    return torch.bfloat16 if c["dtype"] == "bf16" else torch.float32


def _schedule(c):
    """(slices, first latent frame) of each chunk: 3 slices, then 1 each."""
    return [(3, 0)] + [(1, 6 + 2 * i) for i in range(c["chunks"] - 1)]


def _windows(bh, bw, r):
    """(s, s) bool: key blocks visible to a query block (a window of r x r blocks from r // 2 before it)."""
    y, x = torch.arange(bh), torch.arange(bw)

    def near(i):
        d = i[None, :] - i[:, None]
        return (d >= -(r // 2)) & (d <= -(r // 2) + r - 1)
    return (near(y)[:, None, :, None] & near(x)[None, :, None, :]).reshape(bh * bw, bh * bw)


def _layer_topk(c):
    s = c["bh"] * c["bw"]
    nk = -(-c["k_frames"] * s * 64 // D)
    return int(c["keep"] * int(_windows(c["bh"], c["bw"], c["local"])[:, torch.arange(nk) % s].sum()))


def _clip_topk(c):
    s = c["bh"] * c["bw"]
    return int(s * s * c["ratio"]) - 1


def _calls(c):
    """(query blocks, key blocks, kept pairs of one head) of every attention call of the case."""
    if c["kind"] == "masked":
        nq, nk = -(-c["lq"] // D), -(-c["lk"] // D)
        return [(nq, nk, c["density"] * nq * nk)]
    s = c["bh"] * c["bw"]
    win = int(_windows(c["bh"], c["bw"], c["local"]).sum()) if "local" in c else 0
    if c["kind"] == "layer":
        qs, nk = c["q_frames"] // 2, -(-c["k_frames"] * s * 64 // D)
        return [(qs * s, nk, qs * _layer_topk(c))]
    if c["kind"] == "epilogue":
        return []
    out, held = [], 0
    for n, _ in _schedule(c):
        nk = (held + n) * s
        out.append((n * s, nk, n * min(_clip_topk(c), win * (held + n))))
        held = min(3, held + n)
    return out


def work(case):
    c = case
    es, C = (2 if c["dtype"] == "bf16" else 4), c["heads"] * D
    flops = sum(c["heads"] * (4.0 * D ** 3 * kept) for _, _, kept in _calls(c))
    if c["kind"] == "masked":
        nq, nk = -(-c["lq"] // D), -(-c["lk"] // D)
        return {"flops": flops, "bytes": (2 * c["lq"] + 2 * c["lk"]) * C * es + 4 * c["heads"] * nq * nk}
    if c["kind"] == "epilogue":
        return {"flops": 0, "bytes": 6 * c["slices"] * c["bh"] * c["bw"] * D * C * es}
    flops += sum(c["heads"] * 2.0 * D * nq * nk for nq, nk, _ in _calls(c))   # pooled scores
    if c["kind"] == "layer":
        lq, lk = (c[f] * c["bh"] * c["bw"] * 64 for f in ("q_frames", "k_frames"))
        lists = c["heads"] * sum(4 * nq * nk for nq, nk, _ in _calls(c)) * (1 if c["api"] == "lists" else 4)
        return {"flops": flops, "bytes": (2 * lq + 2 * lk) * C * es + lists}
    tokens = sum(nq for nq, _, _ in _calls(c)) * D
    cached = sum(nk - nq for nq, nk, _ in _calls(c)) * D                      # keys and values of earlier chunks
    if c["kind"] in ("clip", "windows"):
        return {"flops": flops, "bytes": (4 * tokens + 2 * cached) * C * es}
    flops += 2.0 * tokens * (6 * C * C + 2 * C * c["ffn"]) + 4.0 * tokens * c["context"] * C
    weights = (6 * C * C + 2 * C * c["ffn"]) * c["chunks"]
    return {"flops": flops, "bytes": (2 * tokens * C + 2 * cached * C + weights) * es}


def _cost(c):
    """Rough seconds of a pass: what draw() keeps within the listed cases' range."""
    w, walked = work(c), 0.0
    for nq, nk, kept in _calls(c):   # the dense fallback visits every block
        s = c["bh"] * c["bw"] if "bh" in c else 0
        dense = c.get("mode") == "dense" or ("ratio" in c and (_clip_topk(c) + 1) / (s * nk) > 0.45)
        walked += c["heads"] * 4.0 * D ** 3 * (nq * nk if dense else kept)
    return max(w["flops"], walked) / (0.95e15 if c["dtype"] == "bf16" else 5e13) + w["bytes"] / 4e12 + 4e-5


def tolerance(case):
    """About four times the measured error against exact(): 2.3e-3 (bf16 attention: the output's rounding and the
    probabilities'), 8e-7 to 1.9e-6 (fp32), 1.7e-3 (a block), 2e-5 (the bf16 epilogue: single roundings)."""
    if case["kind"] == "epilogue":
        return {"rel": 1e-4, "max": 0.02} if case["dtype"] == "bf16" else {"rel": 1e-6, "max": 1e-5}
    if case["kind"] == "block":
        return {"rel": 7e-3, "max": 0.3}
    if case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 0.4, "differ": 0.002}
    return {"rel": 8e-6, "max": 1e-3, "differ": 0.002}


# ---------------------------------------------------------------------------------------------------------------
# inputs: plain tensors from the seed, on the GPU
# ---------------------------------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda")


def _field(gen, f, h, w, C, modes=6):
    """A low-frequency random field over (t, y, x): plane waves of random phase and amplitude per channel."""
    t, y, x = torch.meshgrid(torch.arange(f, device="cuda") / max(f, 1), torch.arange(h, device="cuda") / h,
                             torch.arange(w, device="cuda") / w, indexing="ij")
    pos = torch.stack([t.reshape(-1), y.reshape(-1), x.reshape(-1)], 1).float()
    out = torch.zeros((pos.shape[0], C), device="cuda")
    for _ in range(modes):
        k = torch.randint(-2, 3, (3,), generator=gen, device="cuda").float()
        k[1] += (k.abs().sum() == 0).float()
        arg = 2 * math.pi * (pos * k).sum(1, keepdim=True)
        out += torch.cos(arg + 2 * math.pi * torch.rand((1, C), generator=gen, device="cuda")) * _randn(gen, 1, C)
    return out


def _rope(x, heads, f, h, w, t0):
    """3-D RoPE of natural-order tokens: 22 | 21 | 21 rotations of (even, odd) pairs by t, y and x, in x's precision."""
    ang = []
    pos = torch.meshgrid(torch.arange(t0, t0 + f, device="cuda", dtype=torch.float64),
                         torch.arange(h, device="cuda", dtype=torch.float64),
                         torch.arange(w, device="cuda", dtype=torch.float64), indexing="ij")
    for p, dim in zip(pos, (44, 42, 42)):
        freq = 10000.0 ** (-torch.arange(0, dim, 2, device="cuda", dtype=torch.float64) / dim)
        ang.append(p.reshape(-1, 1) * freq)
    ang = torch.cat(ang, 1)[:, None, :]
    cos, sin = torch.cos(ang).float().to(x.dtype), torch.sin(ang).float().to(x.dtype)
    y = x.reshape(x.shape[0], heads, D // 2, 2)
    return torch.stack([y[..., 0] * cos - y[..., 1] * sin, y[..., 0] * sin + y[..., 1] * cos], -1).reshape(x.shape)


def _head_norm(x, heads):
    y = x.reshape(x.shape[0], heads, D)
    return (y * torch.rsqrt(y.square().mean(-1, keepdim=True) + EPS)).reshape(x.shape)


def _partition(x, f, h, w):
    return x.reshape(f // 2, 2, h // 8, 8, w // 8, 8, -1).permute(0, 2, 4, 1, 3, 5, 6).reshape(f * h * w, -1).contiguous()


def _reverse(x, f, h, w):
    return x.reshape(f // 2, h // 8, w // 8, 2, 8, 8, -1).permute(0, 3, 1, 4, 2, 5, 6).reshape(f * h * w, -1).contiguous()


def _inputs(c, seed):
    gen, dt, heads = _gen(seed), _dtype(c), c["heads"]
    C = heads * D
    if c["kind"] == "masked":
        q, k, v = (_randn(gen, c[n], C).to(dt) for n in ("lq", "lk", "lk"))
        mask = torch.rand((heads, -(-c["lq"] // D), -(-c["lk"] // D)), generator=gen, device="cuda") < c["density"]
        return dict(q=q, k=k, v=v, mask=mask.float())
    h, w = 8 * c["bh"], 8 * c["bw"]
    if c["kind"] == "epilogue":
        f = 2 * c["slices"]
        q, k, v = (_randn(gen, f * h * w, C).to(dt) for _ in range(3))
        wq, wk = ((0.5 + torch.rand(C, generator=gen, device="cuda")).to(dt) for _ in range(2))
        return dict(q=q, k=k, v=v, wq=wq, wk=wk)
    if c["kind"] == "layer":
        qf, kf = c["q_frames"], c["k_frames"] + c["k_frames"] % 2
        q, k, v = (_randn(gen, n * h * w, C) for n in (qf, kf, kf))
        if c["noise"] > 0:
            fk = _field(gen, kf, h, w, C)
            k = fk + c["noise"] * k
            q = fk[(kf - qf) * h * w:] + c["noise"] * q
        q, k = _head_norm(q, heads), _head_norm(k, heads)
        if c["rope"]:
            q, k = _rope(q, heads, qf, h, w, kf - qf), _rope(k, heads, kf, h, w, 0)
        lk = c["k_frames"] * h * w
        return dict(q=_partition(q, qf, h, w).to(dt), k=_partition(k, kf, h, w)[:lk].to(dt).contiguous(),
                    v=_partition(v, kf, h, w)[:lk].to(dt).contiguous())
    frames = 2 * sum(n for n, _ in _schedule(c))
    field = _field(gen, frames, h, w, C)
    part = [slice(t0 * h * w, (t0 + 2 * n) * h * w) for n, t0 in _schedule(c)]
    if c["kind"] == "block":
        def mat(o, i):
            return (_randn(gen, o, i) * i ** -0.5).to(dt)

        def vec(n, scale, base=0.0):
            return (base + scale * _randn(gen, n)).to(dt)
        F, W = c["ffn"], {}
        W["modulation"] = (0.1 * _randn(gen, 6, C)).to(dt)
        for p in ("q", "k", "v", "o", "cross_q", "cross_k", "cross_v", "cross_o"):
            W[p + "_weight"], W[p + "_bias"] = mat(C, C), vec(C, 0.05)
        for p in ("norm_q", "norm_k", "cross_norm_q", "cross_norm_k", "norm3"):
            W[p + "_weight"] = vec(C, 0.1, 1.0)
        W["norm3_bias"] = vec(C, 0.05)
        W["ffn1_weight"], W["ffn1_bias"] = mat(F, C), vec(F, 0.05)
        W["ffn2_weight"], W["ffn2_bias"] = mat(C, F), vec(C, 0.05)
        xs = [(field[p] + 0.5 * _randn(gen, p.stop - p.start, C)).to(dt) for p in part]
        return dict(xs=xs, W=W, context=_randn(gen, c["context"], C).to(dt), t_mod=(0.1 * _randn(gen, 6, C)).to(dt))
    chunks = []
    for p, (n, t0) in zip(part, _schedule(c)):
        q, k = (field[p] + 0.5 * _randn(gen, p.stop - p.start, C) for _ in range(2))
        v = _randn(gen, p.stop - p.start, C)
        if c["kind"] == "windows":   # normed and rotated by the caller
            q, k = (_rope(_head_norm(x, heads), heads, 2 * n, h, w, t0) for x in (q, k))
        chunks.append(tuple(x.to(dt).contiguous() for x in (q, k, v)))
    # norm weights of about 2, as trained ones: the scores of a row span a wide range
    wq, wk = ((2.0 * (0.5 + torch.rand(C, generator=gen, device="cuda"))).to(dt) for _ in range(2))
    return dict(chunks=chunks, wq=wq, wk=wk)


# ---------------------------------------------------------------------------------------------------------------
# the framework's calls
# ---------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    c, x = case, _inputs(case, seed)
    st = dict(c=c, **x)
    if "local" in c:
        st["local"] = fvsr_lcsa.local_block_mask(c["bh"], c["bw"], c["local"])
    if c["kind"] == "layer":
        st["topk"], st["out"] = _layer_topk(c), torch.empty_like(x["q"])
    elif c["kind"] == "masked":
        ops = fvsr_lcsa.FlashVSRAttentionOps
        st["op"] = ops.dense if c["mode"] == "dense" else ops.kernel
    elif c["kind"] in ("clip", "windows", "block"):
        st["topk"], st["schedule"] = _clip_topk(c), _schedule(c)
        st["ring"] = fvsr_lcsa.KVRing(1, c["heads"], c["bh"], c["bw"], capacity=4, kv_len=3, dtype=_dtype(c))
        if c["kind"] == "clip":
            st["outs"] = [torch.empty_like(q) for q, _, _ in x["chunks"]]
            st["q_work"] = [torch.empty_like(q) for q, _, _ in x["chunks"]]
        if c["kind"] == "block":
            st["block"] = fvsr_lcsa.DiTBlock(x["W"], c["heads"])
            st["block"].set_context(x["context"])
    return st


def run(state):
    c, st = state["c"], state
    if c["kind"] == "layer":
        s, qs = c["bh"] * c["bw"], c["q_frames"] // 2
        q, k, v = st["q"], st["k"], st["v"]
        if c["api"] == "mask":
            mask, probs, kidx, kcnt = fvsr_lcsa.draft_block_mask_and_probs(q, k, c["heads"], qs, s, st["local"], st["topk"])
            o = fvsr_lcsa.kernel_block_attention(q, k, v, mask, c["heads"], out=st["out"])
            return dict(mask=mask, probs=probs, kidx=kidx, kcnt=kcnt, o=o)
        _, _, kidx, kcnt = fvsr_lcsa.draft_block_mask_and_probs(q, k, c["heads"], qs, s, st["local"], st["topk"],
                                                                want_mask=False, want_probs=False)
        o = fvsr_lcsa.block_sparse_attention(q, k, v, kidx, kcnt, c["heads"], out=st["out"])
        return dict(kidx=kidx, kcnt=kcnt, o=o)
    if c["kind"] == "masked":
        return st["op"](st["q"], st["k"], st["v"], st["mask"], c["heads"])
    h, w = 8 * c["bh"], 8 * c["bw"]
    if c["kind"] == "epilogue":
        return fvsr_lcsa.qkv_epilogue(st["q"], st["k"], st["v"], 2 * c["slices"], h, w, c["heads"], 6, st["wq"], st["wk"])
    ring, outs = st["ring"], []
    ring.reset()
    for i, (n, t0) in enumerate(st["schedule"]):
        if c["kind"] == "clip":
            q, k, v = st["chunks"][i]
            o, _, _ = ring.layer_call_qkv(0, q, k, v, n, t0, st["wq"], st["wk"], st["local"], st["topk"],
                                          out=st["outs"][i], q_work=st["q_work"][i])
        elif c["kind"] == "windows":
            q, k, v = st["chunks"][i]
            qw = fvsr_lcsa.window_partition(q, 2 * n, h, w)
            o, _, _ = ring.layer_call(0, qw, k, v, n, n, st["local"], st["topk"], layout=fvsr_lcsa.LAYOUT_GRID)
            o = fvsr_lcsa.window_reverse(o, 2 * n, h, w)
        else:
            x = st["xs"][i].clone()   # the block updates its tokens in place
            o = st["block"].forward(ring, 0, x, st["t_mod"], n, t0, st["local"], st["topk"])
        outs.append(o)
    return outs


# ---------------------------------------------------------------------------------------------------------------
# the same results in 64 bits (storage roundings of the declared dtype where the path stores a tensor)
# ---------------------------------------------------------------------------------------------------------------
def _select64(q, k, heads, q_slices, s, local, topk):
    """(mask, probs) over blocks from float64 tokens in window order."""
    def pool(x):
        n = -(-x.shape[0] // D)
        tail = x.shape[0] - (n - 1) * D
        p = torch.zeros((n, x.shape[1]), dtype=x.dtype, device=x.device)
        p[:n - 1] = x[:(n - 1) * D].reshape(n - 1, D, -1).mean(1)
        p[n - 1] = x[(n - 1) * D:].sum(0) / tail
        return p.reshape(n, heads, D).permute(1, 0, 2).contiguous()
    pq, pk = pool(q), pool(k)
    nq, nk = pq.shape[1], pk.shape[1]
    see = local.to(q.device)[torch.arange(nq, device=q.device) % s][:, torch.arange(nk, device=q.device) % s]
    probs = torch.stack([torch.softmax((pq[h] @ pk[h].T.contiguous() / math.sqrt(D)).masked_fill(~see, -math.inf), -1)
                         for h in range(heads)])
    rows = probs.reshape(heads, q_slices, -1)
    n = rows.shape[-1]
    thr = rows.sort(-1, descending=True).values[..., min(n - 1, topk)]
    return (rows > thr[..., None]).reshape(heads, nq, nk), probs


def _attend64(q, k, v, heads, mask):
    """softmax(q k^T / sqrt(128)) v per head over the kept blocks; rows that keep none give zeros."""
    o = torch.zeros_like(q)
    step = 16 * D
    for h in range(heads):
        ch = slice(h * D, (h + 1) * D)
        kh, vh = k[:, ch].T.contiguous(), v[:, ch].contiguous()
        for r in range(0, q.shape[0], step):
            rows = torch.arange(r, min(q.shape[0], r + step), device=q.device) // D
            keep = mask[h][rows][:, torch.arange(k.shape[0], device=q.device) // D]
            sc = (q[r:r + step, ch] @ kh / math.sqrt(D)).masked_fill(~keep, -math.inf)
            m = sc.max(-1, keepdim=True).values
            p = torch.exp(sc - torch.where(torch.isinf(m), torch.zeros_like(m), m))
            l = p.sum(-1, keepdim=True)
            o[r:r + step, ch] = (p @ vh) / torch.where(l > 0, l, torch.ones_like(l))
    return o


def _epilogue64(x, wt, heads, f, h, w, t0, dt):
    def rnd(y):
        return y.to(dt).double()
    n = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    if dt == torch.float32:
        return _partition(_rope(n * wt.double(), heads, f, h, w, t0), f, h, w)
    return _partition(rnd(_rope(rnd(rnd(n) * wt.double()), heads, f, h, w, t0)), f, h, w)


def _linear64(x, W, name, dt, gelu=False):
    y = x @ W[name + "_weight"].double().T.contiguous() + W[name + "_bias"].double()
    if gelu:
        y = 0.5 * y * (1 + torch.tanh(math.sqrt(2 / math.pi) * (y + 0.044715 * y ** 3)))
    return y.to(dt).double()


def exact(case, seed):
    c, x, dt = case, _inputs(case, seed), _dtype(case)
    heads = c["heads"]

    def rnd(y):
        return y.to(dt).double()
    if c["kind"] == "masked":
        return _attend64(x["q"].double(), x["k"].double(), x["v"].double(), heads, x["mask"] > 0.5)
    h, w = 8 * c["bh"], 8 * c["bw"]
    s = c["bh"] * c["bw"]
    if c["kind"] == "epilogue":
        f = 2 * c["slices"]
        q, k = (_epilogue64(x[n].double(), x["w" + n], heads, f, h, w, 6, dt) for n in ("q", "k"))
        return q, k, _partition(x["v"].double(), f, h, w)
    local = _windows(c["bh"], c["bw"], c["local"])
    if c["kind"] == "layer":
        q, k, v = (x[n].double() for n in "qkv")
        mask, probs = _select64(q, k, heads, c["q_frames"] // 2, s, local, _layer_topk(c))
        o = _attend64(q, k, v, heads, mask)
        if c["api"] == "mask":
            return dict(mask=None, probs=probs, kidx=None, kcnt=None, o=o)
        return dict(kidx=None, kcnt=None, o=o)
    topk, outs, kc, vc = _clip_topk(c), [], None, None
    if c["kind"] == "block":
        W, C = x["W"], heads * D
        mod = rnd(W["modulation"].double() + x["t_mod"].double())

        def norm(y, wt=None, b=None):
            y = (y - y.mean(-1, keepdim=True)) * torch.rsqrt(y.var(-1, unbiased=False, keepdim=True) + EPS)
            return rnd(y if wt is None else y * wt.double() + b.double())

        def modulate(y, scale, shift):
            return rnd(rnd(norm(y) * rnd(1 + scale)) + shift)

        def rms(y, wt):
            return rnd(rnd(y * torch.rsqrt(y.square().mean(-1, keepdim=True) + EPS)) * wt.double())
        ctx = x["context"].double()
        ck, cv = rms(_linear64(ctx, W, "cross_k", dt), W["cross_norm_k_weight"]), _linear64(ctx, W, "cross_v", dt)
    for i, (n, t0) in enumerate(_schedule(c)):
        f = 2 * n
        if c["kind"] == "windows":
            q, k, v = (_partition(y.double(), f, h, w) for y in x["chunks"][i])
        else:
            if c["kind"] == "clip":
                q, k, v = (y.double() for y in x["chunks"][i])
                wq, wk = x["wq"], x["wk"]
            else:
                xi = x["xs"][i].double()
                a = modulate(xi, mod[1], mod[0])
                q, k, v = (_linear64(a, W, p, dt) for p in "qkv")
                wq, wk = W["norm_q_weight"], W["norm_k_weight"]
            q, k = (_epilogue64(y, wt, heads, f, h, w, t0, dt) for y, wt in ((q, wq), (k, wk)))
            v = _partition(v, f, h, w)
        kc, vc = (y if z is None else torch.cat([z, y]) for y, z in ((k, kc), (v, vc)))
        mask, _ = _select64(q, kc, heads, n, s, local, topk)
        o = _reverse(_attend64(q, kc, vc, heads, mask), f, h, w)
        if kc.shape[0] > 3 * s * D:
            kc, vc = kc[s * D:], vc[s * D:]
        if c["kind"] == "block":
            xi = rnd(xi + rnd(mod[2] * _linear64(rnd(o), W, "o", dt)))
            q = rms(_linear64(norm(xi, W["norm3_weight"], W["norm3_bias"]), W, "cross_q", dt), W["cross_norm_q_weight"])
            every = torch.ones((heads, -(-q.shape[0] // D), -(-ck.shape[0] // D)), dtype=torch.bool, device="cuda")
            xi = rnd(xi + _linear64(rnd(_attend64(q, ck, cv, heads, every)), W, "cross_o", dt))
            y = _linear64(modulate(xi, mod[4], mod[3]), W, "ffn1", dt, gelu=True)
            o = rnd(xi + rnd(mod[5] * _linear64(y, W, "ffn2", dt)))
        outs.append(o)
    return outs
