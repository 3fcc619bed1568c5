"""Attention in float64 on the device, written without the package: what the GPU tests hold whole outputs against."""
import torch


def masked_attention64(q, k, v, heads, mask, step=64):
    """Yields (head, first token, result) of softmax(q k^T / sqrt(128)) v over ALL keys with the unselected blocks'
    scores at -inf (`blockMaskedAttention`, DiT.swift:279-313), in float64, `step` query blocks at a time; rows that
    select nothing are zeros."""
    block_of_key = torch.arange(k.shape[0], device=k.device) // 128
    for h in range(heads):
        c = slice(h * 128, (h + 1) * 128)
        kt, vh = k[:, c].double().t().contiguous(), v[:, c].double()
        for t in range(0, q.shape[0], step * 128):
            rows = torch.arange(t, min(q.shape[0], t + step * 128), device=q.device) // 128
            keep = (mask[h] > 0.5)[rows][:, block_of_key]
            s = (q[t:t + step * 128, c].double() @ kt / 128 ** 0.5).masked_fill(~keep, -float("inf"))
            yield h, t, torch.softmax(s, -1).nan_to_num(0.0) @ vh


def rel_everywhere(got, q, k, v, heads, mask, step=64):
    """max |got - ref| / max |ref| over the whole output, the largest of the heads; NaN outputs count as infinite."""
    err = torch.zeros(heads, dtype=torch.float64, device=got.device)
    top = torch.zeros_like(err)
    for h, t, ref in masked_attention64(q, k, v, heads, mask, step):
        d = (got[t:t + ref.shape[0], h * 128:(h + 1) * 128].double() - ref).abs().nan_to_num(float("inf"))
        err[h] = torch.maximum(err[h], d.max())
        top[h] = torch.maximum(top[h], ref.abs().max())
    return float((err / top.clamp_min(1e-30)).max())
