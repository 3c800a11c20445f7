"""Pure-PyTorch fp32 reference implementations of every HIP op.

Used (a) as the CPU execution path (no GPU in CI), and (b) as the numerics
oracle the HIP kernels are tested against (tests/test_ops_gpu.py).
"""

from __future__ import annotations

from typing import NamedTuple, Optional, Tuple

import torch


class Glu(NamedTuple):
    """A gated linear unit by its constants: the gate is capped at `limit`,
    the linear part clamped to +-limit and moved by `shift`;
    y = g * sigmoid(alpha * g * (1 + cubic * g^2)) * (u + shift)."""
    alpha: float = 1.0
    limit: float = float("inf")
    shift: float = 0.0
    cubic: float = 0.0


SWIGLU = Glu()


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float,
            residual: Optional[torch.Tensor] = None
            ) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """Returns (y, residual_out). fp32 math, output in x.dtype."""
    z = x.float()
    if residual is not None:
        z = z + residual.float()
    var = z.pow(2).mean(dim=-1, keepdim=True)
    y = z * torch.rsqrt(var + eps) * weight.float()
    res_out = z.to(x.dtype) if residual is not None else None
    return y.to(x.dtype), res_out


def rope_tables(head_dim: int, max_seq: int, theta: float = 500000.0,
                device: str = "cpu") -> Tuple[torch.Tensor, torch.Tensor]:
    """Precomputed cos/sin tables [max_seq, D/2] (f32). Llama-3 theta=5e5."""
    half = head_dim // 2
    inv_freq = 1.0 / (theta ** (torch.arange(0, half, dtype=torch.float32,
                                             device=device) / half))
    t = torch.arange(max_seq, dtype=torch.float32, device=device)
    freqs = torch.outer(t, inv_freq)
    return freqs.cos().contiguous(), freqs.sin().contiguous()


def prompt_positions(t: int, slot: int, start: int, seq_lens: torch.Tensor,
                     smax: int) -> Tuple[torch.Tensor, torch.Tensor]:
    """Positions start .. start + t - 1 and slot * smax + those, of a slot of
    seq_lens."""
    if not (0 <= slot < seq_lens.shape[0]):
        raise IndexError(f"slot {slot} of {seq_lens.shape[0]}")
    pos = torch.arange(start, start + t, dtype=torch.int32,
                       device=seq_lens.device)
    return pos, pos + slot * smax


def prompt_end(t: int, slot: int, start: int, seq_lens: torch.Tensor,
               rope_off: torch.Tensor) -> None:
    """Sets the slot's length, and its rope_off to 0 if start is 0."""
    seq_lens[slot] = start + t
    if start == 0:
        rope_off[slot] = 0


def prompts_end(seq_lens: torch.Tensor, rope_off: torch.Tensor,
                slots: torch.Tensor, lens: torch.Tensor,
                x: Optional[torch.Tensor], lasts: torch.Tensor
                ) -> Optional[torch.Tensor]:
    """Sets the lengths of slots [B], their rope_off to 0; x[lasts]."""
    seq_lens[slots.long()] = lens
    rope_off.index_fill_(0, slots.long(), 0)
    return None if x is None else x[lasts.long()]


def decode_positions(seq_lens: torch.Tensor, slot_map: torch.Tensor,
                     rope_off: torch.Tensor, smax: int
                     ) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """(slot * smax + length, length + rope_off[slot], length + 1) of slots
    slot_map [B]."""
    slots = slot_map.long()
    pos = seq_lens[slots]
    return slot_map * smax + pos, pos + rope_off[slots], pos + 1


def advance_lengths(seq_lens: torch.Tensor, slot_map: torch.Tensor) -> None:
    seq_lens.index_add_(0, slot_map.long(),
                        torch.ones_like(slot_map, dtype=seq_lens.dtype))


def rope(q: torch.Tensor, k: torch.Tensor, cos: torch.Tensor,
         sin: torch.Tensor, pos: torch.Tensor
         ) -> Tuple[torch.Tensor, torch.Tensor]:
    """Neox-style (split-half) rotary. q: [T,Hq,D], k: [T,Hk,D]; pos: [T]."""
    def rot(x: torch.Tensor) -> torch.Tensor:
        d = x.shape[-1]
        half = d // 2
        c = cos[pos.long()].unsqueeze(1).float()   # [T,1,half]
        s = sin[pos.long()].unsqueeze(1).float()
        xf = x.float()
        x1, x2 = xf[..., :half], xf[..., half:]
        return torch.cat([x1 * c - x2 * s, x1 * s + x2 * c], dim=-1).to(x.dtype)
    return rot(q), rot(k)


def swiglu(gateup: torch.Tensor, glu: Glu = SWIGLU) -> torch.Tensor:
    f = gateup.shape[-1] // 2
    g = gateup[..., :f].float().clamp(max=glu.limit)
    u = gateup[..., f:].float().clamp(-glu.limit, glu.limit)
    z = glu.alpha * g * (1 + glu.cubic * g * g)
    return (g * torch.sigmoid(z) * (u + glu.shift)
            ).to(gateup.dtype)


def rope_kv(qkv: torch.Tensor, kcache: torch.Tensor, vcache: torch.Tensor,
            cos: torch.Tensor, sin: torch.Tensor, pos: torch.Tensor,
            slot: torch.Tensor, hq: int, hk: int, d: int,
            bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Reference of the fused RoPE+KV-write: slice the QKV GEMM output,
    rope q/k, append k/v to the caches. Returns roped q [N, hq, d]."""
    n = qkv.shape[0]
    if bias is not None:
        qkv = qkv + bias
    q = qkv[:, :hq * d].reshape(n, hq, d)
    k = qkv[:, hq * d:(hq + hk) * d].reshape(n, hk, d)
    v = qkv[:, (hq + hk) * d:].reshape(n, hk, d).contiguous()
    q, k = rope(q.contiguous(), k.contiguous(), cos, sin, pos)
    if hk:
        kv_append(kcache, vcache, k, v, slot)
    return q


def kv_append(kcache: torch.Tensor, vcache: torch.Tensor, k_new: torch.Tensor,
              v_new: torch.Tensor, slot: torch.Tensor) -> None:
    """caches [B,Hk,Smax,D]; k_new [N,Hk,D]; slot[N]=b*Smax+pos."""
    smax = kcache.shape[2]
    b = torch.div(slot.long(), smax, rounding_mode="floor")
    p = slot.long() % smax
    kcache[b, :, p] = k_new
    vcache[b, :, p] = v_new


def attn_decode(q: torch.Tensor, kcache: torch.Tensor, vcache: torch.Tensor,
                seqlen: torch.Tensor, scale: float,
                slot_map: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Single-token GQA attention vs cache, fp32 math.
    q [B,Hq,D], caches [Slots,Hk,Smax,D], seqlen [B] -> out [B,Hq,D]."""
    bsz, hq, d = q.shape
    hk = kcache.shape[1]
    g = hq // hk
    idx = slot_map.long() if slot_map is not None else \
        torch.arange(bsz, device=q.device)
    n = seqlen.long()
    nmax = int(n.max()) if bsz else 0
    if nmax == 0:
        return torch.zeros_like(q)
    kk = kcache[idx, :, :nmax].float()                  # [B,Hk,nmax,D]
    vv = vcache[idx, :, :nmax].float()
    qq = q.float().view(bsz, hk, g, d)
    scores = torch.einsum("bhgd,bhnd->bhgn", qq, kk) * scale
    mask = torch.arange(nmax, device=q.device).view(1, 1, 1, nmax) >= \
        n.view(bsz, 1, 1, 1)
    scores = scores.masked_fill(mask, float("-inf"))
    p = torch.softmax(scores, dim=-1)
    o = torch.einsum("bhgn,bhnd->bhgd", p, vv)
    empty = n == 0                                      # all -inf -> nan
    if bool(empty.any()):
        o[empty] = 0
    return o.reshape(bsz, hq, d).to(q.dtype)


def attn_prefill(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                 scale: float, causal_offset: int = 0) -> torch.Tensor:
    """Causal GQA prefill, fp32 math.
    q [B,T,Hq,D], k/v [B,S,Hk,D] with S >= T; query t attends keys
    <= causal_offset + t (so causal_offset = S - T for cached prefix)."""
    bsz, t, hq, d = q.shape
    s, hk = k.shape[1], k.shape[2]
    g = hq // hk
    qq = q.float().permute(0, 2, 1, 3).view(bsz, hk, g, t, d)
    kk = k.float().permute(0, 2, 1, 3)                 # [B,Hk,S,D]
    vv = v.float().permute(0, 2, 1, 3)
    scores = torch.einsum("bhgtd,bhsd->bhgts", qq, kk) * scale
    idx_t = torch.arange(t, device=q.device).view(t, 1)
    idx_s = torch.arange(s, device=q.device).view(1, s)
    mask = idx_s > (idx_t + causal_offset)
    scores = scores.masked_fill(mask, float("-inf"))
    p = torch.softmax(scores, dim=-1)
    o = torch.einsum("bhgts,bhsd->bhgtd", p, vv)
    return o.view(bsz, hq, t, d).permute(0, 2, 1, 3).contiguous().to(q.dtype)
