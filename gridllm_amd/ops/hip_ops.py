"""ctypes binding to the gfx950 kernel library (libgridllm_hip.so).

Launches go onto torch's current HIP stream, so the whole decode step is
hipGraph-capturable via torch.cuda.CUDAGraph (= hipGraph on ROCm).
Fails LOUDLY if the library is missing on a GPU machine — there is no
silent eager fallback on the GPU path.
"""

from __future__ import annotations

import array
import ctypes
import functools
import os
from typing import Optional

import torch

from gridllm_amd.ops.reference import SWIGLU, Glu

_LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)),
                         "libgridllm_hip.so")
_lib: Optional[ctypes.CDLL] = None


class HipExtensionMissing(RuntimeError):
    pass


def _load() -> ctypes.CDLL:
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(_LIB_PATH):
        raise HipExtensionMissing(
            f"GridLLM HIP kernel library not found at {_LIB_PATH}. "
            "Build it with: python -m gridllm_amd.ops.build "
            "(this is required on GPU machines; there is no eager fallback).")
    lib = ctypes.CDLL(_LIB_PATH)
    c_vp, c_i, c_l, c_f = ctypes.c_void_p, ctypes.c_int, ctypes.c_long, ctypes.c_float
    lib.gl_rmsnorm.argtypes = [c_vp, c_vp, c_vp, c_vp, c_vp, c_vp, c_l, c_i, c_f]
    lib.gl_rmsnorm.restype = c_i
    lib.gl_rmsnorm_parts.argtypes = [c_vp] * 3 + [c_i] + [c_vp] * 3 + [
        c_i, c_i, c_f]
    lib.gl_rmsnorm_parts.restype = c_i
    lib.gl_decode_start.argtypes = [c_vp] * 9 + [c_i] * 3
    lib.gl_decode_start.restype = c_i
    lib.gl_advance_lengths.argtypes = [c_vp] * 3 + [c_i] * 2
    lib.gl_advance_lengths.restype = c_i
    lib.gl_prompt_positions.argtypes = [c_vp] * 3 + [c_i] * 4
    lib.gl_prompt_positions.restype = c_i
    lib.gl_prompt_end.argtypes = [c_vp] * 3 + [c_i] * 3
    lib.gl_prompt_end.restype = c_i
    lib.gl_prompts_end.argtypes = [c_vp] * 5 + [c_i, c_i] + [c_vp] * 3 + [
        c_i, c_i]
    lib.gl_prompts_end.restype = c_i
    lib.gl_embed_norm.argtypes = [c_vp] * 6 + [c_l, c_i, c_i, c_f]
    lib.gl_embed_norm.restype = c_i
    lib.gl_rope.argtypes = [c_vp, c_vp, c_vp, c_vp, c_vp, c_vp, c_i, c_i, c_i, c_i]
    lib.gl_rope.restype = c_i
    lib.gl_swiglu.argtypes = [c_vp, c_vp, c_vp, c_l, c_i, c_f, c_f, c_f, c_f]
    lib.gl_swiglu.restype = c_i
    lib.gl_rope_kv.argtypes = [c_vp, c_vp, c_i] + [c_vp] * 8 + [c_i] * 5
    lib.gl_rope_kv.restype = c_i
    lib.gl_prompt_layer.argtypes = [c_vp, c_vp, c_f, c_f]
    lib.gl_prompt_layer.restype = c_i
    lib.gl_kv_append.argtypes = [c_vp, c_vp, c_vp, c_vp, c_vp, c_vp, c_i, c_i, c_i, c_i]
    lib.gl_kv_append.restype = c_i
    lib.gl_attn_decode.argtypes = [c_vp, c_vp, c_vp, c_vp, c_vp, c_vp, c_vp,
                                   c_vp, c_vp, c_i, c_i, c_i, c_i, c_i, c_i, c_f]
    lib.gl_attn_decode.restype = c_i
    lib.gl_rope_attn_decode.argtypes = [c_vp] * 3 + [c_i] + [c_vp] * 10 + [
        c_i] * 6 + [c_f]
    lib.gl_rope_attn_decode.restype = c_i
    lib.gl_gemm_skinny.argtypes = [c_vp, c_vp, c_vp, c_vp, c_vp,
                                   c_i, c_i, c_i, c_i, c_i]
    lib.gl_gemm_skinny.restype = c_i
    lib.gl_gemm_rows.argtypes = [c_vp] * 4 + [c_i] * 4 + [c_f] * 4
    lib.gl_gemm_rows.restype = c_i
    lib.gl_gemm_tile.argtypes = [c_vp] * 5 + [c_i] * 8 + [c_f] * 4
    lib.gl_gemm_tile.restype = c_i
    lib.gl_gemm_wide.argtypes = [c_vp] * 4 + [c_i] * 6 + [c_f] * 4
    lib.gl_gemm_wide.restype = c_i
    lib.gl_gemm_plan.argtypes = [c_i] * 5 + [c_vp]
    lib.gl_gemm_plan.restype = c_i
    lib.gl_gemm_tile_once.argtypes = [c_i] * 5
    lib.gl_gemm_tile_once.restype = c_i
    lib.gl_prefill_place.argtypes = [c_i] * 3 + [c_vp]
    lib.gl_prefill_place.restype = c_i
    lib.gl_attn_prefill.argtypes = [c_vp, c_vp, c_vp, c_vp, c_vp, c_i, c_i,
                                    c_i, c_i, c_i, c_i, c_i, c_i, c_f]
    lib.gl_attn_prefill.restype = c_i
    lib.gl_attn_prefill_batch.argtypes = [c_vp, c_vp, c_vp, c_vp, c_vp, c_vp,
                                          c_i, c_i, c_i, c_i, c_i, c_f]
    lib.gl_attn_prefill_batch.restype = c_i
    lib.gl_swiglu_il.argtypes = [c_vp, c_vp, c_vp, c_l, c_i,
                                 c_f, c_f, c_f, c_f]
    lib.gl_sample_gumbel.argtypes = [c_vp] * 10 + [c_i] * 4
    lib.gl_sample_gumbel.restype = c_i
    lib.gl_sample_slots.argtypes = [c_vp] * 9 + [c_i] * 4
    lib.gl_sample_slots.restype = c_i
    lib.gl_swiglu_il.restype = c_i
    lib.gl_device_sync.argtypes = []
    lib.gl_device_sync.restype = c_i
    _lib = lib
    return lib


def available() -> bool:
    return os.path.exists(_LIB_PATH)


def _stream() -> int:
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device())


def _check(rc: int, op: str) -> None:
    if rc != 0:
        raise RuntimeError(f"HIP kernel {op} failed with code {rc}")


# Addresses stay plain numbers, which the declared signatures convert: a prompt
# of a few layers and tokens is bound by what its launches cost the host (4 us
# each less than with ctypes objects and torch's Stream object).
def _ptr(t: Optional[torch.Tensor]) -> Optional[int]:
    return None if t is None else t.data_ptr()


# Debug validation (the sanitizer analog for a ctypes-bound kernel layer):
# GRIDLLM_VALIDATE=1 makes every wrapper range-check its index tensors BEFORE
# launching — a device sync per call, debug only. (It catches a slot_t that
# overflows, as a graph's warm-up at bucket >= max_seq once did.)
_VALIDATE = os.environ.get("GRIDLLM_VALIDATE", "") == "1"


def _check_range(name: str, t: torch.Tensor, hi: int) -> None:
    if not _VALIDATE or t.numel() == 0:
        return
    mx, mn = int(t.max().item()), int(t.min().item())
    if mn < 0 or mx >= hi:
        raise RuntimeError(
            f"GRIDLLM_VALIDATE: {name} out of range [{mn},{mx}] vs [0,{hi})")


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float,
            residual: Optional[torch.Tensor] = None,
            residual_out: Optional[torch.Tensor] = None,
            out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """y = rmsnorm(x [+ residual]) * weight; bf16. x: [..., H]."""
    lib = _load()
    h = x.shape[-1]
    n = x.numel() // h
    if out is None:
        out = torch.empty_like(x)
    _check(lib.gl_rmsnorm(_stream(), _ptr(out), _ptr(x), _ptr(weight),
                          _ptr(residual), _ptr(residual_out), n, h,
                          eps), "rmsnorm")
    return out


def _check_ints(op: str, slot_map: torch.Tensor, *by_slot: torch.Tensor
                ) -> None:
    """Dense int32 vectors on one GPU, those by slot of one length. (A slot that
    they have not ends the program, as an index out of bounds does in torch.)"""
    slots = by_slot[0].shape[0]
    for t in (slot_map, *by_slot):
        if not (t.is_cuda and t.device == slot_map.device and t.dim() == 1
                and t.dtype == torch.int32 and t.is_contiguous()):
            raise ValueError(f"{op}: int32 vectors on one GPU")
    if any(t.shape[0] != slots for t in by_slot):
        raise ValueError(f"{op}: lengths by slot differ")


_ROWS_ORDERED = 1024           # rows that decode_start puts in order


def _decode_start(seq_lens: torch.Tensor, slot_map: torch.Tensor,
                  rope_off: Optional[torch.Tensor], smax: int, ordered: bool,
                  what: str) -> tuple[torch.Tensor, Optional[torch.Tensor]]:
    """[lengths | cache places | rotary positions | key counts] (without rope_off the
    lengths alone), and the rows in order."""
    b = slot_map.shape[0]
    _check_ints(what, slot_map, seq_lens, *(() if rope_off is None else (rope_off,)))
    _check_range(what + ".slot_map", slot_map, seq_lens.shape[0])
    out = torch.empty(1 if rope_off is None else 4, b, dtype=torch.int32,
                      device=seq_lens.device)
    rows = torch.empty(b, 4, dtype=torch.int32, device=seq_lens.device) \
        if ordered and 1 < b <= _ROWS_ORDERED else None
    _check(_load().gl_decode_start(
        _stream(), _ptr(out[0]), *((None,) * 3 if rope_off is None else map(
            _ptr, out[1:])), _ptr(rows), _ptr(seq_lens), _ptr(rope_off),
        _ptr(slot_map), b, seq_lens.shape[0], smax), what)
    return out, rows


def decode_positions(seq_lens: torch.Tensor, slot_map: torch.Tensor,
                     rope_off: torch.Tensor, smax: int
                     ) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Start of a decode step over slots slot_map [B] int32 of seq_lens: cache
    places slot * smax + length, rotary positions length + rope_off[slot], and
    key counts length + 1, all int32 [B]."""
    out, _ = _decode_start(seq_lens, slot_map, rope_off, smax, False,
                           "decode_positions")
    return out[1], out[2], out[3]


def decode_start(seq_lens: torch.Tensor, slot_map: torch.Tensor,
                 rope_off: torch.Tensor, smax: int) -> tuple:
    """decode_positions, and rows [B, 4] {row, keys, slot, rotary position}, the
    longest first, for attn_decode (None for a single row, or more than are put in order)."""
    out, rows = _decode_start(seq_lens, slot_map, rope_off, smax, True,
                              "decode_start")
    return out[1], out[2], out[3], rows


def advance_lengths(seq_lens: torch.Tensor, slot_map: torch.Tensor) -> None:
    """End of a decode step: the lengths of slots slot_map [B] int32, one or more
    rows each, go up by one a row."""
    _check_ints("advance_lengths", slot_map, seq_lens)
    _check_range("advance_lengths.slot_map", slot_map, seq_lens.shape[0])
    _check(_load().gl_advance_lengths(
        _stream(), _ptr(seq_lens), _ptr(slot_map), slot_map.shape[0],
        seq_lens.shape[0]), "advance_lengths")


def prompt_positions(t: int, slot: int, start: int, seq_lens: torch.Tensor,
                     smax: int) -> tuple[torch.Tensor, torch.Tensor]:
    """Positions start .. start + t - 1 and cache places slot * smax + those,
    int32 [t], of a slot of seq_lens."""
    if not (0 <= slot < seq_lens.shape[0]):
        raise IndexError(f"slot {slot} of {seq_lens.shape[0]}")
    out = torch.empty(2, t, dtype=torch.int32, device=seq_lens.device)
    _check(_load().gl_prompt_positions(
        _stream(), _ptr(out[0]), _ptr(out[1]), slot, start, t, smax),
        "prompt_positions")
    return out[0], out[1]


def prompt_end(t: int, slot: int, start: int, seq_lens: torch.Tensor,
               rope_off: torch.Tensor) -> None:
    """Sets the slot's length to start + t, and its rope_off to 0 if start is
    0."""
    if not (0 <= slot < min(seq_lens.shape[0], rope_off.shape[0])):
        raise IndexError(f"slot {slot} of {seq_lens.shape[0]}")
    _check(_load().gl_prompt_end(_stream(), _ptr(seq_lens), _ptr(rope_off),
                                 slot, start, t), "prompt_end")


def prompts_end(seq_lens: torch.Tensor, rope_off: torch.Tensor,
                slots: torch.Tensor, lens: torch.Tensor,
                x: Optional[torch.Tensor], lasts: torch.Tensor
                ) -> Optional[torch.Tensor]:
    """Sets the lengths of slots [B] int32 to lens, their rope_off to 0, and
    returns x[lasts] (x [n, H] bf16), if there is an x."""
    _check_ints("prompts_end", slots, seq_lens, rope_off)
    _check_ints("prompts_end", slots, lens, lasts)
    b = slots.shape[0]
    if lens.shape != (b,) or (x is not None and not (
            x.dtype == torch.bfloat16 and x.dim() == 2 and x.is_contiguous()
            and x.device == slots.device and x.data_ptr() % 16 == 0)):
        raise ValueError("prompts_end: lengths and rows [B], dense bf16 x")
    _check_range("prompts_end.slots", slots, seq_lens.shape[0])
    out = None if x is None else torch.empty(b, x.shape[1], dtype=x.dtype,
                                             device=x.device)
    _check(_load().gl_prompts_end(
        _stream(), _ptr(seq_lens), _ptr(rope_off), _ptr(slots), _ptr(lens), b,
        seq_lens.shape[0], _ptr(out), _ptr(x), _ptr(lasts),
        0 if x is None else x.shape[0], 0 if x is None else x.shape[1]),
        "prompts_end")
    return out


def decode_lengths(seq_lens: torch.Tensor,
                   slot_map: torch.Tensor) -> torch.Tensor:
    """The lengths of slots slot_map [B] int32."""
    return _decode_start(seq_lens, slot_map, None, 0, False, "decode_lengths")[0][0]


def decode_ordered(seq_lens: torch.Tensor, slot_map: torch.Tensor) -> tuple:
    """decode_lengths, and decode_start's rows."""
    out, rows = _decode_start(seq_lens, slot_map, None, 0, True, "decode_ordered")
    return out[0], rows


def embed_norm(tokens: torch.Tensor, emb: torch.Tensor, weight: torch.Tensor,
               eps: float) -> tuple[torch.Tensor, torch.Tensor]:
    """x = emb[tokens] [n, H] and rmsnorm(x) * weight; tokens [n] int64, counted
    from the end if negative. Others than the table has end the program, as they
    do in torch's lookup."""
    n, h = tokens.shape[0], emb.shape[1]
    if not (tokens.is_cuda and tokens.device == emb.device == weight.device and
            tokens.dtype == torch.int64 and weight.shape == (h,)):
        raise ValueError("embed_norm: tokens [n] int64, emb [vocab, H] and "
                         "weight [H] on one GPU")
    _check_range("embed_norm.tokens", tokens, emb.shape[0])
    x = torch.empty(n, h, dtype=emb.dtype, device=emb.device)
    y = torch.empty_like(x)
    _check(_load().gl_embed_norm(
        _stream(), _ptr(x), _ptr(y), _ptr(emb), _ptr(tokens), _ptr(weight), n,
        h, emb.shape[0], eps), "embed_norm")
    return x, y


def rope(q: torch.Tensor, k: torch.Tensor, cos: torch.Tensor,
         sin: torch.Tensor, pos: torch.Tensor) -> None:
    """In-place rotary embedding. q: [T,Hq,D], k: [T,Hk,D] bf16;
    cos/sin: [S,D/2] f32; pos: [T] int32."""
    lib = _load()
    t, hq, d = q.shape
    hk = k.shape[1]
    _check(lib.gl_rope(_stream(), _ptr(q), _ptr(k), _ptr(cos), _ptr(sin),
                       _ptr(pos), t, hq, hk, d), "rope")


def rope_kv(qkv: torch.Tensor, kcache: torch.Tensor, vcache: torch.Tensor,
            cos: torch.Tensor, sin: torch.Tensor, pos: torch.Tensor,
            slot: torch.Tensor, hq: int, hk: int, d: int,
            bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Fused RoPE + KV write from the raw QKV GEMM output.
    qkv: [N, (hq+2*hk)*d] bf16 (row-dense), or f32 partial sums of it [parts, N,
    ..] (d % 16 == 0); bias: [(hq+2*hk)*d] bf16, added to it; returns roped q [N,
    hq, d]."""
    lib = _load()
    n, width = qkv.shape[-2:]
    parts = qkv.shape[0] if qkv.dim() == 3 else 0
    if qkv.dtype != (torch.float32 if parts else torch.bfloat16) or (
            bias is not None and (bias.dtype != torch.bfloat16 or
                                  bias.shape != (width,)
                                  or not bias.is_contiguous())):
        raise ValueError("rope_kv: bf16 rows, or their f32 parts, and a dense "
                         "bf16 bias")
    smax = kcache.shape[2]
    _check_range("rope_kv.slot", slot, kcache.shape[0] * smax)
    _check_range("rope_kv.pos", pos, cos.shape[0])
    q_out = torch.empty(n, hq, d, dtype=torch.bfloat16, device=qkv.device)
    _check(lib.gl_rope_kv(_stream(), _ptr(qkv), parts, _ptr(q_out),
                          _ptr(kcache), _ptr(vcache), _ptr(cos), _ptr(sin),
                          _ptr(pos), _ptr(slot), _ptr(bias), n, hq, hk, d, smax),
           "rope_kv")
    return q_out


def swiglu(gateup: torch.Tensor, out: Optional[torch.Tensor] = None,
           glu: Glu = SWIGLU) -> torch.Tensor:
    """out[n,F] = glu(gateup[:, :F], gateup[:, F:]); gateup: [..., 2F] bf16."""
    lib = _load()
    f2 = gateup.shape[-1]
    f = f2 // 2
    n = gateup.numel() // f2
    if out is None:
        out = torch.empty(gateup.shape[:-1] + (f,), dtype=gateup.dtype,
                          device=gateup.device)
    _check(lib.gl_swiglu(_stream(), _ptr(out), _ptr(gateup), n, f, *glu),
           "swiglu")
    return out


def kv_append(kcache: torch.Tensor, vcache: torch.Tensor, k_new: torch.Tensor,
              v_new: torch.Tensor, slot: torch.Tensor) -> None:
    """Append rows into [B,Hk,Smax,D] caches. k_new: [N,Hk,D]; slot[N]=b*Smax+pos."""
    lib = _load()
    n, hk, d = k_new.shape
    smax = kcache.shape[2]
    _check_range("kv_append.slot", slot, kcache.shape[0] * smax)
    _check(lib.gl_kv_append(_stream(), _ptr(kcache), _ptr(vcache), _ptr(k_new),
                            _ptr(v_new), _ptr(slot), n, hk, d, smax), "kv_append")


_MAX_SPLIT = 64                # what the combining kernel takes


def decode_splits(blocks: int, keys: int) -> int:
    """Into how many parts decode attention splits rows of up to `keys` keys,
    `blocks` of them counting their kv heads: up to six workgroups a CU, none
    for less than 128 keys. A row of fewer keys takes as many as it needs; the
    others end at once, and the combining kernel takes longer. The number is odd:
    workgroups go round the XCDs and their shader engines, which are powers of
    two, and with an even one the first parts of all rows, all that short rows
    have, would meet on some of them.
    Measured in us, 8 kv heads of 128, in a cache of 8192: one row of 8000 keys 26
    in 6 parts, 18 in 12, 15 in 32, 20 in 64; 24 rows of 50 to 300 9 in one, 13 in
    7 and 9, 20 in 8, of 1000 to 6000 84 in one, 78 in 8 and 9; 64 rows of 50 to
    300 12 in one, 16 in 3, 24 in 4, of 500 to 2000 59 in one, 60 in 3; 96 rows of
    50 to 300 17 in one, 23 in 2 and 3, of 100 to 8000 323 in one, 292 in 2, 270 in
    3; 256 rows of up to 384 47 in one, 62 in 2."""
    parts = min(1536 // max(1, blocks) | 1, 31 if blocks <= 16 else 15,
                (keys + 127) // 128)
    return max(1, parts - 1 | 1)


def _check_rows(op: str, rows: Optional[torch.Tensor], b: int) -> None:
    """decode_start's order is of a step's b rows, by which kernels find them."""
    if rows is not None and not (rows.shape == (b, 4) and rows.dtype == torch.int32
                                 and rows.is_contiguous()):
        raise ValueError(f"{op}: rows [{b}, 4], dense int32")


def attn_decode(q: torch.Tensor, kcache: torch.Tensor, vcache: torch.Tensor,
                seqlen: torch.Tensor, scale: float, nsplit: int = 0,
                slot_map: Optional[torch.Tensor] = None,
                ws: Optional[torch.Tensor] = None,
                out: Optional[torch.Tensor] = None,
                rows: Optional[torch.Tensor] = None) -> torch.Tensor:
    """GQA decode attention. q/out: [B,Hq,D]; caches [Slots,Hk,Smax,D];
    seqlen [B] int32; slot_map [B] int32 maps batch row -> cache slot
    (None -> identity). nsplit=0 -> auto. rows: decode_start's, which say the
    same as seqlen and slot_map."""
    lib = _load()
    b, hq, d = q.shape
    hk, smax = kcache.shape[1], kcache.shape[2]
    if nsplit <= 0:
        nsplit = decode_splits(b * hk, smax)
    nsplit = min(nsplit, _MAX_SPLIT)
    _check_range("attn_decode.seqlen", seqlen, smax + 1)
    if slot_map is not None:
        _check_range("attn_decode.slot_map", slot_map, kcache.shape[0])
    _check_rows("attn_decode", rows, b)
    if out is None:
        out = torch.empty_like(q)
    if nsplit > 1 and ws is None:
        g = hq // hk
        ws = torch.empty(b * hk * g * nsplit * (d + 2), dtype=torch.float32,
                         device=q.device)
    _check(lib.gl_attn_decode(_stream(), _ptr(out), _ptr(q), _ptr(kcache),
                              _ptr(vcache), _ptr(seqlen), _ptr(slot_map),
                              _ptr(rows), _ptr(ws), b, hq, hk, d, smax, nsplit,
                              scale), "attn_decode")
    return out


def rope_attn_decode(qkv: torch.Tensor, kcache: torch.Tensor, vcache: torch.Tensor,
                     cos: torch.Tensor, sin: torch.Tensor, pos: torch.Tensor,
                     slot: torch.Tensor, seqlen: torch.Tensor, hq: int, scale: float,
                     slot_map: torch.Tensor, bias: Optional[torch.Tensor] = None,
                     rows: Optional[torch.Tensor] = None, nsplit: int = 0
                     ) -> torch.Tensor:
    """rope_kv and attn_decode of a decode step in one kernel, which makes a row's
    queries, key and value where they are read (sizes and addresses that it does not
    take: in two). slot: place slot_map * Smax + seqlen - 1 of each row's key; a row
    of no keys gives zeros and writes none.

    In us, two kernels and one, rows of a product, and its sums in 5 parts: 24 heads
    of 128 over 8, one row of 900 keys 12.5 and 9.9, 13.5 and 11.3; 24 of up to 6000
    71.1 and 67.3, 70.7 and 69.6; 256 of up to 384 52.9 and 48.0, 56.8 and 52.9. Each
    part of a row makes the queries anew: sums of 4 heads or more of a kv head are left
    to two kernels if there are more than two blocks a CU (16 rows of up to 3000, 32
    heads of 64 over 8, 1664 blocks: 27.9, 28.5; 64 of up to 2000, 12 of 128 over 2, 37.9,
    40.0; 8 of up to 3000, 496 blocks, 20.1, 19.3)."""
    b, d = qkv.shape[-2], kcache.shape[3]
    hk, smax = kcache.shape[1:3]
    _check_rows("rope_attn_decode", rows, b)
    if vcache.shape != kcache.shape or any(
            t.dim() != 1 or t.shape[0] < b for t in (pos, seqlen, slot_map)):
        raise ValueError("rope_attn_decode: caches of one shape, and a position, a "
                         "length and a slot of each row")
    parts = qkv.shape[0] if qkv.dim() == 3 else 0
    nsplit = min(nsplit if nsplit > 0 else decode_splits(b * hk, smax), _MAX_SPLIT)
    many = parts and nsplit > 1 and hq // hk >= 4 and b * hk * nsplit > 512
    dense = [qkv, kcache, vcache, cos, sin] + ([] if bias is None else [bias])
    if many or not (b and d in (64, 128) and hq and hq % hk == 0 and hq // hk <= 8 and
            qkv.dtype == (torch.float32 if parts else torch.bfloat16) and
            kcache.dtype == vcache.dtype == torch.bfloat16 and
            cos.dtype == sin.dtype == torch.float32 and
            cos.shape[1] * 2 == d == sin.shape[1] * 2 and
            qkv.shape[-1] == (hq + 2 * hk) * d and
            (bias is None or (bias.dtype == torch.bfloat16 and
                              bias.shape == qkv.shape[-1:])) and
            all(t.is_contiguous() and t.data_ptr() % 16 == 0 for t in dense) and
            all(t.dtype == torch.int32 and t.is_contiguous()
                for t in (pos, seqlen, slot_map))):
        q = rope_kv(qkv, kcache, vcache, cos, sin, pos, slot, hq, hk, d, bias)
        return attn_decode(q, kcache, vcache, seqlen, scale, nsplit, slot_map,
                           rows=rows)
    _check_range("rope_attn_decode.seqlen", seqlen, smax + 1)
    _check_range("rope_attn_decode.slot_map", slot_map, kcache.shape[0])
    _check_range("rope_attn_decode.pos", pos, cos.shape[0])
    out = torch.empty(b, hq, d, dtype=torch.bfloat16, device=qkv.device)
    ws = torch.empty(b * hq * nsplit * (d + 2), dtype=torch.float32,
                     device=qkv.device) if nsplit > 1 else None
    _check(_load().gl_rope_attn_decode(
        _stream(), _ptr(out), _ptr(qkv), parts, _ptr(kcache), _ptr(vcache),
        _ptr(cos), _ptr(sin), _ptr(pos), _ptr(bias), _ptr(seqlen), _ptr(slot_map),
        _ptr(rows), _ptr(ws), b, hq, hk, d, smax, nsplit, scale),
        "rope_attn_decode")
    return out


def attn_prefill_cache(q: torch.Tensor, kcache: torch.Tensor,
                       vcache: torch.Tensor, slot: int, s_total: int,
                       causal_offset: int, scale: float,
                       out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Flash-style MFMA GQA prefill straight off the slot cache.
    q/out: [T,Hq,D] bf16; caches [Slots,Hk,Smax,D]; keys 0..s_total-1 of
    `slot` attendable, causally masked at position causal_offset+t."""
    lib = _load()
    t, hq, d = q.shape
    hk, smax = kcache.shape[1], kcache.shape[2]
    if out is None:
        out = torch.empty_like(q)
    _check(lib.gl_attn_prefill(_stream(), _ptr(out), _ptr(q), _ptr(kcache),
                               _ptr(vcache), t, hq, hk, d, smax, slot,
                               s_total, causal_offset,
                               scale), "attn_prefill")
    return out


def attn_prefill_cache_batch(q: torch.Tensor, kcache: torch.Tensor,
                             vcache: torch.Tensor, meta: torch.Tensor,
                             scale: float,
                             out: Optional[torch.Tensor] = None
                             ) -> torch.Tensor:
    """Varlen batched MFMA GQA prefill: many fresh sequences packed in q
    ([sum(T_i), Hq, D]), one launch per layer. meta: [ntiles, 4] int32 on
    device, rows {q_off, len, slot, q0} (built once per admission batch by
    LlamaModel.forward_prefill_batch and reused across layers)."""
    lib = _load()
    hq, d = q.shape[1], q.shape[2]
    hk, smax = kcache.shape[1], kcache.shape[2]
    ntiles = meta.shape[0]
    if out is None:
        out = torch.empty_like(q)
    if _VALIDATE:
        _check_range("meta.slot", meta[:, 2], kcache.shape[0])
        _check_range("meta.len", meta[:, 1] - 1, smax)
        _check_range("meta.q_off", meta[:, 0], q.shape[0])
    _check(lib.gl_attn_prefill_batch(_stream(), _ptr(out), _ptr(q),
                                     _ptr(kcache), _ptr(vcache), _ptr(meta),
                                     ntiles, hq, hk, d, smax,
                                     scale),
           "attn_prefill_batch")
    return out


def gemm_skinny_supported(m: int, n: int, k: int) -> bool:
    return m <= 256 and n % 64 == 0 and k % 32 == 0


def gemm_skinny(x: torch.Tensor, w: torch.Tensor,
                out: Optional[torch.Tensor] = None,
                splitk: int = 0) -> torch.Tensor:
    """out[M,N] = x[M,K] @ w[N,K]^T, bf16, M<=256 (decode projections).
    Streams w once into MFMA fragments; split-K sized to fill
    256 CUs with f32 partial slabs + combine."""
    lib = _load()
    m, k = x.shape
    n = w.shape[0]
    ntiles = max(1, n // 64)
    if splitk <= 0:
        # target ~2048 blocks; kslice is a multiple of the kernel's 256-k
        # panel and every split is useful (no idle blocks)
        splitk = max(1, min(k // 256, 2048 // ntiles))
    kslice = ((k + splitk - 1) // splitk + 255) // 256 * 256
    splitk = (k + kslice - 1) // kslice
    if out is None:
        out = torch.empty(m, n, dtype=x.dtype, device=x.device)
    ws = None
    if splitk > 1:
        ws = torch.empty(splitk * m * n, dtype=torch.float32, device=x.device)
    _check(lib.gl_gemm_skinny(_stream(), _ptr(out), _ptr(ws), _ptr(x), _ptr(w),
                              m, n, k, splitk, kslice), "gemm_skinny")
    return out


def gemm_rows_fits(m: int, n: int, k: int, fuse_swiglu: bool = False) -> bool:
    """Whether gemm_rows has these sizes."""
    return (0 < m <= 16 and 0 < n < 65536 and k > 0 and k % 32 == 0
            and n % (128 if fuse_swiglu else 16) == 0)


def gemm_rows_supported(x: torch.Tensor, w: torch.Tensor,
                        fuse_swiglu: bool = False) -> bool:
    """Whether gemm_rows takes x [M, K] @ w [N, K]^T."""
    return (x.shape[1] == w.shape[1]
            and gemm_rows_fits(x.shape[0], *w.shape, fuse_swiglu)
            and x.is_contiguous() and w.is_contiguous()
            and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16
            and (x.data_ptr() | w.data_ptr()) % 16 == 0)


def gemm_rows(x: torch.Tensor, w: torch.Tensor,
              out: Optional[torch.Tensor] = None, fuse_swiglu: bool = False,
              glu: Glu = SWIGLU) -> torch.Tensor:
    """out[M,N] = x[M,K] @ w[N,K]^T, bf16, M <= 16: blocks of 16 columns over
    all of K, without a workspace. fuse_swiglu: as in gemm_tile."""
    lib = _load()
    m, k = x.shape
    n = w.shape[0]
    if out is None:
        out = torch.empty(m, n // 2 if fuse_swiglu else n,
                          dtype=x.dtype, device=x.device)
    _check(lib.gl_gemm_rows(_stream(), _ptr(out), _ptr(x), _ptr(w), m, n, k,
                            1 if fuse_swiglu else 0, *glu), "gemm_rows")
    return out


_TILE_ROWS = (32, 64, 96, 128, 160, 192, 256)


def _tile_grid(m: int, n: int, k: int, fuse_swiglu: bool,
               narrow: bool = False) -> list[tuple[int, int, int]]:
    """(rows, columns, blocks of these) of gemm_tile that are worth a thought:
    rows in as few blocks as can be, or twice as many, or, with few columns, in
    up to 4. narrow: columns in 48 too, which more than 64 rows have."""
    if m < 1 or k % 64 or (fuse_swiglu and n % 128):
        return []
    out = []
    base = -(-m // 128)
    for blocks in sorted({-(-m // r) for r in _TILE_ROWS}):
        rows = next((r for r in _TILE_ROWS if r >= -(-m // blocks)), 0)
        for cols in (64, 128) if fuse_swiglu else (
                48, 64, 96, 128)[not narrow or rows <= 64:]:
            tiles = n // cols * blocks
            if n % cols == 0 and rows and (
                    blocks <= base or (blocks <= 4 and tiles <= 256)):
                out.append((rows, cols, tiles))
    return out


def gemm_tilings(m: int, n: int, k: int,
                 fuse_swiglu: bool = False) -> list[tuple[int, int, int]]:
    """(rows, columns, K parts) worth trying for gemm_tile: K in as many parts,
    of 128 or more, as give each of the 256 CUs a block, or in half as many; and 256
    columns, if these are still more tiles than CUs."""
    out = set()
    rows = next((r for r in _TILE_ROWS if r >= m), 256)
    if 0 < m <= 160 and n % 256 == 0 and n > 65536 and k % 64 == 0 and \
            not fuse_swiglu:
        out.add((rows, 256, 1))
    for rows, cols, tiles in _tile_grid(m, n, k, fuse_swiglu, True):
        most = max(1, min(256 // tiles, k // 128))
        for parts in (most, (most + 1) // 2, 1 if k <= 4096 else most):
            out.add((rows, cols, parts))
    return sorted(out)


@functools.lru_cache(maxsize=4096)
def gemm_tiling(m: int, n: int, k: int,
                fuse_swiglu: bool = False) -> Optional[tuple[int, int, int]]:
    """The tiling of gemm_tile for sizes that were not timed, or None if they are
    better left to the library.

    Up to 64 rows: one block of rows, or two of 32 if the weights are few, and 64
    columns as long as that is a block a CU or less, K in parts of 512 or more for
    the others (us, the library's time behind it: 48 rows of 2048 x 8192 13.0, 15.6; 896
    x 4864 8.3 in two blocks and 9 parts, 9.2 in one, 11 in 18 parts, 17.3; 2048 x 2048
    8.0, in one block 8.8, 11.6; 5120 x 3072 12.6, in two 13.9, 17.6; 128256 x 2048 107,
    141).
    Up to 256: what _tile_us says of a block a CU or less, with K whole, in the
    parts that then fill the CUs, or in half as many. It takes 1.003 of the best
    choice's time in the mean, 1.07 at most, .70 of the library's (246 sizes). More
    blocks than CUs are a library product's sizes (17920 x 1536, 256 rows: 22.9 us,
    22.2), but for the gated unit that it would need a second kernel for."""
    if not 0 < m <= 256 or n < 1 or k < 1 or k % 64 or (
            fuse_swiglu and n % 128):
        return None
    if m <= 64:
        cols = 128 if n // 64 > 256 and n % 128 == 0 else 64
        if n % cols:
            return None
        rows = 32 if m <= 32 or n * k <= 8_000_000 else 64
        tiles = n // cols * (-(-m // rows))
        return rows, cols, max(1, min(256 // tiles, k // 512))
    best, least = None, float("inf")
    for rows, cols, tiles in _tile_grid(m, n, k, fuse_swiglu):
        if tiles > 256:
            continue
        most = max(1, min(256 // tiles, k // 384))
        for parts in sorted({1, (most + 1) // 2, most}):
            us = _tile_us(m, n, k, rows, cols, tiles, parts, fuse_swiglu)
            if us < least:
                best, least = (rows, cols, parts), us
    if best is None and fuse_swiglu:
        return 128 if m <= 128 else 256, 128, 1
    return best


def _tile_us(m: int, n: int, k: int, rows: int, cols: int, tiles: int,
             parts: int, fuse_swiglu: bool = False) -> float:
    """What a tiling takes of gemm_tile's time, in us, beside 3.9 that all have: for
    each round of CUs its start, a CU's loads of its share of K (a row of x half as
    long as one of w, which comes from memory), its products and gated units, and
    with K in parts the second kernel, which reads the partial sums. (Fitted to 5800
    timings of 65 to 1200 rows, 6.4 % standard deviation. gl_gemm_plan has the same for
    more rows; a test holds the two together.)"""
    kslice = -(-(-(-k // parts)) // 64) * 64
    parts = -(-k // kslice)
    us = -(-tiles * parts // 256) * (
        3 + kslice * (rows * 1.42e-5 + cols * 3.2e-5 + rows * cols * 1.09e-7) +
        (rows * cols * 5.8e-5 if fuse_swiglu else 0))
    return us if parts == 1 else us + parts * m * n * 2.4e-6


def gemm_tile(x: torch.Tensor, w: torch.Tensor, rows: int, cols: int,
              splitk: int = 1, out: Optional[torch.Tensor] = None,
              fuse_swiglu: bool = False, glu: Glu = SWIGLU) -> torch.Tensor:
    """out[M,N] = x[M,K] @ w[N,K]^T, bf16, by blocks of rows x cols and one of
    splitk parts of K (f32 partials that a second kernel adds up).
    fuse_swiglu: w rows interleaved [64 gate | 64 up]; returns [M, N/2] =
    glu(gate, up) with no separate activation pass."""
    lib = _load()
    m, k = x.shape
    n = w.shape[0]
    kslice = ((k + splitk - 1) // splitk + 63) // 64 * 64
    splitk = (k + kslice - 1) // kslice
    if out is None:
        out = torch.empty(m, n // 2 if fuse_swiglu else n,
                          dtype=x.dtype, device=x.device)
    ws = None
    if splitk > 1:
        ws = torch.empty(splitk * m * n, dtype=torch.float32, device=x.device)
    _check(lib.gl_gemm_tile(_stream(), _ptr(out), _ptr(ws), _ptr(x), _ptr(w),
                            m, n, k, splitk, kslice, rows, cols,
                            1 if fuse_swiglu else 0, *glu), "gemm_tile")
    return out


def gemm_tile_once(m: int, n: int, k: int, rows: int, splitk: int) -> bool:
    """Whether gemm_tile reads w past the Infinity Cache."""
    kslice = ((k + splitk - 1) // splitk + 63) // 64 * 64
    return _load().gl_gemm_tile_once(m, n, k, rows, kslice) == 1


def gemm_tile_f32(x: torch.Tensor, w: torch.Tensor, rows: int,
                  cols: int) -> torch.Tensor:
    """gemm_tile(...).float(), K in one part, without the bf16 copy."""
    lib = _load()
    m, k = x.shape
    n = w.shape[0]
    out = torch.empty(m, n, dtype=torch.float32, device=x.device)
    _check(lib.gl_gemm_tile(_stream(), None, _ptr(out), _ptr(x), _ptr(w), m, n,
                            k, 1, (k + 63) // 64 * 64, rows, cols, 0,
                            *SWIGLU), "gemm_tile")
    return out


def gemm_tile_parts(x: torch.Tensor, w: torch.Tensor, rows: int, cols: int,
                    splitk: int) -> torch.Tensor:
    """gemm_tile's partial sums, f32 [parts, M, N], for a kernel that adds them
    up itself (and rounds their sum to bf16)."""
    lib = _load()
    m, k = x.shape
    n = w.shape[0]
    kslice = ((k + splitk - 1) // splitk + 63) // 64 * 64
    splitk = (k + kslice - 1) // kslice
    assert splitk > 1
    ws = torch.empty(splitk, m, n, dtype=torch.float32, device=x.device)
    _check(lib.gl_gemm_tile(_stream(), None, _ptr(ws), _ptr(x), _ptr(w), m, n,
                            k, splitk, kslice, rows, cols, 0, *SWIGLU),
           "gemm_tile")
    return ws


def gemm_tile_rmsnorm(x: torch.Tensor, w: torch.Tensor, rows: int, cols: int,
                      splitk: int, weight: torch.Tensor, eps: float,
                      residual: torch.Tensor
                      ) -> tuple[torch.Tensor, torch.Tensor]:
    """gemm_tile with K in parts and the rmsnorm behind it, which adds them up:
    (rmsnorm(y) * weight, y) of y = x @ w^T + residual [M, N]."""
    m, n = x.shape[0], w.shape[0]
    assert residual.shape == (m, n) and weight.shape == (n,)
    assert residual.is_contiguous() and weight.is_contiguous()
    ws = gemm_tile_parts(x, w, rows, cols, splitk)
    y, total = torch.empty_like(residual), torch.empty_like(residual)
    _check(_load().gl_rmsnorm_parts(
        _stream(), _ptr(y), _ptr(ws), ws.shape[0], _ptr(weight),
        _ptr(residual), _ptr(total), m, n, eps), "rmsnorm_parts")
    return y, total


WIDE_SHAPES = ((256, 256), (192, 192), (256, 192), (192, 128), (192, 256))


def gemm_wide_tilings(m: int, n: int, k: int, fuse_swiglu: bool = False,
                      f32: bool = False) -> list[tuple[int, int]]:
    """(shape, whole tiles) worth trying for gemm_wide: those that give 64 CUs a
    tile, with the last round of CUs whole or in halves."""
    if k % 64 or k < 256 or n % (128 if fuse_swiglu else 8) or \
            max(m, n) * k * 2 > 0xe0000000:
        return []
    out = []
    for i, (rows, cols) in enumerate(WIDE_SHAPES):
        if (0 < i < 4) if fuse_swiglu or f32 else i == 4:
            continue
        tiles = -(-m // rows) * -(-n // cols)
        if 64 <= tiles < 1 << 24:
            out += [(i, t) for t in sorted({tiles, tiles // 256 * 256}
                                           if i == 0 else {tiles})]
    return out


@functools.lru_cache(maxsize=4096)
def gemm_plan(m: int, n: int, k: int, fuse_swiglu: bool = False,
              whole: bool = False, f32: bool = False) -> Optional[tuple]:
    """("tile", rows, columns, parts) or ("wide", shape, whole tiles) for a
    product of more than 256 rows that was not timed, None if it is better left
    to the library (see gl_gemm_plan). whole: K in one part, in order, and a gated
    unit on rounded products. f32: for a result of that."""
    if not (0 < m < 1 << 24 and 0 < n < 1 << 24 and 0 < k < 1 << 20):
        return None
    plan = (ctypes.c_int * 4)()
    _check(_load().gl_gemm_plan(m, n, k, 1 if fuse_swiglu else 2 if f32 else 0,
                                whole, ctypes.addressof(plan)),
           "gemm_plan")
    if plan[0] == 1:
        return ("tile", *plan[1:4])
    return ("wide", plan[1], plan[2]) if plan[0] else None


def gemm_wide(x: torch.Tensor, w: torch.Tensor, shape: int, full: int,
              fuse_swiglu: bool = False, glu: Glu = SWIGLU,
              f32: bool = False) -> torch.Tensor:
    """out[M,N] = x[M,K] @ w[N,K]^T, bf16, by tiles of WIDE_SHAPES[shape] that
    blocks of one a CU take in turn; behind the first `full` of them (shape 0)
    tiles of half the rows. fuse_swiglu: as in gemm_tile. f32: the result, rounded
    to bf16, as f32."""
    m, k = x.shape
    n = w.shape[0]
    out = torch.empty(m, n // 2 if fuse_swiglu else n, device=x.device,
                      dtype=torch.float32 if f32 else x.dtype)
    _check(_load().gl_gemm_wide(
        _stream(), out.data_ptr(), x.data_ptr(), w.data_ptr(), m, n, k, shape,
        full, 1 if fuse_swiglu else 2 if f32 else 0, *glu), "gemm_wide")
    return out


def gemm_proj_supported(m: int, n: int, k: int) -> bool:
    if not (64 < m <= 512 and k % 64 == 0):
        return False
    bn = 64 if m > 256 else 128
    return n % bn == 0


def gemm_proj(x: torch.Tensor, w: torch.Tensor,
              out: Optional[torch.Tensor] = None,
              splitk: int = 0, fuse_swiglu: bool = False,
              mtiles: int = 0, glu: Glu = SWIGLU) -> torch.Tensor:
    """gemm_tile with a tiling by rule, for up to 512 rows: blocks of 128 columns
    (64 from 257 rows on) and all rows, or 1 / mtiles of up to 2048; splitk 0
    takes the number of parts that covers the 256 CUs."""
    m, k = x.shape
    n = w.shape[0]
    cols = 64 if m > 256 and mtiles <= 1 else 128
    if k % 64 or n % cols or m > (2048 if mtiles > 1 else 512) or \
            (fuse_swiglu and cols == 64):
        raise RuntimeError(f"gemm_proj: {m} x {n} x {k} is not supported")
    blocks = mtiles if mtiles > 1 else -(-m // 256)
    rows = next((r for r in _TILE_ROWS if r >= -(-m // blocks)), 256)
    tiles = max(1, n // cols) * blocks
    if splitk <= 0:
        splitk = max(1, min(k // 256, (256 + tiles - 1) // tiles))
    return gemm_tile(x, w, rows, cols, splitk, out, fuse_swiglu, glu)


def gemm_proj_wide_supported(m: int, n: int, k: int) -> bool:
    return 64 < m <= 256 and n % 256 == 0 and k % 64 == 0


def gemm_proj_wide(x: torch.Tensor, w: torch.Tensor,
                   out: Optional[torch.Tensor] = None,
                   splitk: int = 0) -> torch.Tensor:
    """gemm_proj for up to 256 rows and a multiple of 256 columns."""
    if x.shape[0] > 256 or w.shape[0] % 256:
        raise RuntimeError("gemm_proj_wide: shape not supported")
    return gemm_proj(x, w, out, splitk)


def swiglu_il(gu: torch.Tensor, out: Optional[torch.Tensor] = None,
              glu: Glu = SWIGLU) -> torch.Tensor:
    """Gated linear unit over an interleaved [.., 2F] gate/up activation (128-col
    groups [64 gate | 64 up]) — the library-GEMM path for interleaved
    gateup weights."""
    lib = _load()
    n = gu.numel() // gu.shape[-1]
    f = gu.shape[-1] // 2
    if out is None:
        out = torch.empty(*gu.shape[:-1], f, dtype=gu.dtype, device=gu.device)
    _check(lib.gl_swiglu_il(_stream(), _ptr(out), _ptr(gu),
                            n, f, *glu), "swiglu_il")
    return out


def sample_gumbel(logits: torch.Tensor, keys: torch.Tensor,
                  temps: torch.Tensor) -> torch.Tensor:
    """Fused Gumbel-argmax token pick (no-filter sampling path):
    out[b] = argmax_v logits[b,v]/temps[b] + gumbel(splitmix64(v ^ keys[b])),
    key==0 rows greedy. logits [B,V] f32, keys [B] i64, temps [B] f32 ->
    [B] i32. Two launches replacing the eager ~15-op torch chain
    (engine/sampler.py::sample_batch_vectorized)."""
    return _sample(logits, keys, temps)


def sample_gumbel_slots(logits: torch.Tensor, slots: torch.Tensor,
                        temps: torch.Tensor, seeds: torch.Tensor,
                        draws: torch.Tensor, nongreedy: torch.Tensor,
                        marks: Optional[torch.Tensor] = None) -> torch.Tensor:
    """sample_gumbel with the rows' parameters by slot (slots [B] i64, all
    different; temps f32, seeds, draws, nongreedy i64): the keys are made in the
    kernel, and the slots' draws advance by one. A slot that there is not ends the
    program, as an index out of bounds does in torch. marks: i64 [slots, 16] of zeros,
    which stay zeros between calls and belong to the slots as their draws do (a slot is
    in one call at a time): one launch instead of two. (Rows with one slot get that
    slot's key, too, but slowly.)"""
    return _sample(logits, None, temps, slots, seeds, draws, nongreedy, marks)


def _sample(logits, keys, temps, slots=None, seeds=None, draws=None,
            nongreedy=None, marks=None) -> torch.Tensor:
    lib = _load()
    b, v = logits.shape
    f32, i64, dev, n = torch.float32, torch.int64, logits.get_device(), \
        temps.shape
    if slots is None:
        ok = (keys.dtype is i64 and keys.shape == n == (b,)
              and dev == keys.get_device() and keys.is_contiguous())
    else:
        ok = (slots.dtype is i64 and seeds.dtype is i64 and draws.dtype is i64
              and nongreedy.dtype is i64 and slots.shape == (b,)
              and len(n) == 1 and seeds.shape == n and draws.shape == n
              and nongreedy.shape == n and dev == slots.get_device()
              == seeds.get_device() == draws.get_device()
              == nongreedy.get_device() and slots.is_contiguous()
              and seeds.is_contiguous() and draws.is_contiguous()
              and nongreedy.is_contiguous()
              and (marks is None or (
                  marks.dtype is i64 and marks.shape == (*n, 16)
                  and dev == marks.get_device() and marks.is_contiguous())))
    if not (ok and logits.dtype is f32 and temps.dtype is f32 and dev >= 0
            and dev == temps.get_device() and logits.is_contiguous()
            and temps.is_contiguous()):
        raise ValueError("sample_gumbel: f32 logits [B, V] and temps, int64 "
                         "keys [B], or slots [B] and vectors by slot of one "
                         "length, dense and on one GPU")
    if slots is not None:
        _check_range("sample_gumbel.slots", slots, n[0])
    # four blocks a CU, of 2048 elements (what its waves have at a time) or more
    segments = max(1, min(1024 // max(1, b), -(-v // 2048), 64))
    out = torch.empty(b, dtype=torch.int32, device=logits.device)
    if marks is not None and v:
        _check(lib.gl_sample_slots(
            _stream(), out.data_ptr(), logits.data_ptr(), temps.data_ptr(),
            slots.data_ptr(), seeds.data_ptr(), draws.data_ptr(),
            nongreedy.data_ptr(), marks.data_ptr(), b, v, segments, n[0]),
            "sample_slots")
        return out
    ws = torch.empty(b * segments, dtype=i64, device=logits.device)
    at = (keys.data_ptr(), temps.data_ptr(), None, None, None, None) \
        if slots is None else (
            None, temps.data_ptr(), slots.data_ptr(), seeds.data_ptr(),
            draws.data_ptr(), nongreedy.data_ptr())
    _check(lib.gl_sample_gumbel(
        _stream(), out.data_ptr(), ws.data_ptr(), logits.data_ptr(), *at, b, v,
        segments, n[0]), "sample_gumbel")
    return out


_LAYER_KINDS = {"rows": 0, "tile": 1, "wide": 2}


def layer_choice(c: tuple) -> tuple[int, int, int, int]:
    """A product's choice for prompt_layer."""
    return (_LAYER_KINDS[c[0]], *c[1:], *(0,) * (4 - len(c)))


def prompt_layer(fields: list, scale: float, eps: float) -> None:
    """A prompt's layer by one call (the fields of PromptLayer, addresses and
    numbers, in their order)."""
    data = array.array("q", fields)
    assert len(fields) == 50
    _check(_load().gl_prompt_layer(_stream(), data.buffer_info()[0], scale, eps),
           "prompt_layer")


def device_sync() -> None:
    _check(_load().gl_device_sync(), "device_sync")
