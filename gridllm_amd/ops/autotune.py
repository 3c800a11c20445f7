"""Per-shape GEMM dispatch autotuner.

For each decode projection shape (M, N, K) the engine will hit, measure
hipBLASLt (torch F.linear) against the in-house GEMMs at several tilings, and
cache the winner. ops.linear() then dispatches through the table — never slower
than the library, faster where a hand-written kernel wins; shapes that were not
timed go by rule. (PyTorch TunableOp only tunes WITHIN hipBLASLt; measured +2%
on these shapes — profiles/r01_decode_profile.md.)
"""

from __future__ import annotations

import functools
import time
from typing import Optional

import torch
import torch.nn.functional as F
from torch.autograd import forward_ad

from gridllm_amd import ops
from gridllm_amd.ops import hip_ops
from gridllm_amd.ops.reference import SWIGLU, Glu
from gridllm_amd.utils.logging import get_logger

log = get_logger("autotune")

# (m, n, k) -> ("blas",) | ("rows",) | ("ours", splitk) |
# ("tile", rows, cols, splitk) | ("wide", shape, whole tiles)
_CHOICE: dict[tuple[int, int, int], tuple] = {}
# the same with f32 results (a vocabulary's scores), which not all shapes have
_CHOICE_F32: dict[tuple[int, int, int], tuple] = {}
# of products whose parts of K the next kernel adds up (linear_parts,
# linear_rmsnorm): timed with one behind them, so not what linear does best
_CHOICE_JOINED: dict[tuple[int, int, int], tuple] = {}
# gate/up projection with fused SwiGLU (n = 2F interleaved rows):
# (m, n, k) -> ("blas",) | ("rows",) | ("tile", rows, cols, splitk) |
# ("wide", shape, whole tiles)
_CHOICE_GU: dict[tuple[int, int, int], tuple] = {}
_BF16, _transformed = torch.bfloat16, torch._C._are_functorch_transforms_active
_most_rows = 1 << 24            # of a choice by rule; more ones' are timed alone
_CALLS = 128                    # of a timing, at most
_SPLITK_CANDIDATES = (0, 2, 4, 6, 8, 12, 16, 24, 32)


def _copies(size: int, room: float) -> int:
    """Copies of a weight of `size` bytes, 2 GB of them if that is 128 or less: each
    call of a timing reads its own, and as little of it is in the Infinity Cache (256
    MB) as of a model's. (Loads past the caches leave there what is in it: of 640 MB
    that they read in turn two fifths, and the other kernels' loads nothing.) With less
    than 4 GB left, behind the KV cache, 24 and 640 MB: not to fail for want of
    memory."""
    most, total = (_CALLS, 2 << 30) if room >= 4 << 30 else (24, 640 << 20)
    return min(most, max(2, total // max(1, size)))


def _weights(n: int, k: int, device) -> list[torch.Tensor]:
    room = float("inf")
    if device.type == "cuda":
        room = torch.cuda.mem_get_info(device)[0] + torch.cuda.memory_reserved(
            device) - torch.cuda.memory_allocated(device)
    w = torch.randn(n, k, device=device).to(torch.bfloat16) * 0.1
    return [w] + [w.clone() for _ in range(_copies(n * k * 2, room) - 1)]


def _time_fn(fn, ws, limit: float = float("inf")) -> float:
    """Time fn(w) over the weight's copies, so W streams from HBM, not the
    256 MB Infinity Cache — an L3-warm measurement picks kernels that lose
    in-situ (decode reads 6+ GB of weights per step; nothing stays in L3). The
    calls are captured, as a decode step is: launched one by one from here, a
    kernel of less than 10 us takes as long as its launch. Once for what takes
    more than limit, else the best of three."""
    fn(ws[0])
    flush = torch.empty(512 << 20, dtype=torch.uint8, device=ws[0].device)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for w in ws:
            fn(w)
    best = float("inf")
    for _ in range(3):
        flush.fill_(1)
        torch.cuda.synchronize()
        t0 = time.monotonic()
        graph.replay()
        torch.cuda.synchronize()
        best = min(best, (time.monotonic() - t0) / len(ws))
        if best > limit:
            break
    return best


def _run(c: tuple, x: torch.Tensor, w: torch.Tensor,
         glu: Optional[Glu] = None) -> torch.Tensor:
    """x @ w.T by a choice; with glu, of an interleaved gate/up weight and its
    gated unit."""
    fuse = glu is not None
    unit = glu or SWIGLU
    if c[0] == "rows":
        return hip_ops.gemm_rows(x, w, fuse_swiglu=fuse, glu=unit)
    if c[0] == "tile":
        return hip_ops.gemm_tile(x, w, *c[1:], fuse_swiglu=fuse, glu=unit)
    if c[0] == "wide":
        return hip_ops.gemm_wide(x, w, *c[1:], fuse_swiglu=fuse, glu=unit)
    if c[0] == "ours":
        return hip_ops.gemm_skinny(x, w, splitk=c[1])
    out = F.linear(x, w)
    return hip_ops.swiglu_il(out, glu=unit) if fuse else out


def _run_f32(c: tuple, x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    if c[0] == "tile" and c[3] == 1:
        return hip_ops.gemm_tile_f32(x, w, *c[1:3])
    if c[0] == "wide":
        return hip_ops.gemm_wide(x, w, *c[1:], f32=True)
    return _run(c, x, w).float()


def _fit(x: torch.Tensor, w: torch.Tensor) -> Optional[tuple[int, int, int]]:
    """(M, N, K) of x [M, K] @ w [N, K]^T if the kernels here read both as
    F.linear would: bf16 matrices that fit each other, dense and aligned, without
    a forward-mode tangent or a torch.func transform, which pass a kernel by."""
    xs = x.shape
    if len(xs) != 2 or xs[0] > _most_rows:
        return None
    if x.dtype is not _BF16 or w.dtype is not _BF16 or _transformed() or \
            forward_ad._current_level >= 0 or x.device != w.device:
        return None
    ws = w.shape
    if len(ws) != 2 or xs[1] != ws[1] or not ws[0] or \
            not ws[1] or (x.data_ptr() | w.data_ptr()) & 15 or \
            not x.is_contiguous() or not w.is_contiguous():
        return None
    return xs[0], ws[0], ws[1]


@functools.lru_cache(maxsize=4096)
def _rule(m: int, n: int, k: int, fuse: bool = False, whole: bool = False,
          f32: bool = False) -> tuple:
    """The choice for sizes that were not timed. gemm_rows has no second kernel,
    but every block reads all of x, and takes all of K by itself: it is the faster
    one for w of up to 20 MB with up to 4 rows and up to 10 MB with 16, while K is
    short (against gemm_tile, us: 2048 x 2048, one row 5.7, 7.0, 16 rows 7.2, 7.6; 3072 x
    3072, one row 6.7, 7.9, 16 rows 9.9, 8.3; 5120 x 3072, one row 11.1, 9.7; 896 x
    4864, one row 8.3, 7.0; 2048 x 8192 13.0, 10.7; of a second kernel that is there
    anyway gemm_tile's have 1 us). It takes a gated unit's two columns at half the rate
    (9728 x 896, one row 7.8, 6.3)."""
    if m > 256:
        return hip_ops.gemm_plan(m, n, k, fuse, whole, f32) or ("blas",)
    rows = hip_ops.gemm_rows_fits(m, n, k, fuse)
    few, short = (10_000_000, 4096) if m <= 4 else (5_000_000, 3072)
    if rows and not fuse and k <= short and n * k <= few:
        return ("rows",)
    tiling = hip_ops.gemm_tiling(m, n, k, fuse)
    if tiling is not None:
        return ("tile", *tiling)
    return ("rows",) if rows and m <= 4 else ("blas",)


def _tune(x: torch.Tensor, n: int, glu: Optional[Glu] = None,
          f32: bool = False, joined: bool = False) -> tuple:
    """The fastest for x and a weight of n rows; f32: with a result of that; joined:
    with a norm behind it, which adds up the parts of K that there are (and stands for
    the other kernels that do).

    What reads w through the Infinity Cache, the library or tiles of several blocks of
    rows, is taken if it is 5 % faster: it pushes out what other kernels find there
    (decode of 256 rows, 4 layers of llama3.2:3b, 3072 x 3072 by the library, 1 us faster
    alone: 861 -> 915 us; of 82 rows, qwen2.5:1.5b, 1536 x 8960 by two blocks of 64 rows
    instead of one of 96: 2103 -> 2142)."""
    global _most_rows
    m, k = x.shape
    _most_rows = max(_most_rows, m)
    ws = _weights(n, k, x.device)
    if joined:
        norm = torch.ones(n, dtype=torch.bfloat16, device=x.device)
        resid = torch.zeros(m, n, dtype=torch.bfloat16, device=x.device)

    def call(c: tuple, w: torch.Tensor):
        if joined:
            return _run_joined(c, x, w, norm, 1e-5, resid)
        return _run_f32(c, x, w) if f32 else _run(c, x, w, glu)

    def time_of(c: tuple, limit: float = float("inf")) -> float:
        return _time_fn(lambda w: call(c, w), ws, limit)
    best: tuple = ("blas",)
    t_best = 1.05 * time_of(best)
    tried: list[tuple] = [("tile", *t) for t in hip_ops.gemm_tilings(
        m, n, k, glu is not None)]
    if m > 256 or (f32 and m > 128):
        tried += [("wide", *t) for t in hip_ops.gemm_wide_tilings(
            m, n, k, glu is not None, f32)]
    if hip_ops.gemm_rows_supported(x, ws[0], glu is not None):
        tried.append(("rows",))
    if not tried and glu is None and hip_ops.gemm_skinny_supported(m, n, k):
        tried = [("ours", sk) for sk in _SPLITK_CANDIDATES
                 if sk <= max(1, k // 256)]
    for c in tried:
        through = c[0] == "tile" and not hip_ops.gemm_tile_once(
            m, n, k, c[1], c[3])
        try:
            t = time_of(c, 1.3 * t_best) * (1.05 if through else 1)
        except RuntimeError as e:           # one that cannot run is no choice
            log.logger.warning("gemm choice %s of %s failed: %s", c,
                               (m, n, k), e)
            continue
        if t < t_best * (1 if best == ("blas",) else 0.98):   # a real margin
            t_best = t
            best = c
    return best


def tune_shape(m: int, n: int, k: int, device, f32: bool = False,
               joined: bool = False) -> tuple:
    key, table = (m, n, k), _CHOICE_F32 if f32 else \
        _CHOICE_JOINED if joined else _CHOICE
    if key not in table:
        x = torch.randn(m, k, device=device).to(torch.bfloat16) * 0.1
        table[key] = _tune(x, n, f32=f32, joined=joined)
    return table[key]


def tune_gateup(m: int, n: int, k: int, device) -> tuple:
    """Tune the interleaved gate/up projection (n = 2F rows): library GEMM
    + interleaved-SwiGLU pass vs the fused-epilogue kernels."""
    key = (m, n, k)
    if key not in _CHOICE_GU:
        x = torch.randn(m, k, device=device).to(torch.bfloat16) * 0.1
        _CHOICE_GU[key] = _tune(x, n, SWIGLU)
    return _CHOICE_GU[key]


def linear_gateup(x: torch.Tensor, w_il: torch.Tensor, glu: Glu = SWIGLU,
                  whole: bool = False) -> torch.Tensor:
    """Fused gate/up projection + gated linear unit on an INTERLEAVED weight:
    returns [M, F] activated, through the tuned table or by rule. whole: as in
    linear, and the unit of more than 256 rows is that of the products rounded."""
    fit = _fit(x, w_il)
    c = ("blas",) if fit is None else _timed(_CHOICE_GU, fit, whole) or \
        _rule(*fit, True, whole)
    return _run(c, x, w_il, glu)


def _timed(table: dict, fit: tuple[int, int, int], whole: bool
           ) -> Optional[tuple]:
    """The choice that was timed for these sizes, if it is one for `whole`: decode
    batches are timed, with K in parts too, and a prompt may have as many rows."""
    c = table.get(fit)
    return None if whole and c and fit[0] > 256 and c[0] not in (
        "blas", "wide") else c


def choice(m: int, n: int, k: int) -> Optional[tuple[str, int]]:
    key = (m, n, k)
    return _CHOICE.get(key) or _CHOICE_JOINED.get(key)


def _choose(x: torch.Tensor, w: torch.Tensor, whole: bool = False,
            f32: bool = False, joined: bool = False) -> Optional[tuple]:
    """Choice for x @ w.T (f32: a result of that; joined: if the next kernel adds up
    its parts), None for what is not a GPU product of bf16 rows."""
    if not x.is_cuda or (torch.is_grad_enabled() and
                         (x.requires_grad or w.requires_grad)):
        return None
    fit = _fit(x, w)
    if fit is None:
        return None
    if f32:
        return _CHOICE_F32.get(fit) or _rule(*fit, f32=True)
    whole = whole and fit[0] > 256
    return (joined and _timed(_CHOICE_JOINED, fit, whole)) or \
        _timed(_CHOICE, fit, whole) or _rule(*fit, False, whole)


def choice_of(m: int, w: torch.Tensor, fuse: bool = False) -> Optional[tuple]:
    """What linear_parts and linear_rmsnorm (fuse: linear_gateup) run dense aligned
    bf16 rows [m, K] and w by, if that is one of the kernels here."""
    if m > _most_rows or w.dtype is not _BF16 or _transformed() or \
            forward_ad._current_level >= 0 or w.dim() != 2 or \
            not w.is_contiguous() or w.data_ptr() & 15 or not w.numel():
        return None
    key = (m, *w.shape)
    c = (_CHOICE_GU.get(key) if fuse else _CHOICE_JOINED.get(key) or _CHOICE.get(key)
         ) or _rule(*key, fuse)
    return c if c[0] in ("rows", "tile", "wide") else None


def linear(x: torch.Tensor, w: torch.Tensor, whole: bool = False
           ) -> torch.Tensor:
    """Dispatch x @ w.T (GPU bf16 2-D x only) through the tuned table or by
    rule. whole: more than 256 rows' products have their sums over K whole and in
    order, as the library's are where it does not cut K itself (see
    gl_gemm_plan)."""
    c = _choose(x, w, whole)
    return F.linear(x, w) if c is None else _run(c, x, w)


def linear_f32(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """linear(x, w).float(): a vocabulary's scores."""
    c = _choose(x, w, f32=True)
    return F.linear(x, w).float() if c is None else _run_f32(c, x, w)


def linear_parts(x: torch.Tensor, w: torch.Tensor, whole: bool = False
                 ) -> torch.Tensor:
    """linear(x, w), or its f32 partial sums [parts, M, N] if K is in parts, for
    post_norm, join_norm and rope_kv."""
    c = _choose(x, w, whole, joined=True)
    if c is not None and c[0] == "tile" and c[3] > 1 and w.shape[1] > 64:
        return hip_ops.gemm_tile_parts(x, w, *c[1:])
    return F.linear(x, w) if c is None else _run(c, x, w)


def linear_rmsnorm(x: torch.Tensor, w: torch.Tensor, weight: torch.Tensor,
                   eps: float, residual: torch.Tensor
                   ) -> tuple[torch.Tensor, torch.Tensor]:
    """(rmsnorm(y) * weight, y) of y = x @ w.T + residual. A product with its K
    in parts leaves adding them up to the norm."""
    c = _choose(x, w, joined=True)
    if c is None:
        return ops.rmsnorm(F.linear(x, w), weight, eps, residual=residual)
    return _run_joined(c, x, w, weight, eps, residual)


def _run_joined(c: tuple, x: torch.Tensor, w: torch.Tensor,
                weight: torch.Tensor, eps: float, residual: torch.Tensor
                ) -> tuple[torch.Tensor, torch.Tensor]:
    if c[0] == "tile" and c[3] > 1 and \
            w.shape[1] > 64 and w.shape[0] % 8 == 0 and \
            residual.dtype == weight.dtype == torch.bfloat16 and \
            residual.is_contiguous() and weight.is_contiguous():
        return hip_ops.gemm_tile_rmsnorm(x, w, *c[1:], weight, eps, residual)
    return ops.rmsnorm(_run(c, x, w), weight, eps, residual=residual)


def tune_model_shapes(model, buckets) -> None:
    """Pre-tune every decode GEMM shape for the given batch buckets. The
    model lists its plain projections and its gate/up projections as (n, k), and those
    of the plain ones whose parts of K the next kernel adds up."""
    shapes, gu_shapes = model.gemm_shapes()
    joined = model.joined_shapes()
    t0 = time.monotonic()
    for m in buckets:
        for n, k in shapes:             # (the vocabulary's scores are f32)
            f32 = n == model.spec.vocab
            tune_shape(m, n, k, model.device, f32, not f32 and (n, k) in joined)
        for n, k in gu_shapes:
            if getattr(model, "gateup_il", False):
                tune_gateup(m, n, k, model.device)
            else:
                tune_shape(m, n, k, model.device)
    picked = [*_CHOICE.values(), *_CHOICE_F32.values(), *_CHOICE_JOINED.values()]
    log.performance("gemm autotune done", shapes=len(picked),
                    ours=sum(1 for c in picked if c[0] != "blas"),
                    ms=int((time.monotonic() - t0) * 1000))
