"""Pure-PyTorch execution of the layer-list ops on the CPU (no GPU in CI),
function for function the signatures of hip_hybrid, and the description of a
step that both take."""

from __future__ import annotations

from dataclasses import dataclass, field
from typing import Optional

import torch
import torch.nn.functional as F

from gridllm_amd.ops.reference import SWIGLU, Glu, swiglu

PAGE = 64


@dataclass
class ChunkPortions:
    """Prompt portions of a step as talking-heads attention takes them, for one
    chunk size. The keys that they see are laid out in `pages` pages:
    items    [*, 4] {page number, slot, page to write, rows} per page
    tiles16  [*, 8] {first token, length, first page, first row, start, page
             number of that page} per 16 rows of a portion, and
    tiles128 per 128 rows; long spans of keys first
    span     keys that the longest of these sees, about
    """
    pages: int
    span: int
    items: torch.Tensor
    tiles16: torch.Tensor
    tiles128: torch.Tensor


@dataclass
class StepMeta:
    """The tokens of one step: `nd` decode rows (one token of a sequence
    each), then prompt portions. Everything but nd and max_len lives on the
    device.

    tiles      [*, 8] {first token, length, slot, first row, start} per 128
               rows of a portion (attention)
    chunks     [*, 4] {first token, length, portion} per 64 tokens, and
    chunk_segs [*, 4] {slot, start, first chunk, chunks} per portion (mLSTM)
    segs       [*, 4] {first token, length, slot, start} of every entry, decode
               rows included; what the token-by-token paths walk. None: all
               entries are decode rows.

    Latent attention takes the first `absorbed` tokens (decode rows and short
    portions) one by one against the cached latents; for the portions behind
    them it expands their sequences' latents, gathered into `lat_rows` rows:
    lat_items  [*, 4] {page number, slot, first gathered row, rows of the page
               + 256 * rows to write} per page
    lat_tiles  [*, 8] {first token, length, first gathered row, first row,
               start} per 128 rows of a portion
    whole      products of more than 256 rows keep their sums over K whole (of
               steps with first tokens, or portions of prompts)
    rows       [n, 4] {row, keys, slot, ..} of a step of decode rows alone, the
               longest first: the order in which attention takes them. None:
               that of the step
    state_bytes  what all of the model's recurrent layers hold for a sequence, 0
               if that is not known
    """
    nd: int
    pos: torch.Tensor            # [n] int32
    slot: torch.Tensor           # [n] int32
    table: torch.Tensor          # [slots, pages per slot] int32
    max_len: int                 # bound of any sequence's length
    tiles: Optional[torch.Tensor] = None
    chunks: Optional[torch.Tensor] = None
    chunk_segs: Optional[torch.Tensor] = None
    segs: Optional[torch.Tensor] = None
    absorbed: int = 0
    lat_rows: int = 0
    lat_items: Optional[torch.Tensor] = None
    lat_tiles: Optional[torch.Tensor] = None
    # by chunk size: the portions behind the absorbed tokens
    talk: dict[int, ChunkPortions] = field(default_factory=dict)
    whole: bool = False
    rows: Optional[torch.Tensor] = None
    state_bytes: int = 0

    def entries(self) -> list:
        """(first token, length, slot, start) of every entry, on the host."""
        if self.segs is not None:
            return [tuple(r) for r in self.segs.tolist()]
        return [(i, 1, s, p) for i, (s, p) in enumerate(
            zip(self.slot.tolist(), self.pos.tolist()))]


@dataclass(frozen=True)
class Keys:
    """Which keys up to its own a query sees: the last `window` (0: all), its
    own included, and the first `keep`."""
    window: int = 0
    keep: int = 0

    def most(self, length: int) -> int:
        """Bound of the keys that lie in pages with a seen one."""
        if not self.window:
            return length
        return min(length, self.window + self.keep + 2 * PAGE)


ALL_KEYS = Keys()


@dataclass
class Choice:
    """How experts are chosen: `top` of them, by softmax score plus `corr` (f32,
    one per router output), among the `keep` best of `groups` equal groups.
    Weights are the scores over (their sum + eps), times scale; or (sigmoid) the
    sigmoids of the logits as they are. They go with the experts' outputs, or
    (weigh_input) are put on their inputs. Router outputs behind the experts are
    identities. glu: the unit of gated experts."""
    top: int
    corr: Optional[torch.Tensor] = None
    groups: int = 1
    keep: int = 1
    eps: float = 0.0
    scale: float = 1.0
    sigmoid: bool = False
    weigh_input: bool = False
    glu: Glu = SWIGLU


@dataclass
class Talk:
    """A talking-heads attention layer: its constants and weights. rot: cos and
    sin tables [positions, R / 2] of neighbouring pairs; bias f32 [(H + G) * P]
    of the projection; norms f32 [P]; talk f32 [H, H]."""
    heads: int
    dim: int
    scale: float
    cap: float
    chunk: int
    rot: tuple
    bias: torch.Tensor
    qnorm: torch.Tensor
    knorm: torch.Tensor
    talk: torch.Tensor
    # talk in f16 in the tiled kernel's numbering of heads, and the factor that
    # makes up for its scaling
    talk16: Optional[torch.Tensor] = None
    talk16_scale: float = 1.0


@dataclass
class DepthAverage:
    """Results of the embedding and the layers, hist f32 [layers + 1, n, W],
    and the weights coef of what is passed on behind the layer whose result is
    hist[at]; store: whether anyone reads that result again."""
    hist: torch.Tensor
    coef: torch.Tensor
    at: int
    store: bool = True


def decode_lengths(seq_lens, slot_map):
    return seq_lens[slot_map.long()]


def decode_ordered(seq_lens, slot_map):
    return decode_lengths(seq_lens, slot_map), None


def embed(tok, pos, emb, ptab, w=None, w_off=0.0, width=0, eps=0.0, out=None):
    x = emb[tok].float()
    if ptab is not None:
        x = x + ptab[pos.long()].float()
    if w is not None:
        x = _norm(x, w, w_off, width, eps)
    if out is not None:
        x = out.copy_(x)
    return x, (x if emb.dtype == torch.float32 else x.to(emb.dtype))


def _norm(y, w, w_off, width, eps):
    rs = torch.rsqrt(y.pow(2).sum(-1, keepdim=True) / width + eps)
    return y * rs * (w_off + w)


def post_norm(x, xb, y, w, w_off, width, eps, pair_w=None):
    y = y.float()
    if pair_w is not None:
        y = (y.view(*pair_w.shape, -1) * pair_w.unsqueeze(-1)).sum(1)
    x += _norm(y, w, w_off, width, eps)
    if xb is not x:
        xb.copy_(x)


def sum_norm(x, xo, xb, y, w, w_off, alpha, width, eps, pair_w=None,
             ident=None, avg=None):
    y = y.float()
    if pair_w is not None:
        pw = pair_w.unsqueeze(-1)
        y = torch.where(pw != 0, y.view(*pair_w.shape, -1) * pw, 0.0).sum(1)
    if ident is not None:
        y = y + ident.unsqueeze(-1) * x
    r = _norm(alpha * x + y, w, w_off, width, eps)
    if avg is not None:
        if avg.store:
            avg.hist[avg.at] = r
        r = avg.coef[avg.at] * r + torch.einsum(
            "l,lnw->nw", avg.coef[:avg.at], avg.hist[:avg.at])
    xo.copy_(r)
    if xb is not xo:
        xb.copy_(r)


def norm_rows(x, rows, w, w_off, width, eps, dtype):
    z = x if rows is None else x[rows.long()]
    return _norm(z, w, w_off, width, eps).to(dtype)


def group_norm(x, rows, w, groups, width, eps, dtype):
    z = x if rows is None else x[rows.long()]
    parts = z[:, :width].view(z.shape[0], groups, -1)
    rs = torch.rsqrt(parts.pow(2).mean(-1, keepdim=True) + eps)
    out = torch.zeros_like(z)
    out[:, :width] = (parts * rs).flatten(1)
    return (out * w).to(dtype)


def join_norm(x, y, wy, w, groups, width, eps):
    x += group_norm(y.float(), None, wy, groups, width, eps, torch.float32)
    return None if w is None else group_norm(x, None, w, groups, width, eps,
                                             y.dtype)


def poly_norm(z, coef, ff, eps):
    z, out = z.float(), coef[3]
    for i in range(3):
        q = z ** (i + 1)
        out = out + coef[i] * q * torch.rsqrt(
            q.pow(2).sum(-1, keepdim=True) / ff + eps)
    return out


def streams_start(tok, emb, scale, read, w, width, eps):
    x = (emb[tok].float() * scale).unsqueeze(1).repeat(1, read.shape[0], 1)
    return x, _read_streams(x, read, w, width, eps).to(emb.dtype)


def _read_streams(x, read, w, width, eps):
    return _norm(torch.einsum("s,nsw->nw", read, x), w, 0.0, width, eps)


def streams_join(x, y, hc, read, w, width, eps, top=0, extra=None):
    n, ns, _ = x.shape
    out = y.float().view(n, max(1, top), -1).sum(1)
    if extra is not None:
        out = out + extra[0].float() * torch.sigmoid(extra[1])
    mix, put = hc[:ns * ns].view(ns, ns), hc[ns * ns:]
    x.copy_(torch.einsum("st,nsw->ntw", mix, x) +
            put.view(1, ns, 1) * out.unsqueeze(1))
    return None if w is None else _read_streams(x, read, w, width,
                                                eps).to(y.dtype)


def streams_norm(x, rows, w, width, eps, dtype):
    z = x if rows is None else x[rows.long()]
    return _norm(z.sum(1), w, 0.0, width, eps).to(dtype)


def proj_f32(x, w, bias=None):
    return F.linear(x.float(), w.float(), bias)


def _rows_of(cache, table, slot, lo, hi):
    """Rows lo..hi-1 of a slot as (page, offset) index pairs."""
    p = torch.arange(lo, hi)
    return table[slot, p // PAGE].long(), p % PAGE


def silu_cols(rows, at, count):
    cols = rows[:, at:at + count]
    cols.copy_(F.silu(cols.float()))


def qknorm_kv(qkv, kc, vc, st, heads, kv_heads, dim, eps, coef, every,
              rot=None, silu=(0, 0)):
    n, p = qkv.shape[0], kc.shape[3]
    cols = qkv[:, :(heads + 2 * kv_heads) * p].float().view(n, -1, p)
    q, k, v = cols.split([heads, kv_heads, kv_heads], dim=1)

    def unit(z):
        return z * torch.rsqrt(z.pow(2).sum(-1, keepdim=True) / dim + eps)

    if silu[1]:
        silu_cols(qkv, *silu)
    if rot is not None:
        q, k = (_rotate_first(z, st.pos, rot) for z in (q, k))
    steps = torch.div(st.pos + 1, every, rounding_mode="floor").float()
    q = unit(q) * (1 + coef * torch.log(steps + 1)).view(n, 1, 1)
    k = unit(k)
    page = st.table[st.slot.long(), (st.pos // PAGE).long()].long()
    off = (st.pos % PAGE).long()
    kc[page, :, off] = k.to(kc.dtype)
    vc[page, :, off] = v.to(vc.dtype)
    return q.to(qkv.dtype)


def paged_attn(q, kc, vc, st, scale, sink, gate, keys=ALL_KEYS, out=None,
               oscale=1.0):
    n, h, p = q.shape
    g = kc.shape[1]
    o = torch.empty(n, h, p)
    for off, ln, slot, start in st.entries():
        total = start + ln
        page, row = _rows_of(kc, st.table, slot, 0, total)
        k = kc[page, :, row].float().repeat_interleave(h // g, dim=1)
        v = vc[page, :, row].float().repeat_interleave(h // g, dim=1)
        s = torch.einsum("thd,shd->hts", q[off:off + ln].float(), k) * scale
        j = torch.arange(total).view(1, 1, -1)
        i = torch.arange(start, total).view(1, -1, 1)
        hidden = j > i
        if keys.window:
            hidden |= (i - j >= keys.window) & (j >= keys.keep)
        s = s.masked_fill(hidden, float("-inf"))
        if sink is not None:
            s = torch.cat([s, sink.view(h, 1, 1).expand(h, ln, 1)], dim=-1)
        w = torch.softmax(s, dim=-1)[..., :total]
        o[off:off + ln] = torch.einsum("hts,shd->thd", w, v)
    if gate is not None:
        o *= torch.sigmoid(gate.float()).view(n, h, -1)
    o = (o * oscale).to(q.dtype)
    return o if out is None else out.copy_(o.view(n, h * p))


def _rotate(x, pos, rot):
    """Neighbouring pairs of x [n, ..., R] by tables cos, sin [*, R / 2]."""
    c, s = (t[pos.long()].view(-1, *[1] * (x.dim() - 2), t.shape[1])
            for t in rot)
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack([u * c - v * s, v * c + u * s], dim=-1).flatten(-2)


def latent_rows(rows, lat, st, rot, qnorm, kvnorm, qtrue, ktrue, eps):
    qr, kr = qnorm.shape[0], kvnorm.shape[0]
    r = lat.shape[2] - kr
    q, c, k = rows[:, :qr + kr + r].float().split([qr, kr, r], dim=1)
    page = st.table[st.slot.long(), (st.pos // PAGE).long()].long()
    lat[page, (st.pos % PAGE).long()] = torch.cat(
        [_norm(c, kvnorm, 0.0, ktrue, eps), _rotate(k, st.pos, rot)],
        dim=1).to(lat.dtype)
    return _norm(q, qnorm, 0.0, qtrue, eps).to(rows.dtype)


def latent_attn(q, lat, st, rot, wuk, wuv, wukv, scale, gate):
    h, kr, p = wuk.shape
    n, r = q.shape[0], lat.shape[2] - kr
    q = q.view(n, h, p + r).float()
    ql = torch.matmul(wuk.float(), q[..., :p].unsqueeze(-1)).squeeze(-1)
    ql = torch.cat([ql, _rotate(q[..., p:], st.pos, rot)], dim=-1)
    out = torch.empty(n, h, p, dtype=q.dtype)
    for off, ln, slot, start in st.entries():
        total = start + ln
        page, row = _rows_of(lat, st.table, slot, 0, total)
        c = lat[page, row].float()
        s = torch.einsum("thd,sd->hts", ql[off:off + ln], c) * scale
        ahead = torch.arange(total).view(1, 1, -1) > \
            torch.arange(start, total).view(1, -1, 1)
        w = torch.softmax(s.masked_fill(ahead, float("-inf")), dim=-1)
        o = torch.einsum("hts,sk->thk", w, c[:, :kr])
        out[off:off + ln] = torch.matmul(wuv.float(),
                                         o.unsqueeze(-1)).squeeze(-1)
    out *= torch.sigmoid(gate[:, :h].float()).unsqueeze(-1)
    return out.view(n, h * p).to(q.dtype)


def gla(rows, u, wa2, ba2, S, norm, st, dim, vdim, tau, eps):
    n = rows.shape[0]
    h, dv, dk = S.shape[1:]
    q, k, v, g = rows[:, :h * 2 * (dk + dv)].float().split(
        [h * dk, h * dk, h * dv, h * dv], dim=1)
    q, k = q.view(n, h, dk) * dim ** -0.5, k.view(n, h, dk)
    v = v.view(n, h, dv)
    keep = torch.exp(F.logsigmoid(u @ wa2 + ba2) / tau).view(n, h, dk)
    o = torch.empty(n, h, dv)
    for off, ln, slot, start in st.entries():
        s = torch.zeros_like(S[slot]) if start == 0 else S[slot]
        for t in range(off, off + ln):
            s = keep[t].unsqueeze(1) * s + v[t].unsqueeze(2) * \
                k[t].unsqueeze(1)
            o[t] = torch.matmul(s, q[t].unsqueeze(2)).squeeze(2)
        S[slot] = s
    o = o * torch.rsqrt(o.pow(2).sum(-1, keepdim=True) / vdim + eps)
    return (o.reshape(n, -1) * norm * F.silu(g)).to(rows.dtype)


def mlstm(qkv, gates, S, m, norm, st, dim, vdim, cap, eps):
    n = qkv.shape[0]
    h, dv, dk = S.shape[1], S.shape[2] - 1, S.shape[3]
    q, k, v, g = qkv[:, :h * 2 * (dk + dv)].float().split(
        [h * dk, h * dk, h * dv, h * dv], dim=1)
    q = q.view(n, h, dk) * dim ** -0.5
    k = k.view(n, h, dk)
    v = F.pad(v.view(n, h, dv), (0, 1), value=1.0)   # last row: normaliser
    gi = cap * torch.tanh(gates[:, :h] / cap)
    gf = F.logsigmoid(cap * torch.tanh(gates[:, h:] / cap))
    o = torch.empty(n, h, dv)
    for off, ln, slot, start in st.entries():
        s, mm = S[slot], m[slot]
        if start == 0:
            s, mm = torch.zeros_like(s), torch.zeros_like(mm)
        for t in range(off, off + ln):
            m2 = torch.maximum(gf[t] + mm, gi[t])
            keep, put = torch.exp(gf[t] + mm - m2), torch.exp(gi[t] - m2)
            mm = m2
            s = keep.view(h, 1, 1) * s + put.view(h, 1, 1) * \
                v[t].unsqueeze(2) * k[t].unsqueeze(1)
            r = torch.matmul(s, q[t].unsqueeze(2)).squeeze(2)
            den = torch.maximum(r[:, dv].abs(), torch.exp(-mm)) + 1e-6
            o[t] = r[:, :dv] / den.view(h, 1)
        S[slot], m[slot] = s, mm
    o = o * torch.rsqrt(o.pow(2).sum(-1, keepdim=True) / vdim + eps)
    return (o.reshape(n, -1) * norm * torch.sigmoid(g)).to(qkv.dtype)


def lightning(rows, S, decay, norm, st, vdim, eps, out=None):
    n = rows.shape[0]
    h, dv, dk = S.shape[1:]
    q, k, v, g = rows[:, :h * 2 * (dk + dv)].float().split(
        [h * dk, h * dk, h * dv, h * dv], dim=1)
    q, k, v = (t.view(n, h, -1) for t in (q, k, v))
    keep = decay[0].view(h, 1, 1)
    o = torch.empty(n, h, dv)
    for off, ln, slot, start in st.entries():
        s = torch.zeros_like(S[slot]) if start == 0 else S[slot]
        for t in range(off, off + ln):
            s = keep * s + v[t].unsqueeze(2) * k[t].unsqueeze(1)
            o[t] = torch.matmul(s, q[t].unsqueeze(2)).squeeze(2)
        S[slot] = s
    o = (_norm(o.view(n, -1), norm, 0.0, h * vdim, eps) *
         torch.sigmoid(g)).to(rows.dtype)
    return o if out is None else out.copy_(o)


def moe(x, logits, up, down, how):
    if isinstance(how, int):
        how = Choice(how)
    n, experts = x.shape[0], up.shape[0]
    s = torch.sigmoid(logits) if how.sigmoid else torch.softmax(logits, dim=-1)
    choice = logits if how.corr is None else s + how.corr
    if how.groups > 1:
        by = choice.view(n, how.groups, -1)
        best = torch.topk(by.amax(-1), how.keep, dim=-1).indices
        out = torch.ones(n, how.groups, dtype=torch.bool)
        out.scatter_(1, best, False)
        choice = by.masked_fill(out.unsqueeze(-1), float("-inf")).view(n, -1)
    idx = torch.topk(choice, how.top, dim=-1).indices
    wt = s.gather(1, idx)
    if not how.sigmoid:
        wt = wt / (wt.sum(-1, keepdim=True) + how.eps) * how.scale
    ident = None
    if logits.shape[1] > experts:
        same = idx >= experts
        ident = (wt * same).sum(-1)
        wt = wt.masked_fill(same, 0.0)
    flat = idx.reshape(-1)
    xs = x.repeat_interleave(how.top, dim=0).float()
    ye = torch.empty(flat.shape[0], x.shape[1], dtype=x.dtype)
    gated = up.shape[1] != down.shape[2]
    for e in torch.unique(flat).tolist():
        if e >= experts:
            continue
        r = (flat == e).nonzero().squeeze(1)
        a = xs[r] @ up[e].float().T
        if how.weigh_input:
            a = a * wt.reshape(-1)[r].unsqueeze(1)
        if gated:                          # rows in turns of 16 gate | 16 up
            g, u = a.view(len(r), -1, 2, 16).unbind(2)
            a = swiglu(torch.cat([g.reshape(len(r), -1),
                                  u.reshape(len(r), -1)], dim=1), how.glu)
        else:
            a = torch.relu(a) ** 2
        ye[r] = (a @ down[e].float().T).to(x.dtype)
    return ye, wt, ident


def talk_rows(rows, vc, inv, st, tk, eps):
    n, h, (g, _, p) = rows.shape[0], tk.heads, vc.shape[1:]
    cols = rows[:, :(h + g) * p].float() + tk.bias
    q, v = cols.view(n, h + g, p).split([h, g], dim=1)
    rs = torch.rsqrt(v.pow(2).sum(-1) / tk.dim + eps)
    page = st.table[st.slot.long(), (st.pos // PAGE).long()].long()
    off = (st.pos % PAGE).long()
    vc[page, :, off] = v.to(vc.dtype)
    inv[page, :, off] = rs
    return _rotate_first(_norm(q, tk.qnorm, 0.0, tk.dim, eps), st.pos,
                         tk.rot).to(rows.dtype)


def _rotate_first(x, pos, rot):
    """_rotate on the coordinates that the tables cover."""
    r = 2 * rot[0].shape[1]
    if not r:
        return x
    return torch.cat([_rotate(x[..., :r], pos, rot), x[..., r:]], dim=-1)


def talk_attn(q, vc, inv, st, tk):
    n, h, p = q.shape
    g = vc.shape[1]
    out = torch.empty_like(q)
    for off, ln, slot, start in st.entries():
        lo, total = start // tk.chunk * tk.chunk, start + ln
        page, row = _rows_of(vc, st.table, slot, lo, total)
        v = vc[page, :, row].float()
        k = _rotate_first(v * inv[page, :, row].unsqueeze(-1) * tk.knorm,
                          torch.arange(lo, total), tk.rot)
        k, v = (t.repeat_interleave(h // g, dim=1) for t in (k, v))
        s = torch.einsum("thd,shd->hts", q[off:off + ln].float(), k)
        s = tk.cap * torch.tanh(s * tk.scale / tk.cap)
        i = torch.arange(start, total).view(1, -1, 1)
        j = torch.arange(lo, total).view(1, 1, -1)
        s = s.masked_fill((j > i) | (j // tk.chunk != i // tk.chunk),
                          float("-inf"))
        s = torch.cat([s, torch.zeros(h, ln, 1)], dim=-1)
        w = torch.softmax(s, dim=-1)[..., :-1]
        w = torch.einsum("hg,gts->hts", tk.talk, w)
        out[off:off + ln] = torch.einsum("hts,shd->thd", w, v).to(q.dtype)
    return out
