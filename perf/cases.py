"""Performance cases: the work that serving a model comes down to, step by step.

A served request is a prompt pass and then decode steps, many requests at a time,
with a sampled token behind each step. The kinds of case:

  prompt   one call of forward_prefill (one sequence) or forward_prefill_batch
           (several, of different lengths) on fresh sequences
  decode   one decode step of a batch whose sequences hold contexts of different
           lengths, captured in a graph as the engine does
  experts  a layer's routed experts on a batch of tokens, which the models below
           leave out: with random weights a router's close calls fall one way or
           the other by rounding, so that whole models could not be compared
  sample   the token pick behind a decode step

Models are the registry's, at their widths but of few layers: with random
weights each layer of bf16 adds to the rounding error of all behind it, so that
at full depth two correct programs differ by 4 % and more (Birepel, whose
memories multiply three projections, by 10 %). Layer-list models keep their
mixers and norms; routed feed-forwards become dense ones of the same active size
(see experts). Weights are the models' own random ones, by seed.
"""
import math
import random
from dataclasses import dataclass, replace

import numpy as np
import torch

from gridllm_amd.engine.sampler import SamplerState, SlotSampler
from gridllm_amd.models import model_class
from gridllm_amd.models.registry import (AttentionMixer, DenseFF, HybridSpec,
                                         LatentMixer, MlstmMixer, PolyFF,
                                         RoutedFF, TalkingMixer, get_spec)
from gridllm_amd.ops import hybrid as hops
from gridllm_amd.ops.autotune import tune_model_shapes
from gridllm_amd.ops.reference import SWIGLU, Glu
from gridllm_amd.types import SamplingOptions

DEV = "cuda"
PAGE = 64
VOCAB = 128256


def listed():
    return [
        # a chat message to the default engine model: little work, many launches
        dict(name="prompt short", kind="prompt", model="llama3.2:1b", rows=1,
             tokens=45),
        # a burst of requests admitted together
        dict(name="prompt batch", kind="prompt", model="llama3.2:3b", rows=8,
             tokens=1300),
        # a long document at the models' full context
        dict(name="prompt long", kind="prompt", model="llama3.2:3b", rows=1,
             tokens=8000),
        # one user's stream
        dict(name="decode 1", kind="decode", model="llama3.2:3b", rows=1,
             tokens=900),
        # some users with long conversations
        dict(name="decode 24", kind="decode", model="llama3.2:3b", rows=24,
             tokens=6000),
        # a loaded server, short chats
        dict(name="decode 256", kind="decode", model="llama3.2:3b", rows=256,
             tokens=384),
        # layer-list models: matrix memories and attention over pages
        dict(name="birepel prompt", kind="prompt", model="birepel:3b", rows=1,
             tokens=3500),
        dict(name="birepel decode", kind="decode", model="birepel:3b", rows=64,
             tokens=2000),
        # latents and gated linear attention, several prompts in one step
        dict(name="maferax prompts", kind="prompt", model="maferax:5b", rows=4,
             tokens=1100),
        # talking heads, a loaded server
        dict(name="vivepel decode", kind="decode", model="vivepel:2b",
             rows=160, tokens=1000),
        # routed experts of a decode step
        dict(name="experts decode", kind="experts", model="birepel:3b",
             rows=48),
        # tokens of a loaded server's step, temperature alone
        dict(name="sample", kind="sample", rows=64),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["prompt"] * 4 + ["decode"] * 4 + ["experts", "sample"])
    if kind == "sample":
        return dict(kind=kind, rows=spread(1, 512))
    if kind == "experts":
        return dict(kind=kind, model=rng.choice(["birepel:3b", "zinavik:4b"]),
                    rows=spread(1, 4096))
    model = rng.choice(["llama3.2:1b", "llama3.2:3b", "llama3.2:3b",
                        "qwen2.5:0.5b", "qwen2.5:1.5b", "birepel:3b",
                        "maferax:5b", "vivepel:2b"])
    if kind == "prompt":
        most = 3600 if model in ("birepel:3b", "maferax:5b") else 7500
        total = spread(9, most)
        rows = min(spread(1, 24), max(1, total // 8))
        return dict(kind=kind, model=model, rows=rows,
                    tokens=max(8, min(most, 2 * total // (rows + 1))))
    rows = spread(1, 256)
    return dict(kind=kind, model=model, rows=rows,
                tokens=spread(9, min(6000, 100000 // rows)))


def lengths(case):
    """Tokens of each sequence: the longest is the case's, the others spread
    below it."""
    rng = random.Random(case["rows"] * 100003 + case["tokens"])
    top = case["tokens"]
    return [top] + [rng.randint(max(1, top // 6), top)
                    for _ in range(case["rows"] - 1)]


def spec_of(name):
    s = get_spec(name)
    if not isinstance(s, HybridSpec):
        return replace(s, layers=4)

    def dense(ff):
        if not isinstance(ff, RoutedFF):
            return ff
        own = next(ly.ff for ly in s.layers if isinstance(ly.ff, DenseFF))
        return replace(own, ff=ff.top * ff.ff)

    return replace(s, layers=tuple(replace(ly, ff=dense(ly.ff))
                                   for ly in s.layers[:3 if s.family ==
                                                      "birepel" else 8]))


def generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


# ---------------------------------------------------------------- preparation

def build(case, seed):
    """The model with a cache for the case's sequences (one slot to spare), as
    a server would bound them: generously, up to the usual context of 8192."""
    s = spec_of(case["model"])
    room = min(8192, max(1024, 1 << (2 * case["tokens"] - 1).bit_length()))
    extra = {"kv_tokens": sum(-(-(n + 1) // PAGE) * PAGE
                              for n in lengths(case))} \
        if isinstance(s, HybridSpec) else {}
    m = model_class(s)(s, device=DEV, dtype="bf16", seed=seed + 1,
                       kv_slots=case["rows"] + 1, max_seq=room, **extra)
    return s, m


def token_ids(case, seed, vocab, counts):
    g = generator(seed * 7 + 3)
    return [torch.randint(0, vocab, (n,), generator=g, device=DEV)
            for n in counts]


def fill(case, seed, s, m):
    """What a batch's earlier tokens left behind, at random: keys and values,
    latents, recurrent states. Returns the slots."""
    g, lens = generator(seed * 5 + 1), lengths(case)
    slots = [m.cache.alloc(n + 1) for n in lens]
    if isinstance(s, HybridSpec):
        m.cache.extend(slots, lens)
        m.cache.seq_lens[torch.tensor(slots, device=DEV)] = torch.tensor(
            lens, dtype=torch.int32, device=DEV)
        for i, ly in enumerate(s.layers):
            for t in (m.cache.k[i], m.cache.v[i], m.cache.lat[i],
                      m.cache.S[i]):
                if t is not None:
                    t.normal_(generator=g)
            if m.cache.inv[i] is not None:
                v = m.cache.v[i].float()
                m.cache.inv[i].copy_(torch.rsqrt(
                    v.pow(2).mean(-1) + s.norm_eps))
    else:
        top = max(lens)
        for i in range(s.layers):
            m.cache.k[i][:, :, :top].normal_(generator=g)
            m.cache.v[i][:, :, :top].normal_(generator=g)
        m.cache.seq_lens[torch.tensor(slots, device=DEV)] = torch.tensor(
            lens, dtype=torch.int32, device=DEV)
    return slots


@dataclass
class Row:
    slot: int
    state: SamplerState


def expert_inputs(case, seed):
    ff, g = next(ly.ff for ly in get_spec(case["model"]).layers
                 if isinstance(ly.ff, RoutedFF)), generator(seed + 1)
    w = get_spec(case["model"]).hidden

    def t(*shape, std):
        return (torch.randn(*shape, generator=g, device=DEV) * std).to(
            torch.bfloat16)

    x = t(case["rows"], w, std=1.0)
    logits = torch.randn(case["rows"], ff.experts, generator=g, device=DEV)
    up = torch.empty(ff.experts, ff.ff * (2 if ff.gated else 1), w,
                     dtype=torch.bfloat16, device=DEV)
    down = torch.empty(ff.experts, w, ff.ff, dtype=torch.bfloat16, device=DEV)
    for e in range(ff.experts):
        up[e] = t(*up.shape[1:], std=0.02)
        down[e] = t(*down.shape[1:], std=0.02)
    return ff, x, logits, up, down


def prepare(case, seed):
    if case["kind"] == "sample":
        g = generator(seed + 1)
        rows = [Row(i, SamplerState.create(SamplingOptions.from_dict(
            {"temperature": 0.8, "seed": seed * 1000 + i + 1}),
            torch.device(DEV))) for i in range(case["rows"])]
        sampler = SlotSampler(len(rows) + 1, torch.device(DEV))
        sampler.admit(rows, VOCAB)
        return dict(kind="sample", sampler=sampler, rows=rows,
                    slots=torch.arange(len(rows), device=DEV),
                    logits=2 * torch.randn(case["rows"], VOCAB, generator=g,
                                           device=DEV))
    if case["kind"] == "experts":
        ff, x, logits, up, down = expert_inputs(case, seed)
        glu = SWIGLU if ff.unit is None else Glu(
            ff.unit.alpha, ff.unit.limit, ff.unit.shift, ff.unit.cubic)
        return dict(kind="experts", x=x, logits=logits, up=up, down=down,
                    how=hops.Choice(ff.top, sigmoid=ff.sigmoid,
                                    weigh_input=ff.weigh_input, glu=glu))
    s, m = build(case, seed)
    m.interleave_gateup()
    if case["kind"] == "prompt":
        return dict(kind="prompt", model=m,
                    tokens=token_ids(case, seed, s.vocab, lengths(case)))
    slots = fill(case, seed, s, m)
    tokens = token_ids(case, seed, s.vocab, [case["rows"]])[0]
    slot_map = torch.tensor(slots, dtype=torch.int32, device=DEV)
    tune_model_shapes(m, [case["rows"]])
    lens = m.cache.seq_lens.clone()
    kept = [t.clone() if t is not None else None
            for t in getattr(m.cache, "S", [])]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            m.cache.prepare_decode(slots)
            m.forward_decode(tokens, slot_map)
            rewind(m, slots, lens)
    torch.cuda.current_stream().wait_stream(side)
    m.cache.prepare_decode(slots)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = m.forward_decode(tokens, slot_map)
    rewind(m, slots, lens)
    for t, was in zip(getattr(m.cache, "S", []), kept):
        if t is not None:
            t.copy_(was)
    for t in getattr(m.cache, "m", []):
        if t is not None:
            t.zero_()
    return dict(kind="decode", model=m, graph=graph, slots=slots, lens=lens,
                tokens=tokens, slot_map=slot_map, out=out)


def rewind(m, slots, lens):
    """Forget the last decoded tokens."""
    m.cache.seq_lens.copy_(lens)
    if hasattr(m.cache, "lens"):
        m.cache.lens[np.asarray(slots)] -= 1


# ------------------------------------------------------------------- one pass

def run(state):
    kind = state["kind"]
    if kind == "sample":
        return state["sampler"].sample_ids(state["logits"], state["rows"],
                                           state["slots"])
    if kind == "experts":
        y, wt, _ = hops.moe(state["x"], state["logits"], state["up"],
                            state["down"], state["how"])
        return y, wt
    m = state["model"]
    cache = m.cache
    if kind == "decode":
        cache.prepare_decode(state["slots"])
        state["graph"].replay()
        # the next pass decodes the same token again
        rewind(m, state["slots"], state["lens"])
        return [state["out"]] + kept_states(m)
    slots = [cache.alloc(len(t)) for t in state["tokens"]]
    if len(slots) == 1:
        logits = m.forward_prefill(state["tokens"][0], slots[0])
    else:
        logits = m.forward_prefill_batch(state["tokens"], slots)
    for sl in reversed(slots):
        cache.free(sl)
    if not hasattr(cache, "table"):
        return [logits] + [t[sl, :, :len(ids)] for ids, sl in
                           zip(state["tokens"], slots)
                           for t in (cache.k[-1], cache.v[-1])]
    return [logits] + pages_of(m) + kept_states(m)


def pages_of(m):
    """The last attention layer's pages."""
    c = m.cache
    i = max(i for i in range(len(c.v)) if c.v[i] is not None
            or c.lat[i] is not None)
    return [t for t in (c.k[i], c.v[i], c.lat[i]) if t is not None]


def kept_states(m):
    """The last recurrent layer's states."""
    S = [t for t in getattr(m.cache, "S", []) if t is not None]
    return S[-1:]


# ------------------------------------------------------------ work, tolerance

def work(case):
    n = case["rows"]
    if case["kind"] == "sample":
        return {"bytes": n * VOCAB * 4 + n * 8, "flops": 0}
    if case["kind"] == "experts":
        s = get_spec(case["model"])
        ff = next(ly.ff for ly in s.layers if isinstance(ly.ff, RoutedFF))
        mats = 3 if ff.gated else 2
        hit = ff.experts * (1 - (1 - ff.top / ff.experts) ** n)
        return {"bytes": hit * mats * s.hidden * ff.ff * 2
                + n * s.hidden * 2 * (1 + ff.top) + n * ff.experts * 4,
                "flops": 2 * n * ff.top * mats * s.hidden * ff.ff}
    s, lens = spec_of(case["model"]), lengths(case)
    total = sum(lens) if case["kind"] == "prompt" else n
    table = s.vocab * s.hidden
    body = s.params - table * (2 if not getattr(
        s, "tie_embeddings", getattr(s, "tied", True)) else 1)
    flops = 2 * total * body + 2 * n * table
    moved = 2 * (body + table) + 4 * n * s.vocab
    layers = s.layers if isinstance(s, HybridSpec) else [None] * s.layers
    for ly in layers:
        mx = None if ly is None else ly.mixer
        if ly is not None and ly.weights_of is not None:
            flops += 2 * total * (mx.params(s.hidden) + ly.ff.params(s.hidden))
        if mx is None:
            heads, d, row = s.heads, s.head_dim, 4 * s.kv_heads * s.head_dim
        elif isinstance(mx, AttentionMixer):
            heads, d, row = mx.heads, mx.dim, 4 * mx.kv_heads * mx.dim
        elif isinstance(mx, TalkingMixer):
            heads, d, row = mx.heads, mx.dim, 2 * mx.kv_heads * mx.dim
        elif isinstance(mx, LatentMixer):
            heads, d = mx.heads, (mx.dim + mx.rot_dim + mx.vdim) // 2
            row = 2 * (mx.kv_rank + mx.rot_dim)
        else:                          # a state per sequence, in and out
            size = mx.heads * mx.dim * mx.vdim
            flops += 4 * total * size
            moved += n * size * (8 if case["kind"] == "decode" else 4)
            continue
        if case["kind"] == "prompt":
            flops += sum(2 * heads * d * t * (t + 1) for t in lens)
            moved += total * row
        else:
            flops += sum(4 * heads * d * t for t in lens)
            moved += sum(lens) * row
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    if case["kind"] == "sample":
        return "exact"
    if case["kind"] == "experts":
        return {"rel": 0.01}
    return {"rel": 0.03, "max": 0.5}


# -------------------------------------------------------------- 64-bit results

def f64(t):
    return t.to(torch.float64)


def rms(x, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def softmax_attend(q, k, v, scale, past, sink=None):
    """Causal attention of one sequence's q [t, H, d], the first at position
    `past`, over k [n, G, d] and v [n, G, dv] -> [t, H, dv]."""
    t, h, d = q.shape
    n, g = k.shape[:2]
    kk, vv = k.transpose(0, 1).contiguous(), v.transpose(0, 1).contiguous()
    out = q.new_empty(t, h, v.shape[2])
    pos = torch.arange(n, device=q.device)
    for a in range(0, t, 1024):
        b = min(t, a + 1024)
        qq = q[a:b].transpose(0, 1).reshape(g, -1, d)
        sc = (qq @ kk.transpose(1, 2)).view(h, b - a, n).mul_(scale)
        sc.masked_fill_(pos > past + torch.arange(
            a, b, device=q.device).view(-1, 1), -math.inf)
        top = sc.amax(-1, keepdim=True)
        if sink is not None:
            top = torch.maximum(top, sink.view(h, 1, 1))
        sc = sc.sub_(top).exp_()
        den = sc.sum(-1, keepdim=True)
        if sink is not None:
            den = den + torch.exp(sink.view(h, 1, 1) - top)
        o = (sc / den).view(g, -1, n) @ vv
        out[a:b] = o.view(h, b - a, -1).transpose(0, 1)
    return out


def angles(pos, freqs):
    a = torch.outer(f64(pos), freqs)
    return a.cos().unsqueeze(1), a.sin().unsqueeze(1)


def turn_halves(x, pos, theta):
    """Rotate the pairs (i, i + d / 2) of x [t, h, d]."""
    half = x.shape[-1] // 2
    c, s = angles(pos, theta ** (-torch.arange(
        half, dtype=torch.float64, device=x.device) / half))
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def turn_pairs(x, pos, base, dims):
    """Rotate the neighbouring pairs of x's first dims coordinates."""
    c, s = angles(pos, base ** (-2 * torch.arange(
        dims // 2, dtype=torch.float64, device=x.device) / dims))
    a, b = x[..., 0:dims:2], x[..., 1:dims:2]
    r = torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)
    return torch.cat([r, x[..., dims:]], -1)


class Sequences:
    """The case's sequences: where each one's tokens lie among all, how many
    came before, and what those left in the cache."""

    def __init__(self, case, s, m, slots):
        self.m, lens = m, lengths(case)
        self.decode = case["kind"] == "decode"
        self.past = lens if self.decode else [0] * len(lens)
        self.count = [1] * len(lens) if self.decode else lens
        ends = np.cumsum(self.count)
        self.parts = [slice(int(e) - c, int(e))
                      for e, c in zip(ends, self.count)]
        self.pos = torch.cat([torch.arange(p, p + c, device=DEV)
                              for p, c in zip(self.past, self.count)])
        self.last = torch.as_tensor(ends - 1, device=DEV)
        self.slots = slots

    def rows(self, pool, j):
        """Sequence j's rows [past, ...] of a cache tensor."""
        n, sl = self.past[j], self.slots[j]
        if not hasattr(self.m.cache, "table"):
            return f64(pool[sl, :, :n].transpose(0, 1))
        pages = self.m.cache.table[sl, :-(-n // PAGE)].long()
        t = pool[pages]
        if t.dim() == 4:               # [pages, G, 64, P]
            t = t.transpose(1, 2)
        return f64(t.reshape(-1, *t.shape[2:])[:n])

    def each(self, f):
        return torch.cat([f(j, p) for j, p in enumerate(self.parts)])


def join(past, new):
    return new if not past.shape[0] else torch.cat([past, new])


def exact_llama(s, m, sq, tokens):
    x, last = f64(m.embed[tokens]), None
    h, g, d, eps = s.heads, s.kv_heads, s.head_dim, s.norm_eps
    for i, w in enumerate(m.layers):
        qkv = rms(x, eps) * f64(w.attn_norm) @ f64(w.wqkv).T
        if w.bqkv is not None:
            qkv = qkv + f64(w.bqkv)
        q, k, v = qkv.view(-1, h + 2 * g, d).split([h, g, g], 1)
        q = turn_halves(q, sq.pos, s.rope_theta)
        k = turn_halves(k, sq.pos, s.rope_theta)
        last = (k, v)
        o = sq.each(lambda j, p: softmax_attend(
            q[p], join(sq.rows(m.cache.k[i], j), k[p]),
            join(sq.rows(m.cache.v[i], j), v[p]), d ** -0.5, sq.past[j]))
        x = x + o.reshape(len(tokens), -1) @ f64(w.wo).T
        a, b = (rms(x, eps) * f64(w.mlp_norm) @ f64(w.wgateup).T).chunk(2, 1)
        x = x + (a * torch.sigmoid(a) * b) @ f64(w.wdown).T
    logits = rms(x[sq.last], eps) * f64(m.final_norm) @ f64(m.lm_head).T
    if sq.decode:
        return [logits]
    return [logits[0] if len(sq.parts) == 1 else logits] + [
        t[p].transpose(0, 1) for p in sq.parts for t in last]


def recur(sq, S, q, k, v, gates, step, start):
    """Walk every sequence through a recurrence; S takes the final states."""
    def one(j, p):
        carry, o = start(j), []
        for t in range(p.start, p.stop):
            carry, y = step(carry, q[t], k[t], v[t], *(z[t] for z in gates))
            o.append(y)
        S[sq.slots[j]] = carry[0]
        return torch.stack(o)
    return sq.each(one)


def exact_mixer(s, m, i, mx, w, x, sq, pages, states):
    n, eps, c = x.shape[0], s.norm_eps, m.cache
    z = x @ f64(w.wmix).T
    h = mx.heads
    if isinstance(mx, AttentionMixer):
        g, d = mx.kv_heads, mx.dim
        q, k, v, z = z.split([h * d, g * d, g * d,
                              z.shape[1] - (h + 2 * g) * d], 1)
        steps = torch.div(sq.pos + 1, mx.q_every, rounding_mode="floor")
        temp = 1 + mx.q_coef * torch.log(f64(steps) + 1)
        q = rms(q.view(n, h, d), eps) * temp.view(n, 1, 1)
        k, v = rms(k.view(n, g, d), eps), v.view(n, g, d)
        pages[:] = [k, v]
        o = sq.each(lambda j, p: softmax_attend(
            q[p], join(sq.rows(c.k[i], j), k[p]),
            join(sq.rows(c.v[i], j), v[p]), mx.scale, sq.past[j],
            f64(w.sink)))
        o = o * torch.sigmoid(z[:, :h]).unsqueeze(2)
    elif isinstance(mx, LatentMixer):
        kr, qr, r, d = mx.kv_rank, mx.q_rank, mx.rot_dim, mx.dim
        cq, lat, kx, z = z.split([qr, kr, r, z.shape[1] - qr - kr - r], 1)
        q = (rms(cq, eps) * f64(w.qnorm) @ f64(w.wuq).T).view(n, h, d + r)
        q = torch.cat([q[..., :d], turn_pairs(q[..., d:], sq.pos, mx.rot_base,
                                              mx.rot_dims)], -1)
        kx = turn_pairs(kx.unsqueeze(1), sq.pos, mx.rot_base,
                        mx.rot_dims)[:, 0]
        rows = torch.cat([rms(lat, eps) * f64(w.kvnorm), kx], 1)
        pages[:] = [rows]

        def one(j, p):
            a = join(sq.rows(c.lat[i], j), rows[p])
            keys = torch.einsum("nk,hkp->nhp", a[:, :kr], f64(w.wuk))
            keys = torch.cat([keys, a[:, None, kr:].expand(-1, h, -1)], -1)
            vals = torch.einsum("nk,hpk->nhp", a[:, :kr], f64(w.wuv))
            return softmax_attend(q[p], keys, vals, mx.scale, sq.past[j])
        o = sq.each(one) * torch.sigmoid(z[:, :h]).unsqueeze(2)
    elif isinstance(mx, TalkingMixer):
        g, d, tk = mx.kv_heads, mx.dim, w.talk
        z = (z[:, :(h + g) * d] + f64(tk.bias)).view(n, h + g, d)
        q, v = z.split([h, g], 1)
        pages[:] = [v]

        def turned(y, norm, pos):
            return turn_pairs(rms(y, eps) * f64(norm), pos, mx.rot_base,
                              mx.rot_dims)
        q = turned(q, tk.qnorm, sq.pos)

        def one(j, p):
            a = sq.past[j]
            lo = a // mx.chunk * mx.chunk if sq.decode else 0
            vals = join(sq.rows(c.v[i], j)[lo:], v[p])
            at = torch.arange(lo, lo + len(vals), device=DEV)
            keys = turned(vals, tk.knorm, at)
            out = q.new_empty(p.stop - p.start, h, d)
            for b in range(0, len(out), 512):
                qq = q[p][b:b + 512]
                mine = a + b + torch.arange(len(qq), device=DEV).view(-1, 1)
                sc = torch.stack([qq[:, x] @ keys[:, x * g // h].T
                                  for x in range(h)]) * mx.scale
                sc = mx.cap * torch.tanh(sc / mx.cap)
                sc.masked_fill_((at > mine) | (torch.div(
                    at, mx.chunk, rounding_mode="floor") != torch.div(
                        mine, mx.chunk, rounding_mode="floor")), -math.inf)
                top = sc.amax(-1, keepdim=True).clamp(min=0)
                sc = torch.exp(sc - top)
                sc = sc / (torch.exp(-top) + sc.sum(-1, keepdim=True))
                wt = (f64(tk.talk) @ sc.view(h, -1)).view_as(sc)
                out[b:b + 512] = torch.stack(
                    [wt[x] @ vals[:, x * g // h] for x in range(h)], 1)
            return out
        o = sq.each(one)
    else:
        dk, dv = mx.dim, mx.vdim
        q, k, v, gate, _ = z.split([h * dk, h * dk, h * dv, h * dv,
                                    z.shape[1] - 2 * h * (dk + dv)], 1)
        q = q.view(n, h, 1, dk) * dk ** -0.5
        k, v = k.view(n, h, 1, dk), v.view(n, h, dv, 1)
        u = x @ f64(w.wgates).T
        S = f64(c.S[i])
        states[:] = [S]
        if isinstance(mx, MlstmMixer):
            zi, zf = (mx.gate_cap * torch.tanh((u + f64(w.bgates))
                                               / mx.gate_cap)).chunk(2, 1)
            v = torch.cat([v, torch.ones_like(v[:, :, :1])], 2)

            def step(carry, q, k, v, i, f):
                S, m0 = carry
                m1 = torch.maximum(f + m0, i)
                S = torch.exp(f + m0 - m1).view(h, 1, 1) * S + \
                    torch.exp(i - m1).view(h, 1, 1) * v * k
                y = (S * q).sum(-1)
                den = torch.maximum(y[:, -1].abs(), torch.exp(-m1)) + 1e-6
                return (S, m1), y[:, :-1] / den.view(h, 1)

            o = recur(sq, S, q, k, v, (zi, torch.nn.functional.logsigmoid(zf)),
                      step, lambda j: (
                          S[sq.slots[j]] * (1 if sq.decode else 0),
                          torch.zeros(h, dtype=S.dtype, device=DEV)))
            gate = torch.sigmoid(gate)
        else:
            a = torch.nn.functional.logsigmoid(
                u @ f64(w.wa2) + f64(w.ba2)).view(n, h, 1, dk) / mx.tau

            def step(carry, q, k, v, a):
                S = torch.exp(a) * carry[0] + v * k
                return (S,), (S * q).sum(-1)

            o = recur(sq, S, q, k, v, (a,), step, lambda j: (
                S[sq.slots[j]] * (1 if sq.decode else 0),))
            gate = gate * torch.sigmoid(gate)
        o = rms(o, eps).reshape(n, -1) * f64(w.mnorm) * gate
    return o.reshape(n, -1) @ f64(w.wo).T


def exact_feed(s, ff, w, x):
    if isinstance(ff, PolyFF):
        z = x @ f64(w.up).T
        c = f64(w.act)
        z = c[3] + sum(c[k] * rms(z ** (k + 1), s.norm_eps) for k in range(3))
        return z @ f64(w.down).T
    g, u = (x @ f64(w.wgateup).T).chunk(2, 1)
    return glu(g, u, ff) @ f64(w.down).T


def glu(g, u, p):
    g, u = g.clamp(max=p.limit), u.clamp(-p.limit, p.limit)
    return g * torch.sigmoid(p.alpha * g * (1 + p.cubic * g * g)) \
        * (u + p.shift)


def exact_layers(s, m, sq, tokens):
    eps, pages, states = s.norm_eps, [], []
    x = f64(m.embed[tokens])
    if s.positions:
        x = x + f64(m.pos_table[sq.pos])
    if s.embed_norm:
        x = rms(x, eps) * f64(m.embed_norm)

    def norm(y, w):
        parts = y.view(len(y), s.norm_groups, -1)
        return rms(parts, eps).view_as(y) * (f64(w) + m.norm_off)

    def added(x, y, w):
        if s.post_alpha is not None:
            return norm(s.post_alpha * x + y, w)
        return x + norm(y, w)

    results = [x]
    for i, (ly, w) in enumerate(zip(s.layers, m.layers)):
        y = exact_mixer(s, m, i, ly.mixer, w,
                        norm(x, w.pre1) if s.pre_norms else x, sq, pages,
                        states)
        x = added(x, y, w.norm1)
        y = exact_feed(s, ly.ff, w, norm(x, w.pre2) if s.pre_norms else x)
        x = added(x, y, w.norm2)
        if s.depth_average:
            results.append(x)
            x = sum(a * r for a, r in zip(f64(m.averages[i]), results))
    x = x[sq.last]
    x = rms(x.view(len(x), s.norm_groups, -1), eps).view_as(x)
    logits = x * f64(m.head_norm) @ f64(m.head).T
    if sq.decode:
        return [logits] + states
    return [logits[0] if len(sq.parts) == 1 else logits] + \
        in_pages(sq, m, pages) + states


def in_pages(sq, m, rows):
    """Rows of the fresh sequences as the pool holds them: pages in order."""
    out = []
    for t in rows:
        pool = t.new_zeros(m.cache.pages + 1, PAGE, *t.shape[1:])
        at = 1
        for p in sq.parts:
            n = p.stop - p.start
            for c in range(0, n, PAGE):
                pool[at, :min(PAGE, n - c)] = t[p][c:c + PAGE]
                at += 1
        out.append(pool.transpose(1, 2) if pool.dim() == 4 else pool)
    return out


def exact(case, seed):
    if case["kind"] == "sample":
        return None                    # whole numbers
    if case["kind"] == "experts":
        ff, x, logits, up, down = expert_inputs(case, seed)
        z = f64(logits)
        idx = torch.topk(z, ff.top, dim=-1).indices
        wt = (torch.sigmoid(z) if ff.sigmoid else z).gather(1, idx)
        if not ff.sigmoid:
            wt = torch.softmax(wt, -1)
        flat, y = idx.reshape(-1), x.new_zeros(
            idx.numel(), x.shape[1], dtype=torch.float64)
        xs = f64(x).repeat_interleave(ff.top, 0)
        for e in range(ff.experts):
            r = (flat == e).nonzero().squeeze(1)
            a = xs[r] @ f64(up[e]).T
            if ff.weigh_input:
                a = a * wt.reshape(-1)[r].unsqueeze(1)
            if ff.gated:               # rows in turns of 16 gate | 16 up
                g, u = a.view(len(r), -1, 2, 16).unbind(2)
                a = glu(g.reshape(len(r), -1), u.reshape(len(r), -1),
                        ff.unit or DenseFF(ff.ff, alpha=1.0, shift=0.0))
            else:
                a = torch.relu(a) ** 2
            y[r] = a @ f64(down[e]).T
        return y, wt
    with torch.no_grad():
        s, m = build(case, seed)
        if case["kind"] == "decode":
            slots = fill(case, seed, s, m)
            tokens = token_ids(case, seed, s.vocab, [case["rows"]])[0]
        else:
            slots = [m.cache.alloc(n) for n in lengths(case)]
            tokens = torch.cat(token_ids(case, seed, s.vocab, lengths(case)))
        sq = Sequences(case, s, m, slots)
        f = exact_layers if isinstance(s, HybridSpec) else exact_llama
        return f(s, m, sq, tokens)
