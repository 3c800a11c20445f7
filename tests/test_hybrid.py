"""Layer-list models (Birepel) against the plain implementation in
hybrid_oracle: on the CPU in f32, on the GPU in f32 and bf16."""

import array
import io
import json
import os
import subprocess
import sys
import time

import numpy as np
import pytest
import torch

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import hybrid_oracle as oracle  # noqa: E402
from hybrid_helpers import (EXACT, REPO, RUNS, Bytes,  # noqa: E402
                            check_wanted_rows_alone, close, errors, feed,
                            meta_for, one_thread,  # noqa: F401
                            portions, whole)

from gridllm_amd.config import EngineConfig  # noqa: E402
from gridllm_amd.engine import InferenceEngine  # noqa: E402
from gridllm_amd.models.hybrid import HybridModel  # noqa: E402
from gridllm_amd.models.paged import PagedCache  # noqa: E402
from gridllm_amd.models.registry import (get_spec, read_birepel,  # noqa: E402
                                         resolve_spec)
from gridllm_amd.ops import hybrid as hops  # noqa: E402

def attn(heads=4, kv_heads=2, dim=32, vdim=32, scale=0.2, coef=0.25, every=16):
    return {"heads": heads, "kv_heads": kv_heads, "dim": dim, "vdim": vdim,
            "scale": scale, "q_temp": {"coef": coef, "every": every}}


def rec(heads=2, dim=32, vdim=32, gate_cap=6.0):
    return {"heads": heads, "dim": dim, "vdim": vdim, "gate_cap": gate_cap}


def dense(ff=96, limit=0.8):
    return {"kind": "dense", "ff": ff, "limit": limit}


def routed(experts=5, top=2, ff=40):
    return {"kind": "moe", "expert": {"ff": ff},
            "router": {"experts": experts, "top": top}}


def config(*layers, vocab=130, width=96, positions=512, eps=1e-5):
    """layers: (mixer, mlp) or (mixer, mlp, weights_of)."""
    out = []
    for ly in layers:
        d = {"type": "attention" if "kv_heads" in ly[0] else "mlstm",
             "mixer": ly[0], "mlp": ly[1]}
        if len(ly) > 2:
            d["weights_of"] = ly[2]
        out.append(d)
    return {"architecture": "Birepel", "layers": out, "vocab": vocab,
            "width": width, "max_positions": positions, "norm": {"eps": eps}}


# every branch at once, sizes that need padding, a shared layer ahead of and
# behind its owner
FULL = config((attn(6, 3, 40, 24), None),
              (rec(3, 40, 72), dense()),
              (attn(4, 1, 72, 80, every=5), routed()),
              (rec(1, 24, 16, gate_cap=2.5), routed(4, 4, 24)),
              (rec(3, 40, 72), dense(), 1),
              (attn(4, 1, 72, 80, every=5), routed(), 2))


def weights_of(cfg, seed=0):
    return oracle.random_weights(cfg, seed)


def build(cfg, run, seed=0, slots=5, pool=0, W=None):
    dev, dtype = run
    m = HybridModel(read_birepel(cfg), device=dev, dtype=dtype,
                    kv_slots=slots, kv_tokens=pool, random_init=False)
    W = W or weights_of(cfg, seed)
    m._assemble(lambda name: W[name].to(dev))
    if dev != "cpu" and dtype == "bf16":
        m.interleave_gateup()
    return m


def tokens(n, cfg=FULL, seed=0):
    return np.random.default_rng(seed).integers(0, cfg["vocab"], n).tolist()


# ------------------------------------------------------------ each mechanism

ALONE = {
    "attention": config((attn(), None)),
    "attention-one-kv-head": config((attn(12, 1, 64, 64), None)),
    "attention-own-kv-heads": config((attn(3, 3, 96, 128), None)),
    "attention-wide-heads": config((attn(2, 1, 160, 136, scale=0.1), None)),
    "attention-no-temperature": config((attn(coef=0.0, every=1), None)),
    "mlstm": config((rec(), None)),
    "mlstm-narrow-keys": config((rec(2, 48, 200), None)),
    "mlstm-wide-keys": config((rec(1, 130, 40), None)),
    "mlstm-widest-keys": config((rec(1, 300, 64), None)),
    "mlstm-one-head": config((rec(1, 64, 64, gate_cap=1.0), None)),
    "dense": config((rec(1, 16, 16), dense(200, 0.5))),
    "dense-wide-limit": config((rec(1, 16, 16), dense(64, 100.0))),
    "routed": config((rec(1, 16, 16), routed(7, 3, 64))),
    "routed-one": config((rec(1, 16, 16), routed(9, 1, 24))),
    "routed-all": config((rec(1, 16, 16), routed(3, 3, 72))),
    "routed-many": config((rec(1, 16, 16), routed(80, 6, 16))),
    "wide-residual": config((rec(), dense()), width=200),
    "coarse-eps": config((attn(), dense()), eps=0.05),
}


@pytest.mark.parametrize("run", RUNS)
@pytest.mark.parametrize("name", sorted(ALONE))
def test_mechanism_alone(name, run):
    cfg = ALONE[name]
    m = build(cfg, run)
    ids = tokens(150, cfg)
    trail = []
    slot = m.cache.alloc(0)
    got = m.forward_step([(slot, ids, list(range(len(ids))))], trail=trail)
    want, layers = oracle.forward(cfg, weights_of(cfg), ids)
    close(got, want, run)
    close(trail[-1], layers[-1], run)


@pytest.mark.parametrize("run", RUNS)
def test_all_layers(run):
    m = build(FULL, run)
    ids = tokens(200)
    trail = []
    slot = m.cache.alloc(0)
    got = m.forward_step([(slot, ids, list(range(200)))], trail=trail)
    want, layers = oracle.forward(FULL, weights_of(FULL), ids)
    for a, b in zip(trail, layers):
        close(a, b, run, coarse=0.1, odd=0.1)
    close(got, want, run, coarse=0.1, odd=0.1)


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [3, 40, 130, 600])
def test_experts_at_every_batch_size(batch):
    """Few pairs and many take different GEMMs; tiles run over and under."""
    e, w, f, top = 6, 128, 192, 2
    g = torch.Generator().manual_seed(3)
    x = torch.randn(batch, w, generator=g).bfloat16()
    z = torch.randn(batch, e, generator=g)
    up = (torch.randn(e, f, w, generator=g) * w ** -0.5).bfloat16()
    dn = (torch.randn(e, w, f, generator=g) * f ** -0.5).bfloat16()
    # one expert far more popular than the others
    z[:, 2] += 2.0
    ye, wt, _ = hops.moe(x.cuda(), z.cuda(), up.cuda(), dn.cuda(), top)
    idx = torch.topk(z, top).indices
    sm = torch.softmax(torch.topk(z, top).values, -1)
    assert torch.allclose(wt.cpu(), sm, atol=1e-6)
    a = torch.relu(torch.einsum("nw,nkfw->nkf", x.float(), up[idx].float()))
    want = torch.einsum("nkf,nkwf->nkw", (a ** 2).bfloat16().float(),
                        dn[idx].float())
    assert float(errors(ye.view(batch, top, w), want).max()) < 0.02


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [1, 16, 17, 32, 33, 54, 55, 64])
def test_experts_at_the_edges_of_tiles(batch):
    """The same where one block routes and where several do, and with tiles of 16,
    32 and 128 rows."""
    from gridllm_amd.ops import hip_hybrid
    test_experts_at_every_batch_size(batch)
    assert [hip_hybrid._expert_rows(2 * n, 6) for n in (32, 33, 54, 55)] == \
        [16, 32, 32, 128]


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["squared", "gated", "weighed"])
@pytest.mark.parametrize("batch,rows", [(70, 128), (200, 192), (333, 256),
                                        (700, 128)])
def test_experts_by_wide_tiles(batch, rows, act, monkeypatch):
    """What tiles of 128 x 128 give, to the bit: columns that the tiles do not
    divide, behind which the next expert's weights lie, an expert without rows, one
    with most of them, and K of few stages and of many."""
    from gridllm_amd.ops import hip_hybrid
    e, w, f, top = 7, 1088, 320, 2
    g = torch.Generator().manual_seed(batch)
    x, up, dn = (torch.randn(*s, generator=g).bfloat16().cuda() for s in (
        (batch, w), (e, f if act == "squared" else 2 * f, w), (e, w, f)))
    z = torch.randn(batch, e, generator=g)
    z[:, 3] -= 50.0
    z[:, 5] += 2.0
    how = hops.Choice(top, sigmoid=act == "weighed",
                      weigh_input=act == "weighed")
    wide = hip_hybrid._experts_wide
    seen = hip_hybrid._expert_rows
    monkeypatch.setattr(hip_hybrid, "_expert_rows", lambda *a: rows)
    got = hops.moe(x, z.cuda(), up * 0.1, dn, how)
    assert wide(up, dn, batch, batch * top) == (up.shape[1:], dn.shape[1:])
    monkeypatch.setattr(hip_hybrid, "_experts_wide", lambda *a: ())
    monkeypatch.setattr(hip_hybrid, "_expert_rows", lambda *a: 128)
    want = hops.moe(x, z.cuda(), up * 0.1, dn, how)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    sizes = ((1024, 3072), (3072, 1024))
    assert [seen(8 * n, 64, sizes) for n in (512, 768, 1536)] == [128, 192, 256]
    assert not wide(up[..., :192], dn, batch, batch * top)
    assert not wide(up, dn, 1 << 20, 1 << 21)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 64, 100, 300])
def test_fused_gate_projection_takes_the_constants(m):
    """Every gated-unit path with a limit that cuts: the plain op, the
    interleaved one, and the projection with the fused epilogue."""
    from gridllm_amd.ops import hip_ops
    from gridllm_amd.ops.reference import Glu
    glu = Glu(1.702, 0.6, 1.0)
    f, k = 256, 192
    g = torch.Generator().manual_seed(m)
    x = torch.randn(m, k, generator=g).bfloat16().cuda()
    w = (torch.randn(2 * f, k, generator=g) * k ** -0.5).bfloat16().cuda()
    il = w.view(2, f // 64, 64, k).transpose(0, 1).reshape(2 * f, k).contiguous()
    gu = (x.float() @ w.float().T).cpu().double()
    want = oracle.clamped_glu(gu[:, :f], gu[:, f:], 0.6)
    rows = torch.nn.functional.linear(x, w)
    outs = [hip_ops.swiglu(rows, glu=glu),
            hip_ops.swiglu_il(torch.nn.functional.linear(x, il), glu=glu)]
    if m <= 256:
        outs += [hip_ops.gemm_proj(x, il, splitk=s, fuse_swiglu=True, glu=glu)
                 for s in (1, 3)]
    for got in outs:
        assert float(errors(got, want).max()) < 0.02
    exact = hops.glu((x.float() @ w.float().T), glu)
    assert float(errors(exact, want).max()) < 1e-4


# ------------------------------------------- keys and tokens that stand out

CUTS = {"whole": [300], "decode-tail": [190, 1], "pairs": [250, 2],
        "odd": [63, 2, 1, 64, 65]}


@pytest.mark.parametrize("run", RUNS)
@pytest.mark.parametrize("how", sorted(CUTS))
def test_one_key_stands_out(how, run):
    """Every query looks for one key: the first, the neighbours of page
    borders, itself, the previous one; for some it is the next one, which it
    must not see. Sinks from negligible to dominating."""
    dev, dtype = run
    H, G, d, n = 4, 2, 64, 300
    cfg = config((attn(H, G, d, d), None), positions=320)
    cache = PagedCache(read_birepel(cfg), 3, 320, torch.device(dev),
                       torch.float32 if dtype == "fp32" else torch.bfloat16)
    cache.alloc(70)                       # page 1 and 2 belong to another
    slot = cache.alloc(0)
    g = torch.Generator().manual_seed(5)
    k = torch.randn(n, G, d, generator=g)
    v = torch.randn(n, G, d, generator=g)
    gate = torch.randn(n, H, generator=g)
    near = [0, 1, 62, 63, 64, 65, 127, 128, 191, 192, 255, 256]
    q = torch.zeros(n, H, d)
    for p in range(n):
        for h in range(H):
            targets = [t for t in near if t <= p] + [p, max(p - 1, 0),
                                                     min(p + 1, n - 1)]
            q[p, h] = k[targets[(p * 7 + h * 5) % len(targets)], h // (H // G)]
    sink = torch.tensor([-30.0, 0.0, 6.0, 14.0])
    row = torch.cat([q.view(n, -1), k.view(n, -1), v.view(n, -1), gate], 1)
    row = torch.nn.functional.pad(row, (0, 60)).to(cache.k[0].dtype)
    coef, every, scale = 0.35, 32, 0.13
    rr = row.double()
    qd, kd, vd, gd, _ = rr.split([H * d, G * d, G * d, H, 60], dim=1)
    temp = oracle.query_temperature(torch.arange(n), coef, every)
    want = oracle.attend(
        oracle.rms(qd.view(n, H, d), 1e-5) * temp.view(n, 1, 1),
        oracle.rms(kd.view(n, G, d), 1e-5), vd.view(n, G, d), scale,
        sink.double()) * torch.sigmoid(gd)[:, :, None]
    got = []
    for at, ln in portions(n, CUTS[how]):
        cache.extend([slot], [ln])
        st = meta_for(cache, slot, at, ln, dev)
        part = row[at:at + ln].to(dev).contiguous()
        qn = hops.qknorm_kv(part, cache.k[0], cache.v[0], st, H, G, d, 1e-5,
                            coef, every)
        got.append(hops.paged_attn(
            qn, cache.k[0], cache.v[0], st, scale, sink.to(dev),
            part[:, (H + 2 * G) * d:(H + 2 * G) * d + H]))
    got = torch.cat(got).cpu().double()
    assert float((got - want).abs().max()) < (1e-4 if dtype == "fp32"
                                              else 0.06)


@pytest.mark.parametrize("run", RUNS)
@pytest.mark.parametrize("how", sorted(CUTS))
@pytest.mark.parametrize("dk,dv", [(64, 64), (128, 192)])
def test_one_token_is_remembered(how, run, dk, dv):
    """A token with a wide open input gate, at the first place and around
    chunk borders, is what later queries recall; one head forgets at once, one
    keeps everything, one sees a deep forget in the middle."""
    dev, dtype = run
    H, n, cap = 3, 300, 15.0
    cfg = config((rec(H, dk, dv, cap), None), positions=320)
    cache = PagedCache(read_birepel(cfg), 3, 320, torch.device(dev),
                       torch.float32)
    slot = cache.alloc(0)
    S, mst = cache.S[0], cache.m[0]
    S[slot], mst[slot] = 7.0, 3.0         # a predecessor's state
    g = torch.Generator().manual_seed(7)
    el = torch.float32 if dtype == "fp32" else torch.bfloat16
    q, k = torch.randn(2, n, H, dk, generator=g)
    v, gate = torch.randn(2, n, H, dv, generator=g)
    zi = torch.full((n, H), -9.0)
    zf = torch.full((n, H), 30.0)
    loud = [0, 63, 64, 65, 128, 191, 192, 250]
    for t in loud:
        zi[t] = 9.0
    for p in range(n):
        q[p] = k[max([t for t in loud if t <= p])] * 2
    zf[:, 1] = 4.0
    zf[:, 2] = torch.where(torch.arange(n) == 100, -40.0, 6.0)
    row = torch.cat([q.reshape(n, -1), k.reshape(n, -1), v.reshape(n, -1),
                     gate.reshape(n, -1)], 1).to(el)
    gates = torch.cat([zi, zf], 1)
    rr = row.double()
    qd, kd, vd, gd = rr.split([H * dk, H * dk, H * dv, H * dv], dim=1)
    li, lf = oracle.mlstm_log_gates(zi.double(), zf.double(), cap)
    o = oracle.mlstm_run(qd.view(n, H, dk) * dk ** -0.5, kd.view(n, H, dk),
                         vd.view(n, H, dv), li, lf)
    norm = torch.randn(H * dv, generator=g)
    want = oracle.rms(o, 1e-5).reshape(n, -1) * norm.double() * \
        torch.sigmoid(gd)
    got = []
    for at, ln in portions(n, CUTS[how]):
        cache.extend([slot], [ln])
        got.append(hops.mlstm(row[at:at + ln].to(dev).contiguous(),
                              gates[at:at + ln].to(dev).contiguous(), S, mst,
                              norm.to(dev), meta_for(cache, slot, at, ln, dev),
                              dk, dv, cap, 1e-5))
    got = torch.cat(got).cpu().double()
    e = errors(got.view(n, H, dv).transpose(1, 2).reshape(n, -1),
               want.view(n, H, dv).transpose(1, 2).reshape(n, -1))
    assert float(e.max()) < (3e-4 if dtype == "fp32" else 0.02)


# ----------------------------------------------- cuts, batches, pages, slots

@pytest.mark.parametrize("run", RUNS)
@pytest.mark.parametrize("sizes", [[1], [2], [3], [63, 2], [64], [100, 1],
                                   [130, 1, 7]], ids=str)
def test_cuts_do_not_matter(sizes, run):
    m = build(FULL, run)
    ids = tokens(140, seed=1)
    want, _ = oracle.forward(FULL, weights_of(FULL), ids)
    slot = m.cache.alloc(0)
    close(feed(m, slot, ids, sizes), want, run, coarse=0.1, odd=0.1)


@pytest.mark.parametrize("run", RUNS)
def test_wanted_rows_alone(run):
    check_wanted_rows_alone(lambda: build(FULL, run), tokens, run)


@pytest.mark.parametrize("run", RUNS)
@pytest.mark.parametrize("where", [("run", torch.int64), ("run", torch.int32),
                                   ("run", None), ("cpu", torch.int64)])
def test_prompts_tokens_from_anywhere(where, run):
    """Several prompts' tokens of one type on the model's device (one copy), of
    several types, and on the host: the same step, so the same results."""
    m = build(FULL, run)
    lists = [tokens(n, seed=n) for n in (40, 1, 70)]

    def logits(tensors):
        slots = [m.cache.alloc(0) for _ in tensors]
        out = m.forward_prefill_batch(tensors, slots)
        for slot in slots:
            m.cache.free(slot)
        return out
    dev = run[0] if where[0] == "run" else "cpu"
    kinds = [where[1] or kind for kind in (torch.int64, torch.int32, torch.int64)]
    got = logits([torch.tensor(ids, dtype=kind, device=dev)
                  for ids, kind in zip(lists, kinds)])
    assert torch.equal(got, logits([torch.tensor(ids) for ids in lists]))
    # arrays, beside tensors and alone, and an iterator over them
    arrays = [np.array(lists[0], dtype=np.int32), torch.tensor(lists[1], device=dev),
              array.array("q", lists[2])]
    assert torch.equal(got, logits(arrays))
    slots = [m.cache.alloc(0) for _ in lists]
    assert torch.equal(got, m.forward_prefill_batch(
        (np.array(ids) for ids in lists), slots))
    for slot in slots:
        m.cache.free(slot)
    slot = m.cache.alloc(0)
    alone = m.forward_prefill(np.array(lists[2]), slot)
    m.cache.free(slot)
    slot = m.cache.alloc(0)
    assert torch.equal(alone, m.forward_prefill(torch.tensor(lists[2]), slot))
    m.cache.free(slot)


@pytest.mark.parametrize("run", RUNS)
def test_unequal_batch_against_each_alone(run):
    m = build(FULL, run)
    seqs = {s: tokens(n, seed=s) for s, n in ((1, 150), (2, 3), (3, 70),
                                              (4, 97))}
    want = {s: oracle.forward(FULL, weights_of(FULL), ids)[0]
            for s, ids in seqs.items()}
    # portions of some beside single tokens of others; one pauses
    steps = [{1: 64, 2: 1, 3: 2}, {1: 5, 3: 63, 4: 30}, {1: 1, 3: 1, 4: 2},
             {1: 60, 2: 1, 4: 64}, {1: 1, 2: 1, 3: 1, 4: 1}, {3: 2}, {1: 18},
             {1: 1, 3: 1}]
    slots = {s: m.cache.alloc(0) for s in seqs}
    at = {s: 0 for s in seqs}
    got = {s: [] for s in seqs}
    for st in steps:
        out = m.forward_step([(slots[s], seqs[s][at[s]:at[s] + n],
                               list(range(n))) for s, n in st.items()]).cpu()
        for (s, n), part in zip(st.items(), out.split(list(st.values()))):
            got[s].append(part)
            at[s] += n
    assert at == {s: len(v) for s, v in seqs.items()}
    for s in seqs:
        close(torch.cat(got[s]), want[s], run, coarse=0.1, odd=0.2)


@pytest.mark.parametrize("run", RUNS)
def test_wanted_places_come_in_order(run):
    m = build(FULL, run)
    a, b = tokens(20, seed=1), tokens(30, seed=2)
    wa, wb = whole(m, a), whole(m, b)
    s1, s2, s3 = (m.cache.alloc(0) for _ in range(3))
    out = m.forward_step([(s1, a, [19, 3]), (s3, [5], []),
                          (s2, b, [7, 7, 0])]).cpu()
    close(out, torch.cat([wa[[19, 3]], wb[[7, 7, 0]]]), run, exact=1e-4,
          coarse=0.1, odd=0.4)
    assert m.forward_step([(s1, [1, 2], [])]).shape == (0, FULL["vocab"])


@pytest.mark.parametrize("run", RUNS)
def test_pages_and_slots_are_used_again(run):
    """A pool that only fits if everything is given back, in an order that
    scatters the pages of later sequences."""
    m = build(FULL, run, slots=3, pool=64 * 7)
    first = {}
    for rnd in range(3):
        s1, s2 = m.cache.alloc(0), m.cache.alloc(0)
        a, b = tokens(150, seed=10), tokens(140, seed=11)
        ga, gb = [], []
        for i in range(0, 150, 30):           # interleave the page demand
            ga.append(m.forward_step([(s1, a[i:i + 30], [0, 29])]))
            if i < 140:
                part = b[i:i + 30]
                gb.append(m.forward_step([(s2, part, [len(part) - 1])]))
        first.setdefault("a", torch.cat(ga).cpu())
        first.setdefault("b", torch.cat(gb).cpu())
        close(torch.cat(ga).cpu(), first["a"], run, exact=1e-4,
              coarse=0.1, odd=0.1)
        close(torch.cat(gb).cpu(), first["b"], run, exact=1e-4,
              coarse=0.1, odd=0.1)
        m.cache.free(s2 if rnd else s1)
        s3 = m.cache.alloc(0)
        c = tokens(130, seed=12)
        close(feed(m, s3, c, [100, 1])[[0, 129]],
              oracle.forward(FULL, weights_of(FULL), c)[0][[0, 129]], run,
              coarse=0.1, odd=0.5)
        m.cache.free(s3)
        m.cache.free(s1 if rnd else s2)
    assert len(m.cache._free_pages) == 7 and m.cache.n_free == 1


def test_pool_promises():
    spec = read_birepel(config((attn(), None), positions=256))
    c = PagedCache(spec, 4, 256, torch.device("cpu"), torch.float32,
                   pool_tokens=64 * 8)
    assert c.n_free == 2                       # two of full length
    a = c.alloc(130)                           # three pages set aside
    assert c.n_free == 1
    b = c.alloc(0)
    c.extend([b], [256])
    with pytest.raises(RuntimeError, match="pages"):
        c.alloc(128)                           # only one is not spoken for
    c.extend([a], [130])
    with pytest.raises(RuntimeError, match="cache for"):
        c.extend([b], [1])                     # longer than the cache's bound
    d = c.alloc(0)
    c.extend([d], [64])
    with pytest.raises(RuntimeError, match="out of pages"):
        c.extend([d], [1])
    held = [set(c._held[s]) for s in (a, b, d)]
    assert sum(map(len, held)) == len(set().union(*held)) == 8
    assert 0 not in set().union(*held)
    for s in (a, b, d):
        c.free(s)
    assert c.n_free == 2 and c._owed == 0 and len(c._free_pages) == 8
    for _ in range(4):
        c.alloc(0)
    with pytest.raises(RuntimeError, match="slots"):
        c.alloc(0)


def test_bad_steps_are_refused():
    m = build(FULL, ("cpu", "fp32"))
    s = m.cache.alloc(0)
    for entries in ([(s, [], [])], [(s, [1], [1])], [(s, [1], []), (s, [2], [])],
                    [(s, [FULL["vocab"]], [])], [(s, [-1], [])]):
        with pytest.raises(ValueError):
            m.forward_step(entries)


# ------------------------------------------------- configuration and weights

def test_config_reader():
    spec = read_birepel(FULL)
    assert [spec.owner(i) for i in range(6)] == [0, 1, 2, 3, 1, 2]
    assert spec.params == sum(v.numel() for v in weights_of(FULL).values())
    assert spec.max_seq_len == FULL["max_positions"]

    def broken(change):
        c = json.loads(json.dumps(FULL))
        change(c)
        with pytest.raises((ValueError, KeyError)):
            read_birepel(c)

    broken(lambda c: c["layers"][0]["mixer"].pop("scale"))
    broken(lambda c: c["layers"][0]["mixer"].update(window=64))
    broken(lambda c: c["layers"][0].update(type="conv"))
    broken(lambda c: c["layers"][1]["mlp"].update(kind="other"))
    broken(lambda c: c["layers"][4]["mixer"].update(heads=2))
    broken(lambda c: c["layers"][4].update(weights_of=4))
    broken(lambda c: c["layers"][2]["mlp"]["router"].update(top=6))
    broken(lambda c: c["layers"][0]["mixer"].update(kv_heads=4))


@pytest.fixture
def checkpoint(tmp_path):
    from safetensors.torch import save_file
    save_file(weights_of(FULL, 3), str(tmp_path / "model.safetensors"))
    (tmp_path / "config.json").write_text(json.dumps(FULL))
    return tmp_path


def test_checkpoint_describes_itself(checkpoint):
    spec = resolve_spec("llama3.2:1b", str(checkpoint))
    assert (spec.family, spec.name) == ("birepel", "birepel:custom")
    assert resolve_spec("mine", str(checkpoint), 100).max_seq_len == 100
    assert get_spec("mine").hidden == FULL["width"]
    (checkpoint / "config.json").write_text('{"architecture": "Else"}')
    with pytest.raises(ValueError, match="unknown architecture"):
        resolve_spec("mine", str(checkpoint))


def test_checkpoint_errors(checkpoint):
    from safetensors.torch import save_file
    m = HybridModel(read_birepel(FULL), dtype="fp32", random_init=False)
    assert m.load_safetensors(str(checkpoint)) == len(weights_of(FULL))
    W = weights_of(FULL, 3)
    W["l0.norm1"] = W["l0.norm1"][:-1].clone()
    save_file(W, str(checkpoint / "model.safetensors"))
    with pytest.raises(ValueError, match="l0.norm1"):
        m.load_safetensors(str(checkpoint))
    del W["l0.norm1"]
    save_file(W, str(checkpoint / "model.safetensors"))
    with pytest.raises(KeyError, match="l0.norm1"):
        m.load_safetensors(str(checkpoint))


# --------------------------------------------------- engine and its schedule

def engine_for(checkpoint, run, **kw):
    kw = {"max_seq_len": 256, "max_batch_size": 4, "autotune": False} | kw
    return InferenceEngine(EngineConfig(
        weights_path=str(checkpoint), device=run[0], dtype=run[1], **kw))


def greedy(ids, steps, seed=3):
    """Greedy continuation by the plain implementation, and how far the
    winner stood above the second at each step."""
    W, ids, gaps = weights_of(FULL, seed), list(ids), []
    for _ in range(steps):
        z = oracle.forward(FULL, W, ids)[0][-1]
        top = torch.topk(z, 2)
        gaps.append(float(top.values[0] - top.values[1]))
        ids.append(int(top.indices[0]))
    return ids[-steps:], gaps


GREEDY = {"temperature": 0.0, "num_predict": 8}
# bytes below the vocabulary's size
PROMPTS = ["3 + 4 = ", "x", "A much longer prompt, so that it takes more than "
           "one page and a few portions to run it all ...... ", "!"]


@pytest.mark.parametrize("run", EXACT)
@pytest.mark.parametrize("chunk", [8192, 5])
def test_greedy_generation(checkpoint, run, chunk):
    """Through generate, generate_batch and the continuous batcher, with whole
    prompts and with portions of five tokens beside decoding rows."""
    from gridllm_amd.engine.batcher import Batcher
    eng = engine_for(checkpoint, run, prefill_chunk=chunk)
    eng.tokenizer = Bytes(FULL["vocab"])
    want, gaps = zip(*(greedy(eng.tokenizer.encode(p), 8) for p in PROMPTS))
    assert min(min(g) for g in gaps) > 1e-3        # no close call in the test
    free = eng.model.cache.n_free
    assert [eng.generate(p, GREEDY).token_ids for p in PROMPTS] == list(want)
    out = eng.generate_batch([(p, GREEDY) for p in PROMPTS])
    assert [r.token_ids for r in out] == list(want)
    assert all(r.prompt_eval_duration > 0 and r.done_reason == "length"
               for r in out)
    b = Batcher(eng)
    try:
        futs = [b.submit_generate(p, GREEDY) for p in PROMPTS * 3]
        assert [f.result(60).token_ids for f in futs] == list(want) * 3
        deadline = time.time() + 10
        while eng.model.cache.n_free != free and time.time() < deadline:
            time.sleep(0.02)
    finally:
        b.shutdown()
    assert eng.model.cache.n_free == free
    assert len(eng.embed(["abc", "defg"])[1]) == FULL["width"]


def test_small_pool_serves_more_than_it_holds(checkpoint):
    """A pool for two full sequences, a dozen requests in flight."""
    from gridllm_amd.engine.batcher import Batcher
    eng = engine_for(checkpoint, ("cpu", "fp32"), kv_tokens=512)
    eng.tokenizer = Bytes(FULL["vocab"])
    want = [eng.generate(p, GREEDY).token_ids for p in PROMPTS]
    b = Batcher(eng)
    try:
        futs = [b.submit_generate(p, GREEDY) for p in PROMPTS * 3]
        assert [f.result(60).token_ids for f in futs] == want * 3
    finally:
        b.shutdown()


def test_cancel_while_the_prompt_runs(checkpoint):
    import threading
    eng = engine_for(checkpoint, ("cpu", "fp32"), prefill_chunk=4)
    eng.tokenizer = Bytes(FULL["vocab"])
    ev = threading.Event()
    free = eng.model.cache.n_free
    rows = eng.start_rows([(PROMPTS[2], GREEDY, None, ev, None),
                           (PROMPTS[1], GREEDY, None, None, None)])
    rows = eng.step_rows(rows)
    ev.set()
    done = []
    while rows:
        left = eng.step_rows(rows)
        done += [r for r in rows if r.done]
        rows = left
    assert sorted(r.result.done_reason for r in done) == ["cancelled",
                                                          "length"]
    assert eng.model.cache.n_free == free


def test_context_ends_without_a_shift(checkpoint):
    eng = engine_for(checkpoint, ("cpu", "fp32"), max_seq_len=40)
    eng.tokenizer = Bytes(FULL["vocab"])
    r = eng.generate("0123456789", {"temperature": 0.0})
    assert r.done_reason == "length" and 10 + r.eval_count <= 40


def test_registered_model_serves():
    eng = InferenceEngine(EngineConfig(model="tiny-birepel", device="cpu",
                                       max_batch_size=2, max_seq_len=128))
    r = eng.generate("hello", {"temperature": 0.7, "seed": 5,
                               "num_predict": 6})
    assert r.eval_count == 6
    assert "tiny-birepel" in eng.model_names()
    assert eng.spec.model_info()["general.architecture"] == "birepel"


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
def test_long_decode_by_captured_graphs(checkpoint, dtype):
    """Decode-only steps replay captured graphs, between eager mixed steps and
    synchronizations; every step against the eager model, 150 tokens long and
    over page borders."""
    eng = engine_for(checkpoint, ("cuda:0", dtype))
    assert eng._graph_ok() and eng._graphs
    W = weights_of(FULL, 3)
    ref = build(FULL, ("cuda:0", dtype), W=W)
    ids = {i: tokens(190, seed=20 + i) for i in range(3)}
    a = {i: eng.open_sequence() for i in ids}
    b = {i: ref.cache.alloc(0) for i in ids}
    start = {0: 40, 1: 2, 2: 33}
    at = dict(start)
    eng.run_step([(a[i], ids[i][:n], []) for i, n in start.items()])
    ref.forward_step([(b[i], ids[i][:n], []) for i, n in start.items()])
    for step in range(150):
        live = [i for i in ids if not (i == 1 and step % 3 == 0)]
        n = {i: 2 if step % 31 == 30 and i == 2 else 1 for i in live}
        ent = [(i, ids[i][at[i]:at[i] + n[i]], [0]) for i in live
               if at[i] + n[i] <= 190]
        got = eng.run_step([(a[i], t, w) for i, t, w in ent])
        want = ref.forward_step([(b[i], t, w) for i, t, w in ent])
        close(got, want.cpu(), ("cuda:0", dtype), exact=1e-4, coarse=0.1, odd=0.4)
        for i, t, _ in ent:
            at[i] += len(t)
        if step % 10 == 0:
            torch.cuda.synchronize()
    close(eng.run_step([(a[0], [7], [0])]),
          oracle.forward(FULL, W, ids[0][:at[0]] + [7])[0][-1:],
          ("cuda:0", dtype), odd=1.0)


@pytest.mark.gpu
def test_uploads_far_ahead_of_the_stream():
    """Steps that nobody waits for queue up behind a busy stream; what they
    uploaded must not change under them."""
    from gridllm_amd.utils.pinned import PinnedUploader
    up = PinnedUploader(torch.device("cuda:0"))
    up.upload(np.zeros(100, dtype=np.int64))
    a = torch.randn(4096, 4096, device="cuda:0")
    torch.cuda.synchronize()
    for _ in range(20):
        a = a @ a * 1e-3
    got = [up.upload(np.full(100, i, dtype=np.int64)) for i in range(12)]
    assert [int(t.sum()) for t in got] == [100 * i for i in range(12)]


# ------------------------------------------------------------------- traces

def trace_lines():
    a, b = tokens(80, seed=1), tokens(3, seed=2)
    steps = [{"step": 0, "entries": [
                 {"id": "a", "tokens": a[:70], "want": [0, 69]},
                 {"id": "b", "tokens": b[:1], "want": [0]}], "end": []},
             {"step": 1, "entries": [
                 {"id": "b", "tokens": b[1:], "want": []}], "end": ["b"]},
             {"step": 2, "entries": [
                 {"id": "a", "tokens": a[70:71], "want": [0]}], "end": []},
             {"step": 3, "entries": [
                 {"id": "c", "tokens": b, "want": [2]},
                 {"id": "a", "tokens": a[71:], "want": [8]}],
              "end": ["a", "c"]}]
    W = weights_of(FULL, 3)
    la, lb = (oracle.forward(FULL, W, t)[0] for t in (a, b))
    want = {0: torch.stack([la[0], la[69], lb[0]]), 2: la[70:71],
            3: torch.stack([lb[2], la[79]])}
    return "".join(json.dumps(s) + "\n" for s in steps), want


def check_trace(out, want, run):
    assert sorted(os.listdir(out)) == [f"{k}.f32" for k in sorted(want)]
    for k, w in want.items():
        got = np.fromfile(os.path.join(out, f"{k}.f32"), dtype="<f4")
        close(torch.from_numpy(got).view(w.shape), w, run, coarse=0.1, odd=0.5)


@pytest.mark.parametrize("run", RUNS)
def test_trace_replay(checkpoint, tmp_path, run):
    from gridllm_amd import trace
    lines, want = trace_lines()
    out = tmp_path / "out"
    out.mkdir()
    eng = trace.make_engine(str(checkpoint),
                            {"fp32": "float32", "bf16": "bfloat16"}[run[1]],
                            256, run[0])
    acks = io.StringIO()
    trace.replay(eng, io.StringIO(lines), str(out), acks)
    assert acks.getvalue() == "".join(f"done {i}\n" for i in range(4))
    assert eng.model.cache.pages == 4 and len(eng.model.cache._free_pages) == 4
    check_trace(out, want, run)


def test_trace_program(checkpoint, tmp_path):
    lines, want = trace_lines()
    out = tmp_path / "out"
    out.mkdir()
    r = subprocess.run([os.path.join(REPO, "bin", "trace_run"), "--model",
                        str(checkpoint), "--dtype", "float32", "--out",
                        str(out), "--max-tokens", "256", "--device", "cpu"],
                       input=lines, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    assert [x for x in r.stdout.splitlines() if x.startswith("done")] == [
        f"done {i}" for i in range(4)]
    check_trace(out, want, ("cpu", "fp32"))


@pytest.mark.gpu
@pytest.mark.parametrize("entering", [False, True])
@pytest.mark.parametrize("dk,dv", [(64, 64), (128, 256), (64, 192), (192, 128),
                                   (64, 320)])
def test_mlstm_chunk_sizes(dk, dv, entering):
    """Decode rows and portions of whole and cut chunks in one step, for heads
    whose columns a block has all of (up to 256) or not; with normalisers that
    enter a portion's first chunk, and without."""
    from gridllm_amd.ops import reference_hybrid
    h, nd, lens = 2, 2, (1, 64, 130)
    g = torch.Generator().manual_seed(dk + dv)
    n = nd + sum(lens)
    entries, chunks, segs = [(0, 1, 0, 7), (1, 1, 1, 3)], [], []
    at = nd
    for i, ln in enumerate(lens):
        start = 0 if i == 2 else 5
        entries.append((at, ln, nd + i, start))
        segs.append((nd + i, start, len(chunks), -(-ln // 64)))
        chunks += [(at + c, min(64, ln - c), i, 0) for c in range(0, ln, 64)]
        at += ln
    pos = torch.cat([torch.arange(e[3], e[3] + e[1]) for e in entries])
    slot = torch.cat([torch.full((e[1],), e[2]) for e in entries])

    def t(rows):
        return torch.tensor(rows, dtype=torch.int32)
    meta = dict(nd=nd, pos=pos.int(), slot=slot.int(),
                table=torch.zeros(5, 1, dtype=torch.int32), max_len=200)
    rows = torch.randn(n, h * 2 * (dk + dv), generator=g).to(torch.bfloat16)
    gates = torch.randn(n, 2 * h, generator=g) * 3
    S = torch.randn(5, h, dv + 1, dk, generator=g)
    # denominators that no query makes small: sums of what is not negative (which
    # the norm behind them only shows with an eps of its size), or the chunk's own
    eps = 1.0 if entering else 1e-5
    if entering:
        rows[:, :2 * h * dk] = rows[:, :2 * h * dk].abs()
        S[:, :, dv] = S[:, :, dv].abs()
    else:
        S[:, :, dv] = 0.0
    m, norm = torch.rand(5, h, generator=g), torch.rand(h * dv,
                                                        generator=g) + 0.5
    S0, m0 = S.clone(), m.clone()
    want = reference_hybrid.mlstm(rows.float(), gates, S0, m0, norm,
                                  hops.StepMeta(segs=t(entries), **meta), dk,
                                  dv, 15.0, eps)
    dev = "cuda"
    S1, m1 = S.to(dev), m.to(dev)
    st = hops.StepMeta(chunks=t(chunks).to(dev), chunk_segs=t(segs).to(dev),
                       segs=t(entries).to(dev),
                       **{k: v.to(dev) if torch.is_tensor(v) else v
                          for k, v in meta.items()})
    got = hops.mlstm(rows.to(dev), gates.to(dev), S1, m1, norm.to(dev), st, dk,
                     dv, 15.0, eps).cpu().float()
    # bf16 result of a unit RMS row; bf16 weights of a chunk's values, 2^-9 each
    gate = torch.sigmoid(rows[:, -h * dv:].float()) * norm
    assert bool(((got - want).abs() <= 2 ** -8 * want.abs() +
                 2 ** -6 * gate + 1e-6).all())
    used = [e[2] for e in entries]
    assert float((S1.cpu()[used] - S0[used]).abs().max()) < \
        2 ** -11 * float(S0.abs().max())
    assert float((m1.cpu()[used] - m0[used]).abs().max()) < 1e-4


def test_a_step_says_what_its_states_take(monkeypatch):
    """Whether states go past the caches is decided by all recurrent layers' of a step,
    decoded or mixed, and by a call's own where there is no step."""
    from gridllm_amd.models import hybrid
    from gridllm_amd.ops import hip_hybrid
    m = build(FULL, ("cpu", "fp32"))
    states = [t for t in m.cache.S if t is not None]
    each = sum(t[0].numel() * t.element_size() for t in states)
    assert len(states) > 1 and m.cache.state_bytes == each
    seen = []
    real = hybrid.hops.mlstm

    def spy(rows, gates, S, mm, norm, st, *rest):
        seen.append(hip_hybrid._state_bytes(st, S, 3))
        return real(rows, gates, S, mm, norm, st, *rest)
    monkeypatch.setattr(hybrid.hops, "mlstm", spy)
    slot = m.cache.alloc(0)
    m.forward_prefill(np.array(tokens(5)), slot)
    m.cache.prepare_decode([slot])
    m.forward_decode(torch.tensor([3]), torch.tensor([slot], dtype=torch.int32))
    assert seen == [3 * each] * (2 * len(states))
    st = hops.StepMeta(nd=1, pos=None, slot=None, table=None, max_len=4)
    assert hip_hybrid._state_bytes(st, states[0], 3) == 12 * states[0][0].numel()


@pytest.mark.gpu
@pytest.mark.parametrize("n,h,more", [(57, 12, -1), (57, 12, 1), (90, 16, 1)])
def test_states_past_the_caches(n, h, more):
    """Decode rows of a step whose states are just less than what goes past the caches,
    or just more, and of several rounds of a block: the same as the rows one by one."""
    dk, dv = 128, 256
    g = torch.Generator(device="cuda").manual_seed(n)

    def r(*s):
        return torch.randn(*s, generator=g, device="cuda")
    rows = r(n, h * 2 * (dk + dv)).to(torch.bfloat16)
    gates, norm = r(n, 2 * h), r(h * dv).abs() + 0.5
    S, m = r(n, h, dv + 1, dk), r(n, h).abs()
    pos = torch.arange(n, device="cuda", dtype=torch.int32) % 3    # (0: fresh)
    slot = torch.randperm(n, generator=g, device="cuda").int()

    def step(at, S, m):
        st = hops.StepMeta(nd=at.stop - at.start, pos=pos[at], slot=slot[at],
                           table=torch.zeros(n, 1, dtype=torch.int32,
                                             device="cuda"), max_len=4,
                           state_bytes=200_000_000 // n + more)
        return hops.mlstm(rows[at].contiguous(), gates[at].contiguous(), S, m,
                          norm, st, dk, dv, 15.0, 1e-5)
    S1, m1 = S.clone(), m.clone()
    got = step(slice(0, n), S1, m1)
    want = torch.cat([step(slice(i, i + 1), S, m) for i in range(n)])
    assert torch.equal(got, want)
    assert torch.equal(S1, S) and torch.equal(m1, m)


@pytest.mark.gpu
@pytest.mark.parametrize("dk", [64, 128, 192, 512, 576])
@pytest.mark.parametrize("kind", [0, 1, 2])     # mLSTM, decays by channel, by head
def test_states_past_the_caches_of_all_kinds(kind, dk):
    """To the bit what goes through them: each width of a row's lanes, one round of a
    block and several, rows alone and segments of several tokens, whose states are read
    behind the stores of the token before."""
    from gridllm_amd.ops import hip_hybrid
    g = torch.Generator(device="cuda").manual_seed(dk)
    h, dv, lens = 2, 192, (1, 5, 2, 7)
    n, r = sum(lens), 192 + (kind == 0)

    def rand(*s):
        return torch.randn(*s, generator=g, device="cuda")

    def ints(rows):
        return torch.tensor(rows, dtype=torch.int32, device="cuda")
    rows, m = rand(n, h * 2 * (dk + dv)).to(torch.bfloat16), rand(n, h).abs()
    gates = (rand(n, 2 * h), -rand(n, h * dk).abs(), rand(h).abs() / 4)[kind]
    S, slot = rand(n, h, r, dk), torch.randperm(n, generator=g, device="cuda").int()
    segs = ints([(sum(lens[:i]), ln, i, 3 * (i % 2)) for i, ln in enumerate(lens)])
    pos = ints([i % 3 for i in range(n)])
    for of, count in ((segs, len(lens)), (None, n)):
        for rpb in (32, 128):
            out = []
            for step in (0, 1 << 40):
                o, s = torch.zeros(n, h, dv + 4, device="cuda"), S.clone()
                hip_hybrid._call("gh_rec_step", 0, kind, o, s, m, rows, gates, of, pos,
                                 slot, count, h, dk, dv, rows.shape[1], dk ** -0.5,
                                 15.0, rpb, step)
                out.append((o, s))
            assert not torch.equal(out[0][1], S)
            for a, w in zip(*out):
                assert a.isfinite().all() and torch.equal(a, w)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,dv", [(16, 256), (32, 192), (2, 256)])
@pytest.mark.parametrize("kind", ["gla", "mlstm"])
def test_states_of_many_chunks(kind, heads, dv):
    """Portions of one to four chunks, more and fewer blocks of the states than
    the chip has CUs, with columns that go into 128 and that do not."""
    from gridllm_amd.ops import reference_hybrid
    dk, lens = 128, (250, 192, 129, 65, 64, 63, 1, 100)
    n, at = sum(lens), 0
    entries, chunks, segs = [], [], []
    for i, ln in enumerate(lens):
        start = (i % 2) * 9
        entries.append((at, ln, i, start))
        segs.append((i, start, len(chunks), -(-ln // 64)))
        chunks += [(at + c, min(64, ln - c), i, 0) for c in range(0, ln, 64)]
        at += ln
    g = torch.Generator().manual_seed(heads + dv)
    pos = torch.cat([torch.arange(e[3], e[3] + e[1]) for e in entries])
    slot = torch.cat([torch.full((e[1],), e[2]) for e in entries])

    def step(dev):
        def t(rows):
            return torch.tensor(rows, dtype=torch.int32, device=dev)
        own = dict(segs=t(entries)) if dev == "cpu" else \
            dict(segs=t(entries), chunks=t(chunks), chunk_segs=t(segs))
        return hops.StepMeta(nd=0, pos=pos.int().to(dev),
                             slot=slot.int().to(dev), max_len=300,
                             table=torch.zeros(8, 1, dtype=torch.int32,
                                               device=dev), **own)
    rows = torch.randn(n, heads * 2 * (dk + dv), generator=g)
    rows = rows.to(torch.bfloat16)
    S = torch.randn(8, heads, dv + (kind == "mlstm"), dk, generator=g)
    m = torch.rand(8, heads, generator=g)
    norm = torch.ones(heads * dv)
    u, ba = torch.randn(n, 8, generator=g), torch.randn(heads * dk, generator=g)
    wa = torch.randn(8, heads * dk, generator=g)
    gates = torch.randn(n, 2 * heads, generator=g) * 3
    got = []
    for fn, dev, x in ((reference_hybrid, "cpu", rows.float()),
                       (hops, "cuda", rows.cuda())):
        s, mx = S.clone().to(dev), m.clone().to(dev)
        if kind == "gla":
            fn.gla(x, u.to(dev), wa.to(dev), ba.to(dev), s, norm.to(dev),
                   step(dev), dk, dv, 16.0, 1e-5)
        else:
            fn.mlstm(x, gates.to(dev), s, mx, norm.to(dev), step(dev), dk, dv,
                     15.0, 1e-5)
        got.append((s.cpu(), mx.cpu()))
    # keys as (hi, lo) pairs of bf16 are within 2^-17, a sum of 64 of a chunk's
    # products with unequal signs within that of its largest terms
    assert float((got[1][0] - got[0][0]).abs().max()) < \
        2 ** -13 * float(got[0][0].abs().max())
    assert float((got[1][1] - got[0][1]).abs().max()) < 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("heads,dv", [(12, 256), (2, 192)])
@pytest.mark.parametrize("kind", ["gla", "mlstm", "lightning"])
def test_outputs_of_many_chunks(kind, heads, dv):
    """Each token's output, behind the state that enters its chunk, and the state
    behind the last one: with 128 value columns a block, and with 64. Queries and keys
    are not negative, and the norm's eps is so large that it is a factor: results are
    sums of values, and the sums of their sizes bound the errors."""
    from gridllm_amd.ops import reference_hybrid
    dk, lens, eps = 128, (250, 192, 129, 65, 64, 63, 1, 100), 1e18
    n, at = sum(lens), 0
    entries, chunks, segs = [], [], []
    for i, ln in enumerate(lens):
        start = (i % 2) * 9
        entries.append((at, ln, i, start))
        segs.append((i, start, len(chunks), -(-ln // 64)))
        chunks += [(at + c, min(64, ln - c), i, 0) for c in range(0, ln, 64)]
        at += ln
    g = torch.Generator().manual_seed(heads + dv)
    pos = torch.cat([torch.arange(e[3], e[3] + e[1]) for e in entries])
    slot = torch.cat([torch.full((e[1],), e[2]) for e in entries])

    def step(dev):
        def t(rows):
            return torch.tensor(rows, dtype=torch.int32, device=dev)
        own = dict(segs=t(entries)) if dev == "cpu" else \
            dict(segs=t(entries), chunks=t(chunks), chunk_segs=t(segs))
        return hops.StepMeta(nd=0, pos=pos.int().to(dev),
                             slot=slot.int().to(dev), max_len=300,
                             table=torch.zeros(8, 1, dtype=torch.int32,
                                               device=dev), **own)
    rows = torch.randn(n, heads * 2 * (dk + dv), generator=g).to(torch.bfloat16)
    rows[:, :2 * heads * dk] = rows[:, :2 * heads * dk].abs()
    S = torch.randn(8, heads, dv + (kind == "mlstm"), dk, generator=g)
    S[:, :, dv:] = S[:, :, dv:].abs()
    m, norm = torch.rand(8, heads, generator=g), torch.full((heads * dv,), 1e9)
    u, ba = torch.randn(n, 8, generator=g), torch.randn(heads * dk, generator=g)
    wa = torch.randn(8, heads * dk, generator=g)
    gates = torch.randn(n, 2 * heads, generator=g) * 3
    decay = torch.rand(heads, generator=g) * 0.2 + 0.8
    decay = torch.stack([decay, decay.log()])

    def run(fn, dev, x, s):
        x, s, mx, w, st = x.to(dev), s.clone().to(dev), m.clone().to(dev), \
            norm.to(dev), step(dev)
        if kind == "gla":
            o = fn.gla(x, u.to(dev), wa.to(dev), ba.to(dev), s, w, st, dk, dv, 16.0,
                       eps)
        elif kind == "mlstm":
            o = fn.mlstm(x, gates.to(dev), s, mx, w, st, dk, dv, 15.0, eps)
        else:
            o = fn.lightning(x, s, decay.to(dev), w, st, dv, eps)
        return o.cpu().float(), s.cpu(), mx.cpu()
    sizes = rows.float()
    at = 2 * heads * dk
    sizes[:, at:at + heads * dv] = sizes[:, at:at + heads * dv].abs()
    want, S1, m1 = run(reference_hybrid, "cpu", rows.float(), S)
    room = run(reference_hybrid, "cpu", sizes, S.abs())[0].abs()
    got, S2, m2 = run(hops, "cuda", rows, S)
    # bf16: the result, and the weight of each of a chunk's own values
    assert bool(((got - want).abs() <= 2 ** -8 * (want.abs() + room)).all())
    assert float((S2 - S1).abs().max()) < 2 ** -13 * float(S1.abs().max())
    assert float((m2 - m1).abs().max()) < 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("n,w,top", [(3, 2048, 2), (5, 3072, 8), (2, 4160, 3),
                                     (4, 8192, 2)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_post_norm_of_pairs(dtype, n, w, top):
    """A row per (token, expert) by its weight: one turn and two, 256 threads and
    512."""
    from gridllm_amd.ops import reference_hybrid
    g = torch.Generator().manual_seed(w)
    x, a = torch.randn(n, w, generator=g), torch.rand(w, generator=g)
    y = torch.randn(n * top, w, generator=g).to(dtype)
    wt = torch.rand(n, top, generator=g)
    x1, b1 = x.cuda(), torch.empty(n, w, dtype=dtype, device="cuda")
    hops.post_norm(x1, b1, y.cuda(), a.cuda(), 1.0, w, 1e-5, wt.cuda())
    x2, b2 = x.double(), torch.empty(n, w, dtype=torch.float64)
    reference_hybrid.post_norm(x2, b2, y.double(), a.double(), 1.0, w, 1e-5,
                               wt.double())
    # f32: a sum of `top` and one of w squares
    assert float((x1.cpu() - x2).abs().max()) < 1e-5 * float(x2.abs().max())
    assert torch.equal(b1, x1.to(dtype))


@pytest.mark.gpu
@pytest.mark.parametrize("n,w,parts,size", [(1, 64, 2, 8), (24, 3072, 5, 384),
                                            (3, 1088, 9, 4), (5, 4160, 3, 8),
                                            (2, 8192, 2, 128)])
def test_norms_add_parts(n, w, parts, size):
    """Partial sums against the sum that a product would have stored."""
    g = torch.Generator().manual_seed(w)
    y = torch.randn(parts, n, w, generator=g).cuda()
    whole = torch.zeros_like(y[0])
    for part in y:                     # in the kernels' order
        whole = whole + part
    whole = whole.to(torch.bfloat16)
    x = torch.randn(n, w, generator=g).cuda()
    a, b = (torch.rand(w, generator=g).cuda() for _ in range(2))
    x0, x1 = x.clone(), x.clone()
    b0, b1 = (torch.empty(n, w, dtype=torch.bfloat16, device="cuda")
              for _ in range(2))
    hops.post_norm(x0, b0, whole, a, 1.0, w, 1e-5)
    hops.post_norm(x1, b1, y, a, 1.0, w, 1e-5)
    assert torch.equal(x0, x1) and torch.equal(b0, b1)
    x0, x1 = x.clone(), x.clone()
    h0 = hops.join_norm(x0, whole, a, b, w // size, w, 1e-5)
    h1 = hops.join_norm(x1, y, a, b, w // size, w, 1e-5)
    assert torch.equal(x0, x1) and torch.equal(h0, h1)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["mlstm", "gla"])
def test_prompt_gates(kind):
    """A prompt's output gate, far from 0 where the exponential's argument is
    large, is as exact as a decode row's. Tokens are chunks of their own with
    values of +-1, so that the normed sums are +-1 and the result is the norm's
    weight times the gate."""
    h, dk, dv, n = 4, 64, 256, 130
    g = torch.Generator().manual_seed(11)
    sign = torch.randint(0, 2, (n, h * dv), generator=g) * 2.0 - 1
    z = (-16 - 64 * torch.rand(n, h * dv, generator=g)).to(torch.bfloat16)
    rows = torch.cat([torch.ones(n, 2 * h * dk), sign, z.float()],
                     1).to("cuda", torch.bfloat16)
    norm = torch.rand(h * dv, generator=g) + 0.5

    def t(*columns):
        return torch.tensor([[i if c is None else c for c in columns]
                             for i in range(n)], dtype=torch.int32).cuda()
    st = hops.StepMeta(chunks=t(None, 1, None, 0), segs=t(None, 1, None, 0),
                       chunk_segs=t(None, 0, None, 1), nd=0, max_len=200,
                       pos=t(0).view(-1), slot=t(None).view(-1),
                       table=torch.zeros(n, 1, dtype=torch.int32).cuda())
    if kind == "mlstm":
        got = hops.mlstm(rows, torch.zeros(n, 2 * h).cuda(),
                         torch.zeros(n, h, dv + 1, dk).cuda(),
                         torch.zeros(n, h).cuda(), norm.cuda(), st, dk, dv,
                         15.0, 1e-30)
    else:
        got = hops.gla(rows, torch.zeros(n, 8).cuda(),
                       torch.zeros(8, h * dk).cuda(),
                       torch.zeros(h * dk).cuda(),
                       torch.zeros(n, h, dv, dk).cuda(), norm.cuda(), st, dk,
                       dv, 16.0, 1e-30)
    zd = z.double()
    want = sign.double() * norm.double() * torch.sigmoid(zd)
    if kind == "gla":
        want = want * zd
    # f32: an exponential within 2^-23, the norm's 16 sums of a lane at 2^-25
    # each (under a root) and ten further roundings of 2^-24: below 1.5e-6. So
    # results that far from the middle of two bf16 are rounded as the exact ones.
    mant = torch.frexp(want.abs())[0] * 256
    clear = ((mant % 1) - 0.5).abs() > 1.5e-6 * mant
    assert bool(clear.float().mean() > 0.99)
    assert torch.equal(got.cpu()[clear], want.to(torch.bfloat16)[clear])


@pytest.mark.parametrize("name", ["tiny-birepel", "tiny-maferax", "tiny-vivepel",
                                  "tiny-zinavik"])
def test_prompts_products_are_whole(name, monkeypatch):
    """All of a model's products know whether a step has prompts: portions, or
    first tokens; decode batches take the choices that were timed for them."""
    from gridllm_amd.models import hybrid
    m = HybridModel(get_spec(name), dtype="fp32", kv_slots=3, max_seq=256)
    seen = []

    def spy(run):
        def call(x, w, *rest):
            seen.append(rest[-1])
            return run(x, w, *rest)
        return call
    for f in ("_linear", "_linear_parts", "_linear_gateup"):
        monkeypatch.setattr(hybrid, f, spy(getattr(hybrid, f)))

    def flags():
        got, seen[:] = set(seen), []
        return got
    a, b = m.cache.alloc(0), m.cache.alloc(0)
    m.forward_prefill(torch.arange(20), a)
    assert flags() == {True}
    m.forward_step([(a, [3], [0]), (b, [5], [0])])      # b's first token
    assert flags() == {True}
    m.forward_step([(a, [3], [0]), (b, [5], [0])])
    assert flags() == {False}
    m.forward_step([(a, [3], [0]), (b, [5, 6], [0])])
    assert flags() == {True}
    m.cache.extend([a], [1])
    m.forward_decode(torch.tensor([1]), torch.tensor([a], dtype=torch.int32))
    assert flags() == {False}


@pytest.mark.gpu
def test_decode_of_many_rows_against_halves():
    """More than 256 decode rows, whose products may have their K in parts, against
    the same rows in two steps; sizes at which the rule cuts K."""
    from dataclasses import replace
    from gridllm_amd.ops import autotune
    spec = get_spec("birepel:3b")
    own = next(ly.ff for ly in spec.layers if not hasattr(ly.ff, "experts"))
    spec = replace(spec, vocab=1024, layers=tuple(
        replace(ly, ff=own) for ly in spec.layers[:2]))
    n = 300
    c = autotune._rule(n, spec.hidden, own.ff)
    assert c[0] == "tile" and c[3] > 1
    out = []
    for sizes in ((n,), (n // 2, n // 2)):
        m = HybridModel(spec, device="cuda:0", dtype="bf16", seed=5, kv_slots=n,
                        max_seq=64)
        slots = [m.cache.alloc(8) for _ in range(n)]
        g = torch.Generator().manual_seed(1)
        m.forward_prefill_batch(list(torch.randint(0, 1024, (n, 7), generator=g)),
                                slots)
        at, parts = 0, []
        for size in sizes:
            some = slots[at:at + size]
            m.cache.prepare_decode(some)
            parts.append(m.forward_decode(
                torch.arange(at, at + size).cuda(),
                torch.tensor(some, dtype=torch.int32).cuda()))
            at += size
        out.append(torch.cat(parts).cpu())
    close(out[0], out[1], ("cuda:0", "bf16"))


@pytest.mark.gpu
@pytest.mark.parametrize("window", [0, 300])
@pytest.mark.parametrize("start,ln", [(3967, 257), (4033, 70), (4100, 130)])
def test_prompt_attention_past_64_pages(start, ln, window):
    """A prompt block has the numbers of 64 pages at a time. Pages in any order give
    to the bit what a cache of contiguous slots gives (a window is compared with f64:
    outputs of up to 3.3, of which bf16 rounds 2^-9, and the weights 2^-9 of each
    value)."""
    from gridllm_amd.ops import hip_ops
    dev, H, G, d, room = torch.device("cuda"), 6, 2, 64, 8192
    g = torch.Generator(device=dev).manual_seed(start)
    n = start + ln
    k, v = (torch.randn(1, G, room, d, generator=g, device=dev).bfloat16()
            for _ in range(2))
    q = torch.randn(ln, H, d, generator=g, device=dev).bfloat16()
    pages = torch.randperm(room // 64, generator=g, device=dev)
    pool_k, pool_v = (torch.zeros(room // 64, G, 64, d, dtype=t.dtype, device=dev)
                      .index_copy_(0, pages, t[0].view(G, -1, 64, d).transpose(0, 1)
                                   .contiguous()) for t in (k, v))

    class Cache:
        table, max_seq = pages.int().view(1, -1).contiguous(), room
    st = meta_for(Cache, 0, start, ln, dev)
    st.tiles = st.tiles.flip(0).contiguous()          # (tiles in any order, too)
    got = hops.paged_attn(q, pool_k, pool_v, st, 0.11, None, None,
                          hops.Keys(window, 64 if window else 0))
    if not window:
        want = hip_ops.attn_prefill_cache(q, k, v, 0, n, start, 0.11)
        assert torch.equal(got.view_as(want), want)
        return
    kd, vd = (t[0, :, :n].double().repeat_interleave(H // G, 0) for t in (k, v))
    sc = torch.einsum("nhd,hkd->hnk", q.double(), kd) * 0.11
    at, key = torch.arange(start, n, device=dev).view(-1, 1), torch.arange(
        n, device=dev)
    sc.masked_fill_((key > at) | ((at - key >= window) & (key >= 64)), -1e30)
    want = (torch.softmax(sc, -1) @ vd).transpose(0, 1)
    assert float((got.view_as(want).double() - want).abs().max()) < 0.02


def test_prompts_on_the_device_are_copies(monkeypatch):
    """A step has its own copy of token ids on the device, of one prompt and of several:
    the caller may change or free theirs on another stream as soon as the call is back."""
    from gridllm_amd.models import hybrid
    m = build(FULL, ("cpu", "fp32"))
    seen = []
    monkeypatch.setattr(hybrid._DeviceIds, "can", staticmethod(
        lambda t, like: torch.is_tensor(t)))
    run = m._run
    monkeypatch.setattr(m, "_run", lambda t, *a: seen.append(t) or run(t, *a))
    a, b = (torch.tensor(tokens(n, seed=n)) for n in (6, 9))
    want = m.forward_prefill(np.array(a), m.cache.alloc(0))
    assert torch.equal(m.forward_prefill(a, m.cache.alloc(0)), want)
    m.forward_prefill_batch([b], [m.cache.alloc(0)])
    m.forward_prefill_batch([a, b], [m.cache.alloc(0) for _ in "ab"])
    theirs = {t.untyped_storage().data_ptr() for t in (a, b)}
    assert len(seen) == 4 and not any(
        t.untyped_storage().data_ptr() in theirs for t in seen)


@pytest.mark.gpu
def test_prompts_on_the_device():
    """Token ids that a step reads from the device behind its preparation give what
    those of the host give: 64-bit, 32-bit and strided, prompts that a step puts in
    another order. Ones that the vocabulary has not are refused as there."""
    lists = [tokens(40), tokens(1, seed=1), tokens(5, seed=2), tokens(130, seed=3)]
    m = build(FULL, ("cuda", "bf16"), slots=32)
    want = m.forward_prefill_batch([np.array(t) for t in lists],
                                   [m.cache.alloc(0) for _ in lists])
    kinds = (lambda t: torch.tensor(t, device="cuda"),
             lambda t: torch.tensor(t, dtype=torch.int32, device="cuda"),
             lambda t: torch.tensor(t, device="cuda").repeat_interleave(2)[::2])
    for dev in kinds:
        got = m.forward_prefill_batch([dev(t) for t in lists],
                                      [m.cache.alloc(0) for _ in lists])
        assert torch.equal(got, want)
    alone = m.forward_prefill(np.array(lists[0]), m.cache.alloc(0))
    for dev in kinds:
        assert torch.equal(m.forward_prefill(dev(lists[0]), m.cache.alloc(0)), alone)
        with pytest.raises(ValueError):
            m.forward_prefill(dev([3, FULL["vocab"]]), m.cache.alloc(0))
        with pytest.raises(ValueError):
            m.forward_prefill_batch([dev([1]), dev([2, -1])],
                                    [m.cache.alloc(0), m.cache.alloc(0)])
