"""Maferax against the plain implementation in maferax_oracle: on the CPU in
f32, on the GPU in f32 and bf16."""

import io
import json
import os
import sys
import time

import numpy as np
import pytest
import torch

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import maferax_oracle as oracle  # noqa: E402
from hybrid_helpers import (EXACT, RUNS, Bytes,  # noqa: E402
                            check_wanted_rows_alone, close, errors,
                            feed, meta_for, one_thread, portions,  # noqa: F401
                            whole)

from gridllm_amd.config import EngineConfig  # noqa: E402
from gridllm_amd.engine import InferenceEngine  # noqa: E402
from gridllm_amd.models.hybrid import HybridModel  # noqa: E402
from gridllm_amd.models.paged import PagedCache  # noqa: E402
from gridllm_amd.models.registry import (read_maferax,  # noqa: E402
                                         resolve_spec)
from gridllm_amd.ops import hybrid as hops  # noqa: E402
from gridllm_amd.ops.reference import Glu  # noqa: E402


def latent(heads=3, dim=32, rot_dim=16, vdim=24, kv_rank=40, q_rank=48,
           scale=0.15, base=5000.0):
    return {"heads": heads, "dim": dim, "rot_dim": rot_dim, "vdim": vdim,
            "kv_rank": kv_rank, "q_rank": q_rank, "scale": scale,
            "rot": {"base": base, "dims": rot_dim}}


def rec(heads=2, dim=32, vdim=32, tau=8.0):
    return {"heads": heads, "dim": dim, "vdim": vdim, "tau": tau}


def dense(ff=96):
    return {"kind": "dense", "ff": ff}


def routed(experts=6, top=2, ff=40, identity=2, groups=(4, 2), scale=1.5):
    r = {"experts": experts, "top": top, "identity": identity, "scale": scale}
    if groups:
        r["groups"] = {"count": groups[0], "keep": groups[1]}
    return {"kind": "moe", "expert": {"ff": ff}, "router": r}


def config(*layers, vocab=130, width=96, eps=1e-5, alpha=1.8,
           logit_scale=1.5):
    return {"architecture": "Maferax", "vocab": vocab, "width": width,
            "norm": {"eps": eps}, "postln_alpha": alpha,
            "logit_scale": logit_scale,
            "layers": [{"type": "latent_attention" if "kv_rank" in m else
                        "gla", "mixer": m, "mlp": f} for m, f in layers]}


# every branch at once, sizes that need padding
FULL = config((rec(2, 40, 24), None), (latent(5, 40, 24, 72, 100, 56), dense()),
              (rec(1, 24, 72, 3.0), routed()),
              (latent(2, 72, 16, 40, 40, 200, 0.1, 300.0),
               routed(5, 3, 24, 0, None, 0.7)),
              (latent(), None), (rec(), routed(7, 3, 56, 2, (3, 2))))


def weights_of(cfg, seed=0):
    return oracle.random_weights(cfg, seed)


def spec_of(cfg, W):
    return read_maferax(cfg, shape=lambda n: tuple(W[n].shape))


def build(cfg, run, seed=0, slots=5, pool=0, W=None, max_seq=512):
    dev, dtype = run
    W = W or weights_of(cfg, seed)
    m = HybridModel(spec_of(cfg, W), device=dev, dtype=dtype, kv_slots=slots,
                    kv_tokens=pool, max_seq=max_seq, random_init=False)
    m._assemble(lambda name: W[name].to(dev))
    if dev != "cpu" and dtype == "bf16":
        m.interleave_gateup()
    return m


def tokens(n, cfg=FULL, seed=0):
    return np.random.default_rng(seed).integers(0, cfg["vocab"], n).tolist()


# ------------------------------------------------------------ each mechanism

ALONE = {
    "latent": config((latent(), None)),
    "latent-one-head": config((latent(1, 64, 64, 64, 64, 64), None)),
    "latent-many-heads": config((latent(17, 16, 8, 16, 32, 64), None)),
    "latent-wide-rank": config((latent(2, 48, 32, 64, 130, 40), None)),
    "latent-widest-rank": config((latent(2, 128, 64, 128, 300, 130), None)),
    "latent-wide-heads": config((latent(2, 160, 16, 72, scale=0.05), None)),
    "latent-wide-values": config((latent(2, 24, 72, 136, 72, 24), None)),
    "latent-fast-rotation": config((latent(base=3.0), None)),
    "gla": config((rec(), None)),
    "gla-one-head": config((rec(1, 64, 64, 16.0), None)),
    "gla-odd-rank": config((rec(2, 40, 24), None)),
    "gla-wide-rank-tau-1": config((rec(1, 24, 72, 1.0), None)),
    "gla-wide-keys": config((rec(1, 130, 40), None)),
    "gla-widest-keys": config((rec(1, 300, 200), None)),
    "dense": config((rec(1, 16, 16), dense(200))),
    "routed": config((rec(1, 16, 16), routed())),
    "routed-no-groups": config((rec(1, 16, 16), routed(7, 3, 64, 1, None))),
    "routed-no-identity": config((rec(1, 16, 16), routed(8, 3, 24, 0, (2, 1)))),
    "routed-one": config((rec(1, 16, 16), routed(9, 1, 24, 3, (3, 1), 1.0))),
    "routed-all": config((rec(1, 16, 16), routed(3, 4, 72, 1, (2, 2)))),
    "routed-many": config((rec(1, 16, 16), routed(70, 6, 16, 20, (9, 4)))),
    "wide-residual": config((rec(), dense()), width=200),
    "coarse-eps": config((latent(), dense()), (rec(), None), eps=0.05),
    "alpha-one": config((latent(), None), (rec(), dense()), alpha=1.0,
                        logit_scale=0.125),
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


DEVICES = [pytest.param("cpu", id="cpu"),
           pytest.param("cuda:0", id="gpu", marks=pytest.mark.gpu)]


@pytest.mark.parametrize("dev", DEVICES)
@pytest.mark.parametrize("experts,identity,groups,keep,top", [
    (14, 2, 4, 2, 3), (12, 0, 1, 1, 4), (5, 3, 8, 5, 4), (60, 8, 2, 1, 8),
    (200, 40, 12, 3, 8), (1, 1, 1, 1, 2)])
def test_routing(experts, identity, groups, keep, top, dev):
    """Choice and weights of tokens of every sort: corrections that overrule
    the scores, that make all choice scores negative, a leading group whose
    others are poor, chosen scores that are tiny."""
    n, w, f, outs = 50, 64, 64, experts + identity
    g = torch.Generator().manual_seed(outs)
    z = torch.randn(n, outs, generator=g) * 2
    z[10:20] *= 10
    corr = torch.randn(outs, generator=g) * 0.5 - 1.5
    x = torch.randn(n, w, generator=g)
    up = torch.randn(experts, 2 * f, w, generator=g) * w ** -0.5
    dn = torch.randn(experts, w, f, generator=g) * f ** -0.5
    ye, wt, same = hops.moe(
        x.to(dev), z.to(dev), up.to(dev), dn.to(dev), hops.Choice(
            top, corr.to(dev), groups, keep, 1e-20, 2.5))
    il = up.view(experts, f // 16, 2, 16, w)
    gate, lin = (il[:, :, i].reshape(experts, f, w).double() for i in (0, 1))
    ye = ye.view(n, top, w).cpu().double()
    xd = x.double()
    for p in range(n):
        chosen, weight = oracle.route(z[p].double(), corr.double(), top,
                                      groups, keep, 2.5)
        ident = sum((float(v) for e, v in zip(chosen, weight) if e >= experts),
                    0.0)
        if identity:
            assert abs(float(same[p]) - ident) < 1e-5
        for k, (e, v) in enumerate(zip(chosen, weight)):
            assert abs(float(wt[p, k]) - (float(v) if e < experts else 0)) < 1e-5
            if e >= experts:
                continue
            y = (oracle.silu(gate[e] @ xd[p]) * (lin[e] @ xd[p])) @ \
                dn[e].double().T
            assert float((ye[p, k] - y).abs().max()) < 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("experts,identity,groups,keep,top", [
    (14, 2, 4, 2, 3), (60, 8, 2, 1, 8), (70, 0, 1, 1, 64), (200, 40, 12, 3, 8),
    (1, 1, 1, 1, 2)])
@pytest.mark.parametrize("n", [1, 15, 16])
def test_routing_by_one_block(n, experts, identity, groups, keep, top,
                              monkeypatch):
    """What the kernels for more rows give, to the bit, in pair order (two tokens
    alike, and one of NaN)."""
    from gridllm_amd.ops import hip_hybrid
    dev, w, f, outs = "cuda:0", 64, 64, experts + identity
    g = torch.Generator().manual_seed(outs + n)
    z = torch.randn(n, outs, generator=g)
    z[n // 2] = z[0]
    if n > 2:
        z[2] = float("nan")
    x = torch.randn(n, w, generator=g).to(dev, torch.bfloat16)
    up, dn = (torch.randn(*s, generator=g).to(dev, torch.bfloat16) * 0.1
              for s in ((experts, 2 * f, w), (experts, w, f)))
    how = hops.Choice(top, torch.randn(outs, generator=g).to(dev), groups, keep,
                      1e-20, 2.5)
    assert hip_hybrid._routes_alone(n, n * top, outs)
    got = hops.moe(x, z.to(dev), up, dn, how)
    monkeypatch.setattr(hip_hybrid, "_routes_alone", lambda *a: False)
    want = hops.moe(x, z.to(dev), up, dn, how)
    real = (want[1] > 0).view(-1)
    assert torch.equal(got[1].nan_to_num(7), want[1].nan_to_num(7))
    assert torch.equal(got[0][real], want[0][real])
    assert identity == 0 or torch.equal(got[2].nan_to_num(7),
                                        want[2].nan_to_num(7))


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [3, 40, 130, 600])
def test_gated_experts_at_every_batch_size(batch):
    e, ident, w, f, top = 6, 2, 128, 192, 3
    g = torch.Generator().manual_seed(3)
    x = torch.randn(batch, w, generator=g).bfloat16()
    z = torch.randn(batch, e + ident, generator=g)
    z[:, 2] += 2.0                         # one far more popular
    up = (torch.randn(e, 2 * f, w, generator=g) * w ** -0.5).bfloat16()
    dn = (torch.randn(e, w, f, generator=g) * f ** -0.5).bfloat16()
    ye, wt, same = hops.moe(x.cuda(), z.cuda(), up.cuda(), dn.cuda(), top)
    idx = torch.topk(z, top).indices
    sm = torch.softmax(torch.topk(z, top).values, -1)
    real = idx < e
    assert torch.allclose(wt.cpu(), sm * real, atol=1e-6)
    assert torch.allclose(same.cpu(), (sm * ~real).sum(-1), atol=1e-6)
    il = up.float().view(e, f // 16, 2, 16, w)
    gate, lin = (il[:, :, i].reshape(e, f, w) for i in (0, 1))
    at = idx.clamp(max=e - 1)
    h = oracle.silu(torch.einsum("nw,nkfw->nkf", x.float(), gate[at])) * \
        torch.einsum("nw,nkfw->nkf", x.float(), lin[at])
    want = torch.einsum("nkf,nkwf->nkw", h.bfloat16().float(), dn[at].float())
    got = ye.view(batch, top, w).cpu()
    assert float(errors(got[real], want[real]).max()) < 0.02


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 64, 100, 300])
def test_gelu_gate_on_every_path(m):
    """The plain op, the interleaved one, the projection with the fused
    epilogue, the exact one."""
    from gridllm_amd.models.registry import DenseFF
    from gridllm_amd.ops import hip_ops
    ff = DenseFF.gelu_tanh(256)
    glu = Glu(ff.alpha, ff.limit, ff.shift, ff.cubic)
    f, k = 256, 192
    g = torch.Generator().manual_seed(m)
    x = (torch.randn(m, k, generator=g) * 2).bfloat16().cuda()
    w = (torch.randn(2 * f, k, generator=g) * k ** -0.5).bfloat16().cuda()
    il = w.view(2, f // 64, 64, k).transpose(0, 1).reshape(2 * f, k).contiguous()
    gu = (x.float() @ w.float().T).cpu().double()
    want = oracle.gelu_tanh(gu[:, :f]) * gu[:, f:]
    outs = [hip_ops.swiglu(torch.nn.functional.linear(x, w), glu=glu),
            hip_ops.swiglu_il(torch.nn.functional.linear(x, il), glu=glu)]
    if m <= 256:
        outs += [hip_ops.gemm_proj(x, il, splitk=s, fuse_swiglu=True, glu=glu)
                 for s in (1, 3)]
    for got in outs:
        assert float(errors(got, want).max()) < 0.02
    exact = hops.glu((x.float() @ w.float().T), glu)
    assert float(errors(exact, want).max()) < 1e-4


@pytest.mark.parametrize("run", RUNS)
def test_sum_norm_and_average(run):
    """Norm behind the sum with experts, identities and a depth average; a row
    of zero weight is never read."""
    dev, dtype = run
    el = torch.float32 if dtype == "fp32" else torch.bfloat16
    n, wp, wd, top, alpha = 9, 192, 150, 6, 1.7
    g = torch.Generator().manual_seed(1)
    x, y = torch.randn(n, wp, generator=g), torch.randn(n * top, wp, generator=g)
    hist = torch.randn(7, n, wp, generator=g)
    for t in (x, y, hist):
        t[..., wd:] = 0
    y = y.to(el)
    pw, ident = torch.rand(n, top, generator=g), torch.rand(n, generator=g)
    pw[:, 4] = 0
    gain = torch.nn.functional.pad(torch.full((wd,), 0.8), (0, wp - wd))
    coef = torch.randn(6, generator=g)
    v = (y.double().view(n, top, wp) * pw.unsqueeze(-1)).sum(1) + \
        (alpha + ident.unsqueeze(-1)) * x.double()
    r = torch.zeros(n, wp, dtype=torch.float64)
    r[:, :wd] = oracle.scalar_norm(v[:, :wd], 0.8, 1e-3)
    want = (coef[:5, None, None] * hist[:5]).sum(0) + coef[5] * r
    y.view(n, top, wp)[:, 4] = float("nan")
    for store in (False, True):
        h = hist.to(dev).clone()
        xo = torch.empty(n, wp, device=dev)
        xb = xo if dtype == "fp32" else torch.empty(n, wp, dtype=el, device=dev)
        hops.sum_norm(x.to(dev), xo, xb, y.to(dev), gain.to(dev), 0.0, alpha,
                      wd, 1e-3, pw.to(dev), ident.to(dev),
                      hops.DepthAverage(h, coef.to(dev), 5, store))
        assert float((xo.cpu() - want).abs().max()) < 1e-5
        assert torch.equal(xb, xo.to(el))
        assert float((h[5].cpu() - (r if store else hist[5])).abs().max()) < 1e-5
        assert torch.equal(h[6].cpu(), hist[6])


@pytest.mark.parametrize("run", RUNS)
def test_rotation_far_out(run):
    """Rotated part of the cached row at far positions, also where only some
    of its pairs are rotated."""
    dev, dtype = run
    n, dims, base = 6000, 12, 50.0
    cfg = config((latent(1, 16, 20, 16, 24, 16, base=base), None))
    cfg["layers"][0]["mixer"]["rot"]["dims"] = dims
    m = build(cfg, run, max_seq=n, W=weights_of(cfg))
    el = torch.float32 if dtype == "fp32" else torch.bfloat16
    pos = torch.tensor([0, 1, 63, 64, 1000, 4095, 4096, 5999])
    rows = torch.randn(len(pos), 256,
                       generator=torch.Generator().manual_seed(2)).to(el)
    w, c = m.layers[0], m.cache
    slot = c.alloc(n)
    c.extend([slot], [n])
    st = hops.StepMeta(nd=len(pos), pos=pos.to(dev, torch.int32),
                       slot=torch.full((len(pos),), slot, dtype=torch.int32,
                                       device=dev), table=c.table, max_len=n)
    hops.latent_rows(rows.to(dev), c.lat[0], st, m.rot[0], w.qnorm, w.kvnorm,
                     16, 24, 1e-5)
    page = c.table[slot].cpu()[pos // 64].long()
    got = c.lat[0].cpu()[page, pos % 64][:, 64:84].double()
    want = oracle.rotate(rows[:, 128:148].double(), pos, base, dims)
    assert float((got - want).abs().max()) < (1e-5 if dtype == "fp32" else 0.02)


# ------------------------------------------- keys and tokens that stand out

CUTS = {"whole": [300], "decode-tail": [190, 1], "pairs": [250, 2],
        "sixteens": [100, 16, 17], "odd": [63, 2, 1, 64, 65]}


@pytest.mark.parametrize("run", RUNS)
@pytest.mark.parametrize("how", sorted(CUTS))
@pytest.mark.parametrize("sizes", [(4, 64, 64, 64), (19, 64, 64, 128)], ids=str)
def test_one_key_stands_out(sizes, how, run):
    """Every query looks for one key, by the rotated or the unrotated part: the
    first, the neighbours of page borders, itself, the previous one; for some
    it is the next one, which it must not see."""
    dev, dtype = run
    el = torch.float32 if dtype == "fp32" else torch.bfloat16
    (H, d, r, k), n, base = sizes, 300, 700.0
    cfg = config((latent(H, d, r, d, k, 64, base=base), None))
    W = weights_of(cfg)
    m = build(cfg, run, W=W, max_seq=320)
    m.cache.alloc(70)                     # page 1 and 2 belong to another
    cache, w, slot = m.cache, m.layers[0], m.cache.alloc(0)
    g = torch.Generator().manual_seed(5)
    lat = torch.randn(n, k, generator=g)
    kr = torch.randn(n, r, generator=g)
    near = [0, 1, 62, 63, 64, 65, 127, 128, 191, 192, 255, 256]
    pos = torch.arange(n)
    cq = torch.zeros(n, 64)
    rows = torch.cat([cq, lat, kr, torch.randn(n, H, generator=g)], 1)
    rows = torch.nn.functional.pad(rows, (0, 128 - H)).to(el)
    c = oracle.rms(rows[:, 64:64 + k].double(), 1e-5) * \
        W["l0.mix.dkv.norm"].double()
    uk = W["l0.mix.uk"].double().view(H, d, k)
    uv = W["l0.mix.uv"].double().view(H, d, k)
    krot = oracle.rotate(rows[:, 64 + k:64 + k + r].double(), pos, base, r)
    qn, qr = torch.zeros(n, H, d), torch.zeros(n, H, r)
    for h in range(H):
        aim = []
        for p in range(n):
            targets = [t for t in near if t <= p] + [p, max(p - 1, 0),
                                                     min(p + 1, n - 1)]
            aim.append(targets[(p * 7 + h * 5) % len(targets)])
        if h % 2:
            qn[:, h] = c[aim] @ uk[h].T * 1.5
        else:                  # rotated back from the query's own position
            qr[:, h] = oracle.rotate(krot[aim], -pos, base, r) * 1.5
    q = torch.cat([qn, qr], 2).view(n, -1).to(el)
    qd = q.double().view(n, H, d + r)
    scale = 0.25
    gate = rows[:, 64 + k + r:64 + k + r + H]
    want = oracle.latent_attend(
        qd[..., :d], oracle.rotate(qd[..., d:], pos, base, r), c, krot, uk, uv,
        scale) * torch.sigmoid(gate.double())[:, :, None]
    got = []
    for at, ln in portions(n, CUTS[how]):
        cache.extend([slot], [ln])
        st = meta_for(cache, slot, at, ln, dev)
        part = rows[at:at + ln].to(dev).contiguous()
        hops.latent_rows(part, cache.lat[0], st, m.rot[0], w.qnorm, w.kvnorm,
                         64, k, 1e-5)
        got.append(hops.latent_attn(
            q[at:at + ln].to(dev).contiguous(), cache.lat[0], st, m.rot[0],
            w.wuk, w.wuv, w.wukv, scale, part[:, 64 + k + r:]))
    got = torch.cat(got).cpu().double().view(n, H, d)
    err = (got - want).abs().amax(-1)
    assert float(err.max()) < (1e-4 if dtype == "fp32" else 0.08)


@pytest.mark.parametrize("run", RUNS)
@pytest.mark.parametrize("how", sorted(CUTS))
@pytest.mark.parametrize("dk,dv", [(64, 64), (128, 192)])
def test_one_token_is_remembered(how, run, dk, dv):
    """A loud token, at the first place and around chunk borders, is what later
    queries recall. Channels that keep everything stand beside channels that
    forget within a few tokens or at once; one head loses everything in the
    middle of a chunk, and one all the time."""
    dev, dtype = run
    H, n, rank = 3, 300, 3
    cfg = config((rec(H, dk, dv), None))
    cache = PagedCache(read_maferax(cfg), 3, 320, torch.device(dev),
                       torch.float32)
    slot = cache.alloc(0)
    S = cache.S[0]
    S[slot] = 7.0                         # a predecessor's state
    g = torch.Generator().manual_seed(7)
    el = torch.float32 if dtype == "fp32" else torch.bfloat16
    q, k = torch.randn(2, n, H, dk, generator=g)
    v, gate = torch.randn(2, n, H, dv, generator=g)
    k *= 0.02
    loud = [0, 15, 16, 63, 64, 65, 128, 191, 192, 250]
    for t in loud:
        k[t] *= 50
    for p in range(n):
        q[p] = k[max([t for t in loud if t <= p])] * 2
    # log decays by channel: u selects, wa2 holds, the bias is zero
    u = torch.zeros(n, rank)
    u[:, 0] = 1
    u[100, 1] = 1
    u[:, 2] = torch.rand(n, generator=g)
    wa2 = torch.zeros(rank, H, dk)
    wa2[0] = torch.linspace(-5, 16, dk)   # from 5 nats a token to none
    wa2[0, 2] = -40.0                     # 40 nats a token
    wa2[0, 2, ::5] = 12.0
    wa2[1, 1] = -60.0
    wa2[2] = torch.randn(H, dk, generator=g)
    tau = 1.0
    row = torch.cat([t.reshape(n, -1) for t in (q, k, v, gate)], 1).to(el)
    qd, kd, vd, gd = row.double().split([H * dk, H * dk, H * dv, H * dv], dim=1)
    z = (u @ wa2.view(rank, -1)).double()
    o = oracle.gla_run(qd.view(n, H, dk) * dk ** -0.5, kd.view(n, H, dk),
                       vd.view(n, H, dv),
                       oracle.gla_log_decay(z, tau).view(n, H, dk))
    norm = torch.randn(dv, generator=g)
    want = (oracle.rms(o, 1e-5) * norm.double()).reshape(n, -1) * \
        oracle.silu(gd)
    got = []
    for at, ln in portions(n, CUTS[how]):
        cache.extend([slot], [ln])
        got.append(hops.gla(row[at:at + ln].to(dev).contiguous(),
                            u[at:at + ln].to(dev).contiguous(),
                            wa2.view(rank, -1).to(dev).contiguous(),
                            torch.zeros(H * dk, device=dev), S,
                            norm.repeat(H).to(dev),
                            meta_for(cache, slot, at, ln, dev), dk, dv, tau,
                            1e-5))
    got = torch.cat(got).cpu().double()
    e = errors(got.view(n, H, dv).transpose(1, 2).reshape(n, -1),
               want.view(n, H, dv).transpose(1, 2).reshape(n, -1))
    assert float(e.max()) < (3e-4 if dtype == "fp32" else 0.01)
    last = S[slot].cpu().double().transpose(1, 2)         # [H, dk, dv]
    state = torch.zeros(H, dk, dv, dtype=torch.float64)
    for p in range(n):
        a = oracle.gla_log_decay(z[p], tau).view(H, dk, 1)
        state = torch.exp(a) * state + kd.view(n, H, dk, 1)[p] * \
            vd.view(n, H, 1, dv)[p]
    assert float((last - state).abs().max()) < \
        1e-4 * float(state.abs().max())


# ----------------------------------------------- cuts, batches, pages, slots

@pytest.mark.parametrize("run", RUNS)
@pytest.mark.parametrize("sizes", [[1], [2], [3], [63, 2], [64], [100, 1],
                                   [16, 17], [130, 1, 7]], ids=str)
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
        for key, out in (("a", ga), ("b", gb)):
            out = torch.cat(out).cpu()
            close(out, first.setdefault(key, out), run, exact=1e-4,
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


# ------------------------------------------------- configuration and weights

def test_config_reader():
    W = weights_of(FULL)
    spec = spec_of(FULL, W)
    assert spec.params == sum(v.numel() for v in W.values())
    assert [ly.mixer.rank for ly in spec.layers
            if hasattr(ly.mixer, "rank")] == [5, 33, 8]
    assert spec.layers[3].ff.groups == 1 and spec.layers[0].ff is None
    m = HybridModel(spec, dtype="fp32", random_init=False)
    assert m.tensor_shapes() == {k: tuple(v.shape) for k, v in W.items()}

    def broken(change):
        c = json.loads(json.dumps(FULL))
        change(c)
        with pytest.raises((ValueError, KeyError)):
            read_maferax(c)

    broken(lambda c: c.pop("postln_alpha"))
    broken(lambda c: c.update(window=3))
    broken(lambda c: c["layers"][1]["mixer"].pop("scale"))
    broken(lambda c: c["layers"][0]["mixer"].update(conv=4))
    broken(lambda c: c["layers"][0].update(type="conv"))
    broken(lambda c: c["layers"][1]["mixer"]["rot"].update(dims=25))
    broken(lambda c: c["layers"][1]["mixer"]["rot"].update(dims=26))
    broken(lambda c: c["layers"][1]["mlp"].update(kind="other"))
    broken(lambda c: c["layers"][2]["mlp"]["router"].update(top=5))
    broken(lambda c: c["layers"][2]["mlp"]["router"].update(identity=1))
    broken(lambda c: c["layers"][2]["mlp"]["router"]["groups"].update(keep=5))
    big = json.loads(json.dumps(FULL))
    big["layers"][1]["mixer"]["kv_rank"] = 513
    with pytest.raises(ValueError, match="latents of 513"):
        HybridModel(read_maferax(big), random_init=False)


def test_length_is_bound_by_the_pool_alone():
    spec = read_maferax(FULL)
    assert HybridModel(spec, dtype="fp32", random_init=False,
                       kv_tokens=9001).max_seq == 9024
    assert HybridModel(spec, dtype="fp32", random_init=False,
                       kv_tokens=9001, max_seq=100).max_seq == 100
    assert HybridModel(spec, dtype="fp32", random_init=False,
                       kv_slots=1).max_seq == 8192


@pytest.fixture
def checkpoint(tmp_path):
    from safetensors.torch import save_file
    save_file(weights_of(FULL, 3), str(tmp_path / "model.safetensors"))
    (tmp_path / "config.json").write_text(json.dumps(FULL))
    return tmp_path


def test_checkpoint_describes_itself(checkpoint):
    spec = resolve_spec("llama3.2:1b", str(checkpoint))
    assert (spec.family, spec.name) == ("maferax", "maferax:custom")
    assert spec.layers[2].mixer.rank == 33
    m = HybridModel(spec, dtype="fp32", random_init=False)
    assert m.load_safetensors(str(checkpoint)) == len(weights_of(FULL))
    from safetensors.torch import save_file
    W = weights_of(FULL, 3)
    del W["l2.dwa"]
    save_file(W, str(checkpoint / "model.safetensors"))
    with pytest.raises(KeyError, match="l2.dwa"):
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


GREEDY = {"temperature": 0.0, "num_predict": 6}
PROMPTS = ["2 + 3 = ", "q", "A prompt that is long enough to take more than "
           "one page of the cache and several portions ...", "?"]


@pytest.mark.parametrize("run", EXACT)
@pytest.mark.parametrize("chunk", [8192, 5])
def test_greedy_generation(checkpoint, run, chunk):
    """Through generate, generate_batch and the continuous batcher, with whole
    prompts and with portions of five tokens beside decoding rows."""
    from gridllm_amd.engine.batcher import Batcher
    eng = engine_for(checkpoint, run, prefill_chunk=chunk)
    eng.tokenizer = Bytes(FULL["vocab"])
    want, gaps = zip(*(greedy(eng.tokenizer.encode(p), 6) for p in PROMPTS))
    assert min(min(g) for g in gaps) > 1e-3        # no close call in the test
    free = eng.model.cache.n_free
    assert [eng.generate(p, GREEDY).token_ids for p in PROMPTS] == list(want)
    out = eng.generate_batch([(p, GREEDY) for p in PROMPTS])
    assert [r.token_ids for r in out] == list(want)
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


@pytest.mark.parametrize("run", RUNS)
@pytest.mark.parametrize("name", ["tiny-maferax", "tiny-maferax:latest"])
def test_registered_model_serves(name, run):
    eng = InferenceEngine(EngineConfig(model=name, device=run[0], dtype=run[1],
                                       max_batch_size=2, max_seq_len=128))
    r = eng.generate("hello", {"temperature": 0.7, "seed": 5,
                               "num_predict": 6})
    assert r.eval_count == 6
    assert "tiny-maferax" in eng.model_names()
    info = eng.spec.model_info()
    assert info["general.architecture"] == "maferax"
    assert info["maferax.attention.kv_lora_rank"] == 48


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
def test_long_decode_by_captured_graphs(checkpoint, dtype):
    """Decode-only steps replay captured graphs, between eager mixed steps and
    synchronizations; every step against the eager model, 150 tokens long and
    over page borders."""
    run = ("cuda:0", dtype)
    eng = engine_for(checkpoint, run)
    assert eng._graph_ok() and eng._graphs
    W = weights_of(FULL, 3)
    ref = build(FULL, run, W=W)
    ids = {i: tokens(190, seed=20 + i) for i in range(3)}
    a = {i: eng.open_sequence() for i in ids}
    b = {i: ref.cache.alloc(0) for i in ids}
    at = {0: 40, 1: 2, 2: 33}
    got, want = [], []
    eng.run_step([(a[i], ids[i][:n], []) for i, n in at.items()])
    ref.forward_step([(b[i], ids[i][:n], []) for i, n in at.items()])
    for step in range(150):
        live = [i for i in ids if not (i == 1 and step % 3 == 0)]
        n = {i: 2 if step % 31 == 30 and i == 2 else 1 for i in live}
        ent = [(i, ids[i][at[i]:at[i] + n[i]], [0]) for i in live
               if at[i] + n[i] <= 190]
        got.append(eng.run_step([(a[i], t, w) for i, t, w in ent]).clone())
        want.append(ref.forward_step([(b[i], t, w) for i, t, w in ent]))
        for i, t, _ in ent:
            at[i] += len(t)
        if step % 10 == 0:
            torch.cuda.synchronize()
    # (a row whose routing was a close call stays off for some tokens)
    close(torch.cat(got), torch.cat(want).cpu(), run, exact=1e-4, coarse=0.1,
          odd=0.1)
    close(eng.run_step([(a[0], [7], [0])]),
          oracle.forward(FULL, W, ids[0][:at[0]] + [7])[0][-1:], run, odd=1.0)


@pytest.mark.parametrize("run", EXACT)
def test_long_decode(run):
    """Token by token from the first one on, over several pages."""
    cfg = config((latent(2, 32, 16, 32, 40, 32), dense(64)), (rec(), routed()))
    m = build(cfg, run)
    ids = tokens(270, cfg, seed=4)
    slot = m.cache.alloc(0)
    close(feed(m, slot, ids, [1]), oracle.forward(cfg, weights_of(cfg), ids)[0],
          run)


@pytest.mark.parametrize("run", RUNS)
@pytest.mark.parametrize("heads,rank", [(20, 300), (33, 130), (3, 300)])
def test_decode_of_many_heads_and_wide_latents(heads, rank, run):
    cfg = config((latent(heads, 16, 8, 16, rank, 32, scale=0.4), None))
    m = build(cfg, run)
    ids = tokens(170, cfg, seed=6)
    slot = m.cache.alloc(0)
    close(feed(m, slot, ids, [100, 1]),
          oracle.forward(cfg, weights_of(cfg), ids)[0], run)


@pytest.mark.parametrize("run", RUNS)
@pytest.mark.parametrize("heads", [4, 20])
def test_many_rows_decode_at_once(heads, run):
    """Enough rows that no row's keys are split."""
    n = 290 if run[0] != "cpu" else 12
    cfg = config((latent(heads, 16, 8, 16, 40, 32), None), (rec(), routed()))
    m = build(cfg, run, slots=n, max_seq=128)
    seqs = [tokens(k, cfg, seed=k) for k in (71, 3, 40)]
    slots = [m.cache.alloc(0) for _ in range(n)]
    m.forward_step([(s, seqs[i % 3][:-1], []) for i, s in enumerate(slots)])
    got = m.forward_step([(s, seqs[i % 3][-1:], [0])
                          for i, s in enumerate(slots)])
    want = [oracle.forward(cfg, weights_of(cfg), q)[0][-1] for q in seqs]
    close(got, torch.stack([want[i % 3] for i in range(n)]), run, odd=0.1)


@pytest.mark.parametrize("run", RUNS)
def test_trace_replay(checkpoint, tmp_path, run):
    from gridllm_amd import trace
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
    out = tmp_path / "out"
    out.mkdir()
    eng = trace.make_engine(str(checkpoint),
                            {"fp32": "float32", "bf16": "bfloat16"}[run[1]],
                            256, run[0])
    acks = io.StringIO()
    trace.replay(eng, io.StringIO("".join(json.dumps(s) + "\n"
                                          for s in steps)), str(out), acks)
    assert acks.getvalue() == "".join(f"done {i}\n" for i in range(4))
    assert len(eng.model.cache._free_pages) == eng.model.cache.pages == 4
    assert sorted(os.listdir(out)) == [f"{k}.f32" for k in sorted(want)]
    for k, w in want.items():
        got = np.fromfile(os.path.join(out, f"{k}.f32"), dtype="<f4")
        close(torch.from_numpy(got).view(w.shape), w, run, coarse=0.1, odd=0.5)


@pytest.mark.gpu
@pytest.mark.parametrize("dk,dv", [(64, 64), (128, 256), (64, 192), (192, 128),
                                   (64, 320)])
def test_gla_chunk_sizes(dk, dv):
    """Decode rows and portions of whole and cut chunks in one step, for heads
    whose columns a block has all of (up to 256) or not."""
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
    u = torch.randn(n, 8, generator=g)
    wa, ba = torch.randn(8, h * dk, generator=g), torch.randn(h * dk,
                                                              generator=g)
    S = torch.randn(5, h, dv, dk, generator=g)
    norm = torch.rand(h * dv, generator=g) + 0.5
    S0 = S.clone()
    want = reference_hybrid.gla(rows.float(), u, wa, ba, S0, norm,
                                hops.StepMeta(segs=t(entries), **meta), dk, dv,
                                16.0, 1e-5)
    dev = "cuda"
    S1 = S.to(dev)
    st = hops.StepMeta(chunks=t(chunks).to(dev), chunk_segs=t(segs).to(dev),
                       segs=t(entries).to(dev),
                       **{k: v.to(dev) if torch.is_tensor(v) else v
                          for k, v in meta.items()})
    got = hops.gla(rows.to(dev), u.to(dev), wa.to(dev), ba.to(dev), S1,
                   norm.to(dev), st, dk, dv, 16.0, 1e-5).cpu().float()
    # bf16 result; sums of products of (hi, lo) pairs, 2^-16 each, that a unit
    # RMS row of cancelling terms makes up to 16 times as large
    gate = torch.nn.functional.silu(rows[:, -h * dv:].float()).abs() * norm
    assert bool(((got - want).abs() <= 2 ** -8 * want.abs() +
                 2 ** -11 * gate + 1e-6).all())
    used = [e[2] for e in entries]
    assert float((S1.cpu()[used] - S0[used]).abs().max()) < \
        2 ** -11 * float(S0.abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("dk,dv", [(128, 256), (64, 128), (64, 512)])
@pytest.mark.parametrize("tau", [16.0, 0.3])       # (.3: scores pair by pair)
def test_gla_chunk_halves(dk, dv, tau):
    """Chunks that end within either half of their tokens, more of them than 8.
    (With tau .05 a token sees itself alone; where its q . k of 128 terms, 81 in
    absolute sum, cancels to .2, 2^-16 of 81 / .2 is 2^-7.5 of its result, which is more
    than the room here: one of 513 rows is off by 1.6 of it, as it was by 64 tokens.)"""
    from gridllm_amd.ops import reference_hybrid
    h, lens = 3, (1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 97)
    g = torch.Generator().manual_seed(dk + dv)
    n = sum(lens)
    entries, chunks, segs, at = [], [], [], 0
    for i, ln in enumerate(lens):
        entries.append((at, ln, i, i % 2))
        segs.append((i, i % 2, len(chunks), -(-ln // 64)))
        chunks += [(at + c, min(64, ln - c), i, 0) for c in range(0, ln, 64)]
        at += ln
    pos = torch.cat([torch.arange(e[3], e[3] + e[1]) for e in entries])
    slot = torch.cat([torch.full((e[1],), e[2]) for e in entries])

    def t(rows):
        return torch.tensor(rows, dtype=torch.int32, device="cuda")
    meta = dict(nd=0, pos=pos.int(), slot=slot.int(), max_len=200,
                table=torch.zeros(len(lens), 1, dtype=torch.int32))
    rows = torch.randn(n, h * 2 * (dk + dv), generator=g).to(torch.bfloat16)
    u = torch.randn(n, 8, generator=g)
    wa, ba = torch.randn(8, h * dk, generator=g), torch.randn(h * dk,
                                                              generator=g)
    S = torch.randn(len(lens), h, dv, dk, generator=g)
    norm = torch.rand(h * dv, generator=g) + 0.5
    want = reference_hybrid.gla(rows.float(), u, wa, ba, S.clone(), norm,
                                hops.StepMeta(segs=t(entries).cpu(), **meta), dk,
                                dv, tau, 1e-5)
    st = hops.StepMeta(chunks=t(chunks), chunk_segs=t(segs), segs=t(entries),
                       **{k: v.to("cuda") if torch.is_tensor(v) else v
                          for k, v in meta.items()})
    got = hops.gla(rows.cuda(), u.cuda(), wa.cuda(), ba.cuda(), S.cuda(),
                   norm.cuda(), st, dk, dv, tau, 1e-5).cpu().float()
    # as in test_gla_chunk_sizes
    gate = torch.nn.functional.silu(rows[:, -h * dv:].float()).abs() * norm
    assert bool(((got - want).abs() <= 2 ** -8 * want.abs() +
                 2 ** -11 * gate + 1e-6).all())
