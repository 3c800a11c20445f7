"""HIP kernel numerics vs the plain-PyTorch fp32 reference (gpu-only).

Every kernel is compared against gridllm_amd.ops.reference computed in fp32
on the same data; tolerances sized for bf16 I/O (~3 decimal digits).
"""

import math
import os

import pytest
import torch

pytestmark = pytest.mark.gpu

from gridllm_amd.ops import reference as R  # noqa: E402


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available()
    from gridllm_amd.ops import hip_ops
    assert hip_ops.available(), "HIP extension must be built on GPU boxes"
    return torch.device("cuda:0")


def _mx(a, b):
    return (a.float() - b.float()).abs().max().item()


@pytest.mark.parametrize("n,h", [(4, 256), (33, 3072), (128, 8192), (1, 2048)])
def test_rmsnorm_gpu(dev, n, h):
    torch.manual_seed(0)
    from gridllm_amd.ops import hip_ops
    x = torch.randn(n, h, device=dev).to(torch.bfloat16)
    w = torch.randn(h, device=dev).to(torch.bfloat16)
    y = hip_ops.rmsnorm(x, w, 1e-5)
    ref, _ = R.rmsnorm(x.cpu().float(), w.cpu().float(), 1e-5)
    assert _mx(y.cpu(), ref) < 0.05


def test_rmsnorm_residual_gpu(dev):
    torch.manual_seed(1)
    from gridllm_amd.ops import hip_ops
    n, h = 17, 3072
    x = torch.randn(n, h, device=dev).to(torch.bfloat16)
    r = torch.randn(n, h, device=dev).to(torch.bfloat16)
    w = torch.randn(h, device=dev).to(torch.bfloat16)
    res_out = torch.empty_like(x)
    y = hip_ops.rmsnorm(x, w, 1e-5, residual=r, residual_out=res_out)
    ref_y, ref_res = R.rmsnorm(x.cpu().float(), w.cpu().float(), 1e-5,
                               residual=r.cpu().float())
    assert _mx(res_out.cpu(), ref_res) < 0.02
    assert _mx(y.cpu(), ref_y) < 0.05


@pytest.mark.parametrize("t,hq,hk,d", [(7, 24, 8, 128), (64, 32, 8, 64)])
def test_rope_gpu(dev, t, hq, hk, d):
    torch.manual_seed(2)
    from gridllm_amd.ops import hip_ops
    q = torch.randn(t, hq, d, device=dev).to(torch.bfloat16)
    k = torch.randn(t, hk, d, device=dev).to(torch.bfloat16)
    cos, sin = R.rope_tables(d, 256, device=dev)
    pos = torch.randint(0, 256, (t,), dtype=torch.int32, device=dev)
    q_ref, k_ref = R.rope(q.cpu().float(), k.cpu().float(),
                          cos.cpu(), sin.cpu(), pos.cpu())
    hip_ops.rope(q, k, cos, sin, pos)
    assert _mx(q.cpu(), q_ref) < 0.05
    assert _mx(k.cpu(), k_ref) < 0.05


def test_swiglu_gpu(dev):
    torch.manual_seed(3)
    from gridllm_amd.ops import hip_ops
    n, f = 65, 8192
    gu = torch.randn(n, 2 * f, device=dev).to(torch.bfloat16)
    out = hip_ops.swiglu(gu)
    ref = R.swiglu(gu.cpu().float())
    assert _mx(out.cpu(), ref) < 0.1


def test_kv_append_gpu(dev):
    torch.manual_seed(4)
    from gridllm_amd.ops import hip_ops
    b, hk, smax, d, n = 3, 8, 64, 128, 5
    kc = torch.zeros(b, hk, smax, d, device=dev, dtype=torch.bfloat16)
    vc = torch.zeros_like(kc)
    kn = torch.randn(n, hk, d, device=dev).to(torch.bfloat16)
    vn = torch.randn(n, hk, d, device=dev).to(torch.bfloat16)
    slot = torch.tensor([0 * smax + 3, 1 * smax + 0, 2 * smax + 63,
                         0 * smax + 4, 1 * smax + 1],
                        dtype=torch.int32, device=dev)
    hip_ops.kv_append(kc, vc, kn, vn, slot)
    kc_ref = torch.zeros(b, hk, smax, d)
    vc_ref = torch.zeros_like(kc_ref)
    R.kv_append(kc_ref, vc_ref, kn.cpu().float(), vn.cpu().float(), slot.cpu())
    assert _mx(kc.cpu(), kc_ref) < 1e-6  # pure copy, bitwise via bf16
    assert _mx(vc.cpu(), vc_ref) < 1e-6


@pytest.mark.parametrize("b,hq,hk,d,seqs", [
    (2, 24, 8, 128, [1, 5]),
    (4, 32, 8, 64, [64, 100, 128, 7]),
    (1, 64, 8, 128, [1000]),          # forces split-S
    (2, 8, 8, 128, [300, 17]),        # G=1
    (256, 24, 8, 128, None),          # large batch -> one-wave kernel
    (300, 32, 8, 64, None),           # one-wave, D=64, G=4
])
def test_attn_decode_gpu(dev, b, hq, hk, d, seqs):
    torch.manual_seed(5)
    from gridllm_amd.ops import hip_ops
    if seqs is None:
        seqs = [int(x) for x in
                torch.randint(1, 200, (b,), generator=torch.Generator()
                              .manual_seed(b)).tolist()]
    smax = max(seqs)
    kc = torch.randn(b, hk, smax, d, device=dev).to(torch.bfloat16)
    vc = torch.randn(b, hk, smax, d, device=dev).to(torch.bfloat16)
    q = torch.randn(b, hq, d, device=dev).to(torch.bfloat16)
    seqlen = torch.tensor(seqs, dtype=torch.int32, device=dev)
    scale = 1.0 / math.sqrt(d)
    out = hip_ops.attn_decode(q, kc, vc, seqlen, scale)
    ref = R.attn_decode(q.cpu().float(), kc.cpu().float(), vc.cpu().float(),
                        seqlen.cpu(), scale)
    assert _mx(out.cpu(), ref) < 0.03


def test_attn_decode_split_consistency(dev):
    """nsplit=1 and nsplit=8 must agree (same math, different partitioning)."""
    torch.manual_seed(6)
    from gridllm_amd.ops import hip_ops
    b, hq, hk, d, smax = 2, 24, 8, 128, 2048
    kc = torch.randn(b, hk, smax, d, device=dev).to(torch.bfloat16)
    vc = torch.randn(b, hk, smax, d, device=dev).to(torch.bfloat16)
    q = torch.randn(b, hq, d, device=dev).to(torch.bfloat16)
    seqlen = torch.tensor([2048, 777], dtype=torch.int32, device=dev)
    o1 = hip_ops.attn_decode(q, kc, vc, seqlen, 0.0883, nsplit=1)
    o8 = hip_ops.attn_decode(q, kc, vc, seqlen, 0.0883, nsplit=8)
    assert _mx(o1.cpu(), o8.cpu()) < 0.01


def test_attn_decode_slot_map_gpu(dev):
    torch.manual_seed(7)
    from gridllm_amd.ops import hip_ops
    slots, hq, hk, d, smax = 4, 24, 8, 128, 128
    kc = torch.randn(slots, hk, smax, d, device=dev).to(torch.bfloat16)
    vc = torch.randn(slots, hk, smax, d, device=dev).to(torch.bfloat16)
    q = torch.randn(2, hq, d, device=dev).to(torch.bfloat16)
    seqlen = torch.tensor([50, 80], dtype=torch.int32, device=dev)
    slot_map = torch.tensor([3, 1], dtype=torch.int32, device=dev)
    out = hip_ops.attn_decode(q, kc, vc, seqlen, 0.0883, slot_map=slot_map)
    ref = R.attn_decode(q.cpu().float(), kc.cpu().float(), vc.cpu().float(),
                        seqlen.cpu(), 0.0883, slot_map=slot_map.cpu())
    assert _mx(out.cpu(), ref) < 0.03


@pytest.mark.parametrize("b", [1, 63, 1024, 1500])
def test_decode_positions_gpu(dev, b):
    """Rows of one and several turns of the block, several rows on one slot."""
    from gridllm_amd.ops import hip_ops
    g = torch.Generator().manual_seed(b)
    lens = torch.randint(0, 1000, (b + 1,), generator=g, dtype=torch.int32)
    off = torch.randint(0, 1000, (b + 1,), generator=g, dtype=torch.int32)
    slots = torch.randperm(b + 1, generator=g)[:b].int()
    slots[b // 2:] = b
    want = lens.clone()
    ref = R.decode_positions(want, slots, off, 2048)
    got = lens.to(dev)
    out = hip_ops.decode_positions(got, slots.to(dev), off.to(dev), 2048)
    for x, y in zip(out, ref):
        assert torch.equal(x.cpu(), y)
    assert torch.equal(got.cpu(), want)
    assert torch.equal(hip_ops.decode_lengths(got, slots.to(dev)).cpu(),
                       want[slots.long()])


@pytest.mark.parametrize("b", [1, 256, 257, 1500])
def test_advance_lengths_gpu(dev, b):
    """Rows of one and several blocks, several rows on one slot."""
    from gridllm_amd.ops import hip_ops
    g = torch.Generator().manual_seed(b)
    want = torch.randint(0, 1000, (b + 1,), generator=g, dtype=torch.int32)
    slots = torch.randperm(b + 1, generator=g)[:b].int()
    slots[b // 2:] = b
    got = want.to(dev)
    R.advance_lengths(want, slots)
    hip_ops.advance_lengths(got, slots.to(dev))
    assert torch.equal(got.cpu(), want)


@pytest.mark.parametrize("t", [1, 256, 257])
@pytest.mark.parametrize("start", [0, 5])
def test_prompt_positions_gpu(dev, t, start):
    from gridllm_amd.ops import hip_ops
    a, b = (torch.full((4,), 7, dtype=torch.int32) for _ in range(2))
    x, y = a.to(dev), b.to(dev)
    for i, j in zip(hip_ops.prompt_positions(t, 2, start, x, 1024),
                    R.prompt_positions(t, 2, start, a, 1024)):
        assert torch.equal(i.cpu(), j)
    hip_ops.prompt_end(t, 2, start, x, y)
    R.prompt_end(t, 2, start, a, b)
    assert torch.equal(x.cpu(), a) and torch.equal(y.cpu(), b)
    for slot in (4, -1):
        with pytest.raises(IndexError):
            hip_ops.prompt_positions(t, slot, start, x, 1024)
        with pytest.raises(IndexError):
            hip_ops.prompt_end(t, slot, start, x, y)


@pytest.mark.parametrize("n,h", [(1, 8), (5, 896), (3, 2056), (2, 8192),
                                 (2, 8200)])
def test_embed_norm_gpu(dev, n, h):
    """Rows in registers and beyond: the bits of a lookup and of rmsnorm."""
    from gridllm_amd.ops import hip_ops
    emb = torch.randn(50, h, device=dev).to(torch.bfloat16)
    w = torch.randn(h, device=dev).to(torch.bfloat16)
    tok = torch.tensor([49, 0, -1, 7, 7][:n], device=dev)
    x, y = hip_ops.embed_norm(tok, emb, w, 1e-5)
    assert torch.equal(x, emb[tok])
    assert torch.equal(y, hip_ops.rmsnorm(emb[tok], w, 1e-5))
    ref, _ = R.rmsnorm(emb[tok].cpu().float(), w.cpu().float(), 1e-5)
    # one rounding to bf16 of values up to 16
    assert _mx(y.cpu(), ref) < 0.04


def test_embed_norm_other_indices_gpu(dev):
    """Host indices and other layouts, as torch's lookup takes them."""
    from gridllm_amd import ops
    from gridllm_amd.ops import hip_ops
    emb = torch.randn(50, 96, device=dev).to(torch.bfloat16)
    w = torch.randn(96, device=dev).to(torch.bfloat16)
    tok = torch.tensor([49, 0, -1, 7, 7])
    for t, e in ((tok, emb), (tok.to(dev).int(), emb),
                 (tok.to(dev), emb.t().contiguous().t())):
        x, y = ops.embed_norm(t, e, w, 1e-5)
        assert torch.equal(x, emb[tok])
        assert torch.equal(y, hip_ops.rmsnorm(emb[tok], w, 1e-5))


@pytest.mark.parametrize("n,hq,hk,d", [(5, 24, 8, 128), (16, 32, 8, 64),
                                       (7, 4, 2, 20), (1, 3, 1, 16)])
def test_rope_kv_fused_gpu(dev, n, hq, hk, d):
    """Fused rope+kv-write vs the composed reference (strided qkv input)."""
    torch.manual_seed(8)
    from gridllm_amd.ops import hip_ops
    smax, slots = 64, 3
    qkv = torch.randn(n, (hq + 2 * hk) * d, device=dev).to(torch.bfloat16)
    kc = torch.zeros(slots, hk, smax, d, device=dev, dtype=torch.bfloat16)
    vc = torch.zeros_like(kc)
    cos, sin = R.rope_tables(d, 128, device=dev)
    pos = torch.randint(0, 120, (n,), dtype=torch.int32, device=dev)
    slot = (torch.randint(0, slots, (n,), dtype=torch.int32, device=dev) * smax
            + torch.arange(n, dtype=torch.int32, device=dev))  # unique cells
    q = hip_ops.rope_kv(qkv, kc, vc, cos, sin, pos, slot, hq, hk, d)
    kc_ref = torch.zeros(slots, hk, smax, d)
    vc_ref = torch.zeros_like(kc_ref)
    q_ref = R.rope_kv(qkv.cpu().float(), kc_ref, vc_ref, cos.cpu(), sin.cpu(),
                      pos.cpu(), slot.cpu(), hq, hk, d)
    assert _mx(q.cpu(), q_ref) < 0.05
    assert _mx(kc.cpu(), kc_ref) < 0.05
    assert _mx(vc.cpu(), vc_ref) < 1e-6


@pytest.mark.parametrize("b,h", [(1, 8), (3, 896), (70, 3072)])
def test_prompts_end_gpu(dev, b, h):
    """Lengths, offsets and last rows, one of them counted from the end; lengths
    alone."""
    from gridllm_amd.ops import hip_ops
    g = torch.Generator().manual_seed(b)
    lens, off = (torch.randint(1, 99, (b + 2,), generator=g, dtype=torch.int32)
                 for _ in range(2))
    slots = torch.randperm(b + 2, generator=g)[:b].int()
    new = torch.randint(0, 900, (b,), generator=g, dtype=torch.int32)
    x = torch.randn(2 * b + 5, h, generator=g).bfloat16()
    lasts = torch.randint(0, 2 * b + 5, (b,), generator=g, dtype=torch.int32)
    lasts[0] = -1
    args = [t.to(dev) for t in (lens, off, slots, new, x, lasts)]
    got = hip_ops.prompts_end(*args)
    want = R.prompts_end(lens, off, slots, new, x, lasts)
    assert torch.equal(got.cpu(), want)
    assert torch.equal(args[0].cpu(), lens) and torch.equal(args[1].cpu(), off)
    args[1] += 3
    assert hip_ops.prompts_end(*args[:3], args[3] + 1, None, args[5]) is None
    assert torch.equal(args[0][args[2].long()], args[3] + 1)
    assert not args[1][args[2].long()].any()


@pytest.mark.parametrize("n,hq,hk,d,parts,bias", [
    (1, 3, 1, 16, 1, False), (45, 32, 8, 64, 4, True), (7, 24, 8, 128, 9, False)])
def test_rope_kv_of_parts_gpu(dev, n, hq, hk, d, parts, bias):
    """A product's partial sums and its bias: to the bit what its sum (by the
    first part's order, rounded) and the bias' addition by torch give."""
    torch.manual_seed(n)
    from gridllm_amd.ops import hip_ops
    ws = torch.randn(parts, n, (hq + 2 * hk) * d, device=dev)
    qkv = torch.zeros_like(ws[0])
    for x in ws:
        qkv += x
    qkv = qkv.to(torch.bfloat16)
    add = torch.randn_like(qkv[0]) if bias else None
    kc = torch.zeros(2, hk, 64, d, device=dev, dtype=torch.bfloat16)
    caches = [kc, kc.clone(), kc.clone(), kc.clone()]
    cos, sin = R.rope_tables(d, 128, device=dev)
    pos = torch.randint(0, 120, (n,), dtype=torch.int32, device=dev)
    slot = torch.randperm(128)[:n].int().to(dev)
    got = hip_ops.rope_kv(ws, *caches[:2], cos, sin, pos, slot, hq, hk, d, add)
    want = hip_ops.rope_kv(qkv if add is None else qkv + add, *caches[2:], cos,
                           sin, pos, slot, hq, hk, d)
    assert torch.equal(got, want) and torch.equal(caches[0], caches[2])
    assert torch.equal(caches[1], caches[3])


@pytest.mark.parametrize("m,n,k", [
    (1, 3072, 3072), (13, 5120, 3072), (64, 16384, 3072),
    (64, 3072, 8192), (127, 3072, 3072), (256, 128256, 3072),
])
def test_gemm_skinny_gpu(dev, m, n, k):
    """Skinny GEMM vs fp32 matmul of the same bf16 operands."""
    torch.manual_seed(9)
    from gridllm_amd.ops import hip_ops
    x = (torch.randn(m, k, device=dev) * 0.1).to(torch.bfloat16)
    w = (torch.randn(n, k, device=dev) * 0.1).to(torch.bfloat16)
    out = hip_ops.gemm_skinny(x, w)
    ref = x.float() @ w.float().t()
    err = (out.float() - ref).abs().max().item()
    assert err < 0.02 * ref.abs().max().item(), err


@pytest.mark.parametrize("m", [1, 2, 15, 16])
@pytest.mark.parametrize("n,k", [
    (128, 32), (1152, 896), (256, 224), (128, 4864), (2048, 2048),
    (128, 8192), (384, 1056), (128, 2304),
])
def test_gemm_rows_gpu(dev, m, n, k):
    """Rows, parts of K per wave (none, less than a batch, one and a part, two
    and a part, several) and columns at their edges. bf16 operands as given,
    f32 sums over K, one rounding of the result: 2^-9 of it and K 2^-24 of the
    sum of magnitudes."""
    torch.manual_seed(m + k)
    from gridllm_amd.ops import hip_ops
    x = torch.randn(m, k, device=dev).to(torch.bfloat16)
    w = torch.randn(n, k, device=dev).to(torch.bfloat16)
    ref = (x.cpu().double() @ w.cpu().double().t())
    bound = ref.abs() * 2 ** -8 + k * 2 ** -24 * (
        x.cpu().double().abs() @ w.cpu().double().abs().t())
    out = hip_ops.gemm_rows(x, w)
    assert ((out.cpu().double() - ref).abs() <= bound).all()
    w = w * k ** -0.5
    out = hip_ops.gemm_rows(x, w, fuse_swiglu=True)
    v = (x.cpu().double() @ w.cpu().double().t()).view(m, n // 128, 2, 64)
    g, u = v[:, :, 0].reshape(m, -1), v[:, :, 1].reshape(m, -1)
    assert _mx(out.cpu().double(), g * torch.sigmoid(g) * u) < 0.05


def test_gemm_skinny_splitk_consistent(dev):
    torch.manual_seed(10)
    from gridllm_amd.ops import hip_ops
    x = (torch.randn(64, 4096, device=dev) * 0.1).to(torch.bfloat16)
    w = (torch.randn(1024, 4096, device=dev) * 0.1).to(torch.bfloat16)
    o1 = hip_ops.gemm_skinny(x, w, splitk=1)
    o8 = hip_ops.gemm_skinny(x, w, splitk=8)
    assert (o1.float() - o8.float()).abs().max().item() < 0.05


@pytest.mark.parametrize("t,hq,hk,d,cau", [
    (128, 24, 8, 128, 0),     # llama3.2-3B shape, aligned T
    (77, 24, 8, 128, 0),      # ragged T (masked rows / partial tiles)
    (200, 24, 8, 128, 33),    # cached prefix: causal offset, s_total%32!=0
    (256, 32, 8, 64, 0),      # D=64 path, G=4
    (31, 8, 8, 128, 5),       # MHA (G=1), tiny T
])
def test_attn_prefill_mfma_gpu(dev, t, hq, hk, d, cau):
    """MFMA flash prefill vs fp32 torch reference, straight off the cache."""
    torch.manual_seed(t * 7 + cau)
    from gridllm_amd.ops import hip_ops
    smax, slots, slot = 512, 3, 1
    s_total = cau + t
    q = (torch.randn(t, hq, d, device=dev) * 0.5).to(torch.bfloat16)
    kc = (torch.randn(slots, hk, smax, d, device=dev) * 0.5).to(torch.bfloat16)
    vc = (torch.randn(slots, hk, smax, d, device=dev) * 0.5).to(torch.bfloat16)
    scale = 1.0 / math.sqrt(d)
    out = hip_ops.attn_prefill_cache(q, kc, vc, slot, s_total, cau, scale)
    kk = kc[slot, :, :s_total].permute(1, 0, 2).unsqueeze(0)
    vv = vc[slot, :, :s_total].permute(1, 0, 2).unsqueeze(0)
    ref = R.attn_prefill(q.unsqueeze(0).cpu().float(), kk.cpu().float(),
                         vv.cpu().float(), scale, causal_offset=cau)[0]
    assert _mx(out.cpu(), ref) < 0.03


@pytest.mark.parametrize("hq,hk,d", [(6, 2, 64), (8, 1, 128), (5, 1, 128)])
@pytest.mark.parametrize("nsplit", [0, 1, 3, 64, 100])
def test_attn_decode_step_edges_gpu(dev, hq, hk, d, nsplit):
    """Lengths at the edges of steps of 32 and 64 keys and of splits, scores
    that grow by more than the softmax reference's lag, NaN behind the last
    key. Only q, k, v (as given) and the output are bf16: half a unit of 2^-8
    of values up to 4."""
    torch.manual_seed(hq + nsplit)
    from gridllm_amd.ops import hip_ops
    seqs = [1, 15, 16, 17, 31, 32, 33, 64, 65, 127, 128, 129, 257, 640]
    b, smax = len(seqs), 640
    q = torch.randn(b, hq, d, device=dev).to(torch.bfloat16)
    kc = torch.randn(b, hk, smax, d, device=dev)
    kc = (kc * torch.linspace(0.1, 4, smax, device=dev).view(1, 1, -1, 1)).to(
        torch.bfloat16)
    vc = torch.randn(b, hk, smax, d, device=dev).to(torch.bfloat16)
    for i, n in enumerate(seqs):
        kc[i, :, n:], vc[i, :, n:] = float("nan"), float("nan")
    seqlen = torch.tensor(seqs, dtype=torch.int32, device=dev)
    out = hip_ops.attn_decode(q, kc, vc, seqlen, -d ** -0.5, nsplit=nsplit)
    for i, n in enumerate(seqs):
        ref = R.attn_decode(
            q[i:i + 1].cpu().float(), kc[i:i + 1, :, :n].cpu().float(),
            vc[i:i + 1, :, :n].cpu().float(), seqlen[i:i + 1].cpu(),
            -d ** -0.5)
        assert _mx(out[i:i + 1].cpu(), ref) < 0.01, n


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("t,cau,sign", [
    (1, 0, 1), (33, 0, 1), (64, 63, 1), (65, 64, 1), (128, 1, -1),
    (129, 191, 1), (300, 62, 1),
])
def test_attn_prefill_tile_edges_gpu(dev, t, cau, sign, d):
    """Rows and keys at the edges of tiles of 128 and 64, scores that grow by
    more than the softmax reference's lag from tile to tile, and NaN behind the
    last key, which nothing may read. Weights and the output are rounded to
    bf16 (2^-8 each), values are of the order of 1: 0.02 in the worst
    element."""
    torch.manual_seed(t + cau)
    from gridllm_amd.ops import hip_ops
    n, hq, hk = cau + t, 6, 2
    q = torch.randn(t, hq, d, device=dev).to(torch.bfloat16)
    kc = torch.randn(2, hk, 640, d, device=dev)
    kc = (kc * torch.linspace(0.1, 4, 640, device=dev).view(1, 1, -1, 1)).to(
        torch.bfloat16)
    vc = torch.randn(2, hk, 640, d, device=dev).to(torch.bfloat16)
    kc[:, :, n:], vc[:, :, n:] = float("nan"), float("nan")
    scale = sign * d ** -0.5
    out = hip_ops.attn_prefill_cache(q, kc, vc, 1, n, cau, scale)
    kk = kc[1, :, :n].permute(1, 0, 2).unsqueeze(0).cpu().float()
    vv = vc[1, :, :n].permute(1, 0, 2).unsqueeze(0).cpu().float()
    ref = R.attn_prefill(q.unsqueeze(0).cpu().float(), kk, vv, scale,
                         causal_offset=cau)[0]
    assert _mx(out.cpu(), ref) < 0.02


@pytest.mark.parametrize("m,n,k", [
    (256, 5120, 3072), (256, 3072, 8192), (128, 3072, 3072),
    (200, 16384, 3072),       # ragged M
    (512, 3072, 3072), (65, 128, 64),
])
def test_gemm_proj_gpu(dev, m, n, k):
    """Projection GEMM (M in (64,512]) vs fp32 matmul of the same operands."""
    torch.manual_seed(11)
    from gridllm_amd.ops import hip_ops
    x = (torch.randn(m, k, device=dev) * 0.1).to(torch.bfloat16)
    w = (torch.randn(n, k, device=dev) * 0.1).to(torch.bfloat16)
    out = hip_ops.gemm_proj(x, w)
    ref = x.float() @ w.float().t()
    err = (out.float() - ref).abs().max().item()
    assert err < 0.02 * ref.abs().max().item() + 1e-6, err


def test_gemm_proj_splitk_consistent(dev):
    torch.manual_seed(12)
    from gridllm_amd.ops import hip_ops
    x = (torch.randn(256, 8192, device=dev) * 0.1).to(torch.bfloat16)
    w = (torch.randn(1024, 8192, device=dev) * 0.1).to(torch.bfloat16)
    o1 = hip_ops.gemm_proj(x, w, splitk=1)
    o8 = hip_ops.gemm_proj(x, w, splitk=8)
    assert (o1.float() - o8.float()).abs().max().item() < 0.05


def test_gemm_proj_fused_swiglu_gpu(dev):
    """Fused-SwiGLU projection on interleaved weights vs the two-step
    reference (fp32 GEMM + silu*up), plus splitk consistency."""
    torch.manual_seed(13)
    from gridllm_amd.ops import hip_ops
    m, f, k = 256, 1024, 512
    x = (torch.randn(m, k, device=dev) * 0.1).to(torch.bfloat16)
    wg = (torch.randn(f, k, device=dev) * 0.1).to(torch.bfloat16)
    wu = (torch.randn(f, k, device=dev) * 0.1).to(torch.bfloat16)
    g = torch.arange(f)
    perm = torch.empty(2 * f, dtype=torch.int64)
    perm[(g // 64) * 128 + g % 64] = g
    perm[(g // 64) * 128 + g % 64 + 64] = f + g
    w_il = torch.cat([wg, wu])[perm.to(dev)].contiguous()

    gate = x.float() @ wg.float().t()
    up = x.float() @ wu.float().t()
    ref = gate * torch.sigmoid(gate) * up

    out = hip_ops.gemm_proj(x, w_il, fuse_swiglu=True)
    assert out.shape == (m, f)
    assert _mx(out.cpu(), ref.cpu()) < 0.02 * ref.abs().max().item() + 1e-6

    o1 = hip_ops.gemm_proj(x, w_il, splitk=1, fuse_swiglu=True)
    o4 = hip_ops.gemm_proj(x, w_il, splitk=4, fuse_swiglu=True)
    assert (o1.float() - o4.float()).abs().max().item() < 0.05

    # the library-GEMM fallback path over the same interleaved weight
    o_blas = hip_ops.swiglu_il(torch.nn.functional.linear(x, w_il))
    assert _mx(o_blas.cpu(), ref.cpu()) < 0.02 * ref.abs().max().item() + 1e-6


@pytest.mark.parametrize("m,n,k", [
    (256, 5120, 3072), (128, 3072, 8192), (200, 16384, 3072),
    (65, 256, 64),
])
def test_gemm_proj_wide_gpu(dev, m, n, k):
    """16-wave BN=256 variant vs fp32 matmul + splitk consistency."""
    torch.manual_seed(14)
    from gridllm_amd.ops import hip_ops
    x = (torch.randn(m, k, device=dev) * 0.1).to(torch.bfloat16)
    w = (torch.randn(n, k, device=dev) * 0.1).to(torch.bfloat16)
    out = hip_ops.gemm_proj_wide(x, w)
    ref = x.float() @ w.float().t()
    err = (out.float() - ref).abs().max().item()
    assert err < 0.02 * ref.abs().max().item() + 1e-6, err
    o1 = hip_ops.gemm_proj_wide(x, w, splitk=1)
    o4 = hip_ops.gemm_proj_wide(x, w, splitk=4)
    assert (o1.float() - o4.float()).abs().max().item() < 0.05


@pytest.mark.parametrize("b,v", [(1, 1), (3, 63), (2, 2047), (5, 4099),
                                 (1, 128256), (64, 8192), (1100, 515)])
def test_sample_gumbel_segments(dev, b, v):
    """Rows of one and of several segments, of odd lengths, with -inf, +inf,
    NaN, ties and close seconds, against the same formulas in 64-bit torch: the
    picked value has to be the largest to f32's accuracy, by slot with the keys
    of SlotSampler as with given keys."""
    from gridllm_amd.ops import hip_ops
    g = torch.Generator().manual_seed(b * v)
    x = torch.randn(b, v, generator=g) * 3
    x[:, ::3] = x[:, ::3].round()
    x[0, v // 2:] = float("-inf")
    if v > 8:
        x[-1, 5] = float("nan")
    if b > 2:
        x[1] = float("-inf")
        x[2, v - 1] = float("inf")
    seeds = torch.randint(0, 2 ** 62, (b,), generator=g)
    draws = torch.randint(0, 1000, (b,), generator=g)
    live = (torch.arange(b) % 4 != 3).long()
    temps = torch.rand(b, generator=g) + 0.3
    keys = (seeds * 6364136223846793005
            + (draws + 1) * 1442695040888963407) & ((1 << 63) - 1)
    keys = keys * live
    z = (torch.arange(v).unsqueeze(0) ^ keys.unsqueeze(1)) \
        * -7046029254386353131
    z = z ^ (z >> 29)
    z = z * -4658895280553007687
    z = z ^ (z >> 32)
    u = (((z >> 38) & 0xFFFFFF).float() / (1 << 24)).clamp(1e-6, 1 - 1e-6)
    val = x.double() / temps.double().unsqueeze(1) \
        - torch.log(-torch.log(u.double())) * live.unsqueeze(1)
    val = val.nan_to_num(nan=float("-inf"), posinf=1e30)
    slots = torch.randperm(b, generator=g)
    by = [torch.empty_like(t).index_copy(0, slots, t).to(dev)
          for t in (temps, seeds, draws, live)]
    got = hip_ops.sample_gumbel(x.to(dev), keys.to(dev), temps.to(dev))
    got2 = hip_ops.sample_gumbel_slots(x.to(dev), slots.to(dev), *by)
    assert torch.equal(got, got2)
    assert torch.equal(by[2].cpu()[slots], draws + 1)
    for r in range(b):
        best = val[r].max()
        if best == float("-inf"):
            assert got[r] == 0
        elif not live[r]:                     # no noise: the first of ties
            assert got[r] == (x[r] / temps[r]).nan_to_num(
                nan=float("-inf"), posinf=1e30).argmax()
        else:                                 # a logarithm of 1 - 1e-6 is good
            at = val[r, int(got[r])]          # to 2^-24 / 1e-6 in f32
            assert at >= best - 1e-5 * abs(best) - 1e-4


@pytest.mark.parametrize("b,v", [(1, 1), (3, 2047), (2, 4096), (64, 8192), (1, 128256),
                                 (20, 128256), (600, 4352), (1100, 515)])
def test_sample_gumbel_marks(dev, b, v):
    """Picks that meet in the slots' marks are those of the second kernel, call after
    call, with ties in all segments, -inf, +inf, NaN, flat and peaked rows, and
    rows without noise; the marks are zeros again."""
    from gridllm_amd.ops import hip_ops
    g = torch.Generator().manual_seed(b + v)
    x = torch.randn(b, v, generator=g) * 2
    x[::5] = x[::5].round()
    x[::7, ::2] = float("-inf")
    if b > 2:
        x[1] = float("-inf")
        x[2, ::3] = 0.0
        x[2, 1::3] = -0.0
    if b > 20:
        x[20], x[19, v // 3], x[18, v // 2], x[17, ::9] = 1.0, 30.0, float(
            "inf"), float("nan")
    x = x.to(dev)
    slots = torch.randperm(b + 3, generator=g)[:b].to(dev)
    temps = (torch.rand(b + 3, generator=g) + 0.3).to(dev)
    seeds = torch.randint(0, 2 ** 62, (b + 3,), generator=g).to(dev)
    live = (torch.arange(b + 3) % 4 != 3).long().to(dev)
    draws, marks = torch.zeros_like(seeds), torch.zeros(b + 3, 16, dtype=torch.int64,
                                                        device=dev)
    draws2 = draws.clone()
    for _ in range(4):
        got = hip_ops.sample_gumbel_slots(x, slots, temps, seeds, draws, live, marks)
        want = hip_ops.sample_gumbel_slots(x, slots, temps, seeds, draws2, live)
        assert torch.equal(got, want) and torch.equal(draws, draws2)
        assert not marks.any()
    with pytest.raises(ValueError):
        hip_ops.sample_gumbel_slots(x, slots, temps, seeds, draws, live, marks[1:])


@pytest.mark.parametrize("b,v", [(2, 1), (3, 2047), (5, 128256), (40, 8195),
                                 (600, 4352)])
def test_sample_gumbel_slots_twice(dev, b, v):
    """Rows that name one slot get its key each, as without marks, and the marks and
    the other rows' tokens are what they are without such rows."""
    from gridllm_amd.ops import hip_ops
    g = torch.Generator().manual_seed(b + v)
    x = (torch.randn(b, v, generator=g) * 2).to(dev)
    temps = (torch.rand(b, generator=g) + 0.3).to(dev)
    seeds = torch.randint(0, 2 ** 62, (b,), generator=g).to(dev)
    live = (torch.arange(b) % 4 != 3).long().to(dev)
    slots = torch.randperm(b, generator=g)
    slots[b // 2], slots[-1] = slots[0], slots[b // 3]
    count = torch.zeros(b, dtype=torch.int64)
    count[slots] = 1
    keys = (seeds * 6364136223846793005 + 1442695040888963407) & ((1 << 63) - 1)
    slots = slots.to(dev)
    want = hip_ops.sample_gumbel(x, (keys * live)[slots], temps[slots])
    draws, marks = torch.zeros_like(seeds), torch.zeros(b, 16, dtype=torch.int64,
                                                        device=dev)
    got = hip_ops.sample_gumbel_slots(x, slots, temps, seeds, draws, live, marks)
    assert torch.equal(got, want)
    assert torch.equal(draws.cpu(), count) and not marks.any()


@pytest.mark.parametrize("b,v", [(1, 128256), (6, 2048), (6, 2049), (40, 128256),
                                 (600, 9000)])
def test_sample_gumbel_masked(dev, b, v):
    """Rows of which a mask leaves one candidate, some, or none, by -inf or by the
    least number, and rows with +inf: segments of one batch a wave and of several."""
    from gridllm_amd.ops import hip_ops
    g = torch.Generator().manual_seed(b + v)
    x = torch.full((b, v), float("-inf"))
    left = torch.randint(0, v, (b, 9), generator=g)
    x[1::6] = torch.finfo(torch.float32).min
    x.scatter_(1, left, torch.randn(b, 9, generator=g))
    x[2::6] = float("-inf")
    x[3::6].scatter_(1, left[3::6, :2], float("inf"))
    x[4::6].scatter_(1, left[4::6, 1:], float("-inf"))
    temps = torch.rand(b, generator=g) + 0.3
    keys = torch.randint(1, 2 ** 62, (b,), generator=g)
    z = (torch.arange(v).unsqueeze(0) ^ keys.unsqueeze(1)) * -7046029254386353131
    z = (z ^ (z >> 29)) * -4658895280553007687
    z = z ^ (z >> 32)
    u = (((z >> 38) & 0xFFFFFF).float() / (1 << 24)).clamp(1e-6, 1 - 1e-6).double()
    val = x.double() / temps.double().unsqueeze(1) - torch.log(-torch.log(u))
    got = hip_ops.sample_gumbel(x.to(dev), keys.to(dev), temps.to(dev)).cpu()
    # (the first of equal ones; no two of these others are next to each other)
    assert torch.equal(got.long(), val.argmax(1))


@pytest.mark.parametrize("b,v", [(7, 256), (5, 257), (3, 511), (4, 512), (2, 2049),
                                 (3, 4096), (2, 6400), (1, 133000), (600, 4352)])
def test_sample_gumbel_chunks(dev, b, v):
    """The same at the edges of chunks of 256, of a wave's pair of them, and of
    segments, the last of which has nothing where they are rounded up to chunks;
    and behind 2^17 candidates."""
    test_sample_gumbel_segments(dev, b, v)


@pytest.mark.skipif(os.environ.get("GRIDLLM_FUSED_SAMPLER") == "0",
                    reason="fused sampler explicitly disabled")
def test_sample_gumbel_matches_eager(dev):
    """Fused Gumbel-argmax vs the torch eager chain in sampler.py —
    identical splitmix64 stream, so tokens must match except ulp-level
    log() near-ties (allow 0.5% of rows)."""
    from gridllm_amd.engine.sampler import BatchPlan, sample_batch_vectorized
    from gridllm_amd.engine.sampler import SamplerState
    from gridllm_amd.ops import hip_ops
    from gridllm_amd.types import SamplingOptions
    torch.manual_seed(5)
    b, v = 512, 4096
    logits = torch.randn(b, v, device=dev) * 3
    states = [SamplerState.create(
        SamplingOptions.from_dict(
            {"temperature": 0.3 + (r % 7) * 0.2, "seed": r}
            if r % 5 else {"temperature": 0.0}),   # mix in greedy rows
        torch.device(dev)) for r in range(b)]
    plan = BatchPlan()
    plan.refresh(states, logits.device, v)
    fused = hip_ops.sample_gumbel(
        logits.contiguous(),
        plan.keys(states, logits.device).view(-1).contiguous(),
        plan.temps.view(-1).contiguous()).tolist()
    os.environ["GRIDLLM_FUSED_SAMPLER"] = "0"
    try:
        eager = sample_batch_vectorized(logits.clone(), states, BatchPlan())
    finally:
        os.environ["GRIDLLM_FUSED_SAMPLER"] = "1"
    mismatch = sum(1 for a, b2 in zip(fused, eager) if a != b2)
    assert mismatch <= b * 0.005, (mismatch, b)


def test_attn_prefill_batch_varlen(dev):
    """Varlen batched prefill (one meta-driven launch) must match the
    per-sequence kernel on every packed sequence, incl. multi-tile
    (T>128) and single-token rows."""
    torch.manual_seed(11)
    import numpy as np
    from gridllm_amd.ops import hip_ops
    hq, hk, d, smax = 24, 8, 128, 512
    lens = [26, 1, 200, 128, 77]
    slots = [4, 1, 6, 0, 3]
    scale = 1.0 / math.sqrt(d)
    total = sum(lens)
    q = (torch.randn(total, hq, d, device=dev) * 0.5).to(torch.bfloat16)
    kc = (torch.randn(8, hk, smax, d, device=dev) * 0.5).to(torch.bfloat16)
    vc = (torch.randn(8, hk, smax, d, device=dev) * 0.5).to(torch.bfloat16)
    bounds = [0]
    for ln in lens:
        bounds.append(bounds[-1] + ln)
    rows = [(bounds[i], ln, sl, q0)
            for i, (ln, sl) in enumerate(zip(lens, slots))
            for q0 in range(0, ln, 128)]
    meta = torch.from_numpy(np.asarray(rows, dtype=np.int32)).to(dev)
    out = hip_ops.attn_prefill_cache_batch(q, kc, vc, meta, scale)
    for i, (ln, sl) in enumerate(zip(lens, slots)):
        ref = hip_ops.attn_prefill_cache(
            q[bounds[i]:bounds[i + 1]].contiguous(), kc, vc, sl, ln, 0,
            scale)
        err = _mx(out[bounds[i]:bounds[i + 1]].cpu(), ref.cpu())
        assert err < 1e-3, (i, err)


@pytest.mark.parametrize("name", ["qwen2.5:0.5b", "llama3.2:3b"])
def test_prompt_layers_by_call(dev, name, monkeypatch):
    """A prompt's layers by native calls give what their launches from Python
    give, to the bit: rows for each kind of product, with and without a bias, new
    and continued sequences, one and several. A layer that a kernel does not read
    is left to Python."""
    from dataclasses import replace
    from gridllm_amd.models import llama
    from gridllm_amd.models.registry import get_spec
    spec = replace(get_spec(name), layers=3, vocab=1024)
    m = llama.LlamaModel(spec, device=str(dev), dtype="bf16", seed=3, kv_slots=4,
                         max_seq=1024)
    m.interleave_gateup()
    calls, kinds = [], set()
    native = llama.LlamaModel._layers_by_call
    choice = llama._choice_of

    def counted(self, *args):
        calls.append(native(self, *args))
        return calls[-1]

    def seen(*args):
        c = choice(*args)
        kinds.add(c and c[0])
        return c
    monkeypatch.setattr(llama, "_choice_of", seen)

    def run():
        g = torch.Generator().manual_seed(1)
        out = []
        for t in (1, 4, 16, 17, 64, 65, 257, 300):
            ids = torch.randint(0, 1024, (t,), generator=g).to(dev)
            more = torch.randint(0, 1024, (33,), generator=g).to(dev)
            slot = m.cache.alloc(t + 33)
            out.append(m.forward_prefill(ids, slot))
            out.append(m.forward_prefill(more, slot, start_pos=t))
            m.cache.free(slot)
        slots = [m.cache.alloc(40) for _ in range(3)]
        out.append(m.forward_prefill_batch(
            [torch.arange(n, device=dev) for n in (40, 1, 17)], slots))
        for sl in reversed(slots):
            m.cache.free(sl)
        return out + [t.clone() for t in m.cache.k + m.cache.v]
    monkeypatch.setattr(llama.LlamaModel, "_layers_by_call", counted)
    got = run()
    assert len(calls) == 17 and all(calls[:12]) and set(calls) <= {0, 2, 3}
    assert {"tile", "rows"} <= kinds
    monkeypatch.setattr(llama.LlamaModel, "_layers_by_call", lambda *a: 0)
    for a, b in zip(got, run()):
        assert torch.equal(a, b)
    monkeypatch.setattr(llama.LlamaModel, "_layers_by_call", counted)
    lw = m.layers[1]
    lw.wo = lw.wo.t().contiguous().t()
    calls.clear()
    m.forward_prefill(torch.arange(20, device=dev), m.cache.alloc(20))
    assert calls == [0]


def test_prefill_batch_engine_parity(dev):
    """forward_prefill_batch (varlen kernel path) vs sequential
    forward_prefill on the GPU engine: same logits, same KV."""
    from gridllm_amd.models.llama import LlamaModel
    from gridllm_amd.models.registry import get_spec
    spec = get_spec("llama3.2:1b", 512)
    m1 = LlamaModel(spec, device=str(dev), dtype="bf16", kv_slots=8,
                    max_seq=512)
    torch.manual_seed(3)
    prompts = [torch.randint(0, spec.vocab, (n,), device=dev)
               for n in (19, 140, 1, 64)]
    seq_slots = [0, 1, 2, 3]
    bat_slots = [4, 5, 6, 7]
    l_seq = torch.stack([m1.forward_prefill(p, s)
                         for p, s in zip(prompts, seq_slots)])
    l_bat = m1.forward_prefill_batch(prompts, bat_slots)
    # GEMMs run at M=sum(T_i) in the batched pass vs per-sequence M in the
    # sequential one -> different tile/split choices -> different bf16
    # accumulation order through 16 layers. The attention kernel itself is
    # exact (test_attn_prefill_batch_varlen, <1e-3); here bound the
    # logit-level rounding drift instead of bit equality.
    diff = (l_bat.float() - l_seq.float()).abs()
    assert diff.max().item() < 0.25, diff.max().item()
    assert diff.mean().item() < 0.03, diff.mean().item()
    # K comes off the qkv GEMM, which runs at M=sum vs M=T_i: layer 0
    # differs by bf16 output ulps only; deeper layers compound that
    # activation drift (checked via the logit bound above, not per-layer)
    for i in range(len(prompts)):
        n = prompts[i].shape[0]
        dk = _mx(m1.cache.k[0][seq_slots[i], :, :n].cpu(),
                 m1.cache.k[0][bat_slots[i], :, :n].cpu())
        assert dk < 1.6e-2, (i, dk)


@pytest.mark.parametrize("name", ["llama3.2:1b", "qwen2.5:0.5b"])
def test_last_layer_of_wanted_rows_alone(dev, name):
    """Logits and caches of prompts whose last layer runs for their last tokens
    alone, against passes that run it for all (with biases and without)."""
    from dataclasses import replace
    from gridllm_amd.models.llama import LlamaModel
    from gridllm_amd.models.registry import get_spec
    spec = replace(get_spec(name, 1024), layers=2)
    torch.manual_seed(3)
    a, b, c = (torch.randint(0, spec.vocab, (n,), device=dev)
               for n in (257, 300, 7))
    got, want = [], []
    models = [LlamaModel(spec, device=str(dev), dtype="bf16", kv_slots=6,
                         max_seq=1024, seed=1) for _ in range(2)]
    for m, out, hidden in zip(models, (got, want), (False, True)):
        m.interleave_gateup()
        for r in (m.forward_prefill(a, 2, 0, hidden),
                  m.forward_prefill(b, 2, 257, hidden),
                  m.forward_prefill_batch([c, a, b], [1, 4, 3], hidden)):
            out.append(r[0] if hidden else r)
    # products of other row counts: two bf16 roundings a sublayer, 2^-9 each
    for x, y in zip(got, want):
        assert x.shape == y.shape
        assert ((x - y).norm() / y.norm()).item() < 0.02
    for x, y in zip(models[0].cache.k + models[0].cache.v,
                    models[1].cache.k + models[1].cache.v):
        for s, n in ((2, 557), (1, 7), (4, 257), (3, 300)):
            d = (x[s, :, :n].float() - y[s, :, :n].float()).norm()
            assert d.item() <= 0.01 * y[s, :, :n].float().norm().item()


@pytest.mark.parametrize("fuse", [False, True])
@pytest.mark.parametrize("m,n,k,sk", [
    (17, 384, 64, 1),          # one tile of K
    (33, 384, 512, 1),         # as many as buffers, or one more or less
    (1, 128, 576, 3),          # parts of fewer tiles than buffers
    (95, 1152, 896, 4),        # the last part shorter
    (160, 2176, 1088, 1),      # a number of blocks that 8 does not divide
    (161, 640, 3072, 5), (257, 256, 1024, 2), (700, 384, 640, 1),
])
def test_gemm_tile(dev, m, n, k, sk, fuse):
    """Every tile size against f32, at edges of rows, of K's parts and of the
    ring of tiles in LDS."""
    from gridllm_amd.ops import hip_ops
    n = n // 128 * 128 if fuse else n
    g = torch.Generator().manual_seed(m + k)
    x = torch.randn(m, k, generator=g).to(dev, torch.bfloat16)
    w = torch.randn(n, k, generator=g).to(dev, torch.bfloat16)
    ref = x.float() @ w.float().t()
    # bf16 result: 2^-9 of its size; K products' sums: k eps of their sizes' sum
    tol = 2 ** -8 * ref.abs() + k * 2 ** -24 * (x.float().abs() @
                                                w.float().abs().t()) + 1e-6
    if fuse:
        gate, up = ref.view(m, -1, 2, 64).unbind(2)
        ref = (gate * torch.sigmoid(gate) * up).reshape(m, -1)
        # (the unit's exponential is the hardware's)
        gt, ut = tol.view(m, -1, 2, 64).unbind(2)
        tol = (2 ** -8 * (gate * up).abs() + 1.2 * gt * up.abs() +
               gate.abs() * ut).reshape(m, -1) + 1e-4
    out = torch.empty_like(ref, dtype=torch.bfloat16)
    for rows in (32, 64, 96, 128, 160, 192, 256):
        for cols in (64, 128) if fuse else (64, 96, 128):
            if n % cols == 0:
                hip_ops.gemm_tile(x, w, rows, cols, sk, out.fill_(9e9), fuse)
                assert bool(((out.float() - ref).abs() <= tol).all()), \
                    (rows, cols)


@pytest.mark.parametrize("fuse", [False, True])
@pytest.mark.parametrize("m,n,k,sk", [
    (1, 2304, 2048, 1),        # blocks start at every place of K but the last ones
    (33, 4480, 2048, 1),       # at every one, some twice
    (40, 1152, 4096, 9),       # parts of K, the last one shorter
    (257, 384, 2048, 31),      # of fewer tiles than buffers
])
def test_gemm_tile_long_rows(dev, m, n, k, sk, fuse):
    """The same where rows are a multiple of 4096 bytes: blocks start at different
    places of K, and wrap."""
    test_gemm_tile(dev, m, n, k, sk, fuse)


@pytest.mark.parametrize("fuse", [False, True])
@pytest.mark.parametrize("m,n,k,sk", [(257, 1152, 1600, 1), (257, 1152, 3136, 2)])
def test_gemm_tile_several_blocks(dev, m, n, k, sk, fuse):
    """The same where several blocks of rows read weights through the cache: K in one
    part, and in two of unequal length."""
    from gridllm_amd.ops import hip_ops
    for rows in (32, 64, 96, 128, 160, 192, 256):
        assert not hip_ops.gemm_tile_once(m, n, k, rows, sk)
    test_gemm_tile(dev, m, n, k, sk, fuse)


@pytest.mark.parametrize("m,n,k", [(1, 64, 64), (33, 192, 576),
                                   (257, 8256, 128)])
def test_gemm_tile_f32(dev, m, n, k):
    """The result as f32 is that of bf16, widened, to the bit."""
    from gridllm_amd.ops import hip_ops
    g = torch.Generator().manual_seed(n)
    x, w = (torch.randn(*s, generator=g).to(dev, torch.bfloat16)
            for s in ((m, k), (n, k)))
    for cols in (64, 96):
        if n % cols == 0:
            assert torch.equal(hip_ops.gemm_tile_f32(x, w, 64, cols),
                               hip_ops.gemm_tile(x, w, 64, cols).float())


@pytest.mark.parametrize("m,n,k,sk", [(1, 64, 128, 2), (24, 3072, 1024, 5),
                                      (70, 2112, 576, 9), (3, 8256, 256, 2)])
def test_gemm_tile_rmsnorm(dev, m, n, k, sk):
    """Partial sums that the norm adds up: what the two steps give, to a rounding
    of the sum where the parts' sum is taken in another order."""
    from gridllm_amd import ops
    from gridllm_amd.ops import hip_ops
    g = torch.Generator().manual_seed(n)
    x, w, r = (torch.randn(*s, generator=g).to(dev, torch.bfloat16)
               for s in ((m, k), (n, k), (m, n)))
    weight = (torch.rand(n, generator=g) + 0.5).to(dev, torch.bfloat16)
    y, total = hip_ops.gemm_tile_rmsnorm(x, w, 64, 64, sk, weight, 1e-5, r)
    want, res = ops.rmsnorm(hip_ops.gemm_tile(x, w, 64, 64, sk), weight, 1e-5,
                            residual=r)
    # (product, then its sum with the residual: one bf16 step, 2^-8, each)
    size = res.float().abs() + x.float().norm(dim=1, keepdim=True) * 8
    assert bool(((total.float() - res.float()).abs() <= 2 ** -7 * size).all())
    assert float((total != res).float().mean()) < 0.01
    assert bool(((y.float() - want.float()).abs() <=
                 2 ** -6 * want.float().abs() + 2 ** -6).all())


def test_gemm_tilings():
    """What the tuner tries is what the kernel takes."""
    from gridllm_amd.ops import hip_ops
    for m in (1, 16, 17, 64, 129, 160, 256, 300, 1024, 2048):
        for n, k in ((64, 64), (192, 896), (3072, 8192), (128256, 3072),
                     (100, 64), (128, 96)):
            for fuse in (False, True):
                for rows, cols, sk in hip_ops.gemm_tilings(m, n, k, fuse):
                    assert n % cols == 0 and k % 64 == 0 and sk >= 1
                    assert rows in (32, 64, 96, 128, 160, 192, 256)
                    assert sk == 1 or (sk * -(-m // rows) * n // cols <= 256
                                       and k // sk >= 64)
                rule = hip_ops.gemm_tiling(m, n, k, fuse)
                assert rule is None or (rule[0] in (
                    32, 64, 96, 128, 160, 192, 256) and n % rule[1] == 0
                    and k % 64 == 0 and k // rule[2] >= 64)
                assert not (rule and fuse and (n % 128 or rule[1] == 96))


@pytest.mark.parametrize("stages", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 32])
def test_gemm_fed_stages(dev, stages):
    """Blocks that have fewer stages of K than their rings, as many, and some more,
    odd and even; 48 columns too; rows behind the last one."""
    from gridllm_amd.ops import hip_ops
    k = 64 * stages
    g = torch.Generator().manual_seed(stages)
    x, w = (torch.randn(*s, generator=g).to(dev, torch.bfloat16)
            for s in ((261, k), (384, k)))
    ref = x.float() @ w.float().t()
    tol = 2 ** -8 * ref.abs() + k * 2 ** -24 * (x.float().abs() @
                                                w.float().abs().t()) + 1e-6
    for rows in (96, 128, 160, 192, 256):
        for cols in (48, 64, 96, 128):
            out = hip_ops.gemm_tile(x, w, rows, cols, 1,
                                    torch.full_like(ref, 9e9).bfloat16())
            assert bool(((out.float() - ref).abs() <= tol).all()), (rows, cols)
    for rows in (32, 64, 96, 128, 160):        # 256 columns: up to 160 rows
        out = hip_ops.gemm_tile_f32(x, w[:256], rows, 256)
        assert bool(((out - ref[:, :256]).abs() <= tol[:, :256]).all()), rows
    for rows, cols in ((32, 48), (64, 48), (192, 256), (256, 256)):
        with pytest.raises(RuntimeError):
            hip_ops.gemm_tile(x, w[:256] if cols == 256 else w, rows, cols)


@pytest.mark.parametrize("m,n,k,sk", [(1, 192, 576, 2), (100, 960, 1088, 4),
                                      (257, 1536, 2048, 5), (300, 6144, 320, 2)])
def test_gemm_fed_parts(dev, m, n, k, sk):
    """Parts of K, the last one shorter, in 48 columns, too; results as f32; and the
    norm that adds the parts up, of one turn of threads and two."""
    from gridllm_amd import ops
    from gridllm_amd.ops import hip_ops
    g = torch.Generator().manual_seed(m + k)
    x, w, r = (torch.randn(*s, generator=g).to(dev, torch.bfloat16)
               for s in ((m, k), (n, k), (m, n)))
    weight = (torch.rand(n, generator=g) + 0.5).to(dev, torch.bfloat16)
    ref = x.float() @ w.float().t()
    tol = 2 ** -8 * ref.abs() + k * 2 ** -24 * (x.float().abs() @
                                                w.float().abs().t()) + 1e-6
    for rows in (96, 128, 160, 192, 256):
        for cols in (48, 64, 96, 128):
            if n % cols:
                continue
            out = hip_ops.gemm_tile(x, w, rows, cols, sk,
                                    torch.full_like(ref, 9e9).bfloat16())
            assert bool(((out.float() - ref).abs() <= tol).all()), (rows, cols)
            whole = hip_ops.gemm_tile(x, w, rows, cols, 1)
            assert torch.equal(hip_ops.gemm_tile_f32(x, w, rows, cols),
                               whole.float()), (rows, cols)
            parts = hip_ops.gemm_tile_parts(x, w, rows, cols, sk)
            assert bool(((parts.sum(0) - ref).abs() <= tol).all()), (rows, cols)
    # the norm adds up in the order of the parts, and rounds as the product does
    for rows, cols in ((96, 48), (256, 64)):
        parts = hip_ops.gemm_tile_parts(x, w, rows, cols, sk)
        total = torch.zeros_like(parts[0])
        for part in parts:
            total = total + part
        y, res = hip_ops.gemm_tile_rmsnorm(x, w, rows, cols, sk, weight, 1e-5, r)
        want, res2 = ops.rmsnorm(total.bfloat16(), weight, 1e-5, residual=r)
        assert torch.equal(res, res2) and torch.equal(y, want)


@pytest.mark.parametrize("m,n,k", [
    (1, 8, 256),               # one row and 8 columns of a tile; 4 stages
    (255, 256, 256), (257, 264, 320), (384, 1032, 576),
    (192, 512, 832),           # whole tiles, then one row more
    (193, 576, 832),
    (1000, 17 * 256, 256),     # more tiles than an XCD's CUs, 8 divides not
    (2100, 9 * 1024 + 128, 384),       # several tiles a block
])
def test_gemm_wide(dev, m, n, k):
    """Every shape and way to halve the last tiles against f32: edges of rows and
    columns, the least K, blocks of one and of several tiles."""
    from gridllm_amd.ops import hip_ops
    from gridllm_amd.ops.reference import Glu
    g = torch.Generator().manual_seed(m + k)
    x = torch.randn(m, k, generator=g).to(dev, torch.bfloat16)
    w = torch.randn(n, k, generator=g).to(dev, torch.bfloat16)
    ref = x.float() @ w.float().t()
    # bf16 rounding, and f32 sums of k products in another order
    room = 2 ** -8 * ref.abs() + k * 2e-7 * (k ** 0.5)
    tiles = -(-m // 256) * -(-n // 256)
    for shape, whole in [(0, 0), (0, 1), (0, tiles // 2), (0, tiles), (1, 0),
                         (2, 0), (3, 0)]:
        out = hip_ops.gemm_wide(x, w, shape, whole)
        assert bool(((out.float() - ref).abs() <= room).all()), (shape, whole)
    plain = hip_ops.gemm_wide(x, w, 0, tiles)
    for shape, whole in ((0, tiles // 2), (4, 0)):
        out = hip_ops.gemm_wide(x, w, shape, whole, f32=True)
        assert out.dtype == torch.float32 and torch.equal(out, plain.float())
    if n % 128:
        return
    glu = Glu(1.3, 2.0, 0.5, 0.1)
    # the unit is that of the rounded results
    a, b = plain.float().view(m, -1, 2, 64).unbind(2)
    a, b = a.clamp(max=2.0), b.clamp(-2.0, 2.0)
    act = (a * torch.sigmoid(1.3 * a * (1 + 0.1 * a * a))
           * (b + 0.5)).reshape(m, -1)
    for shape, whole in ((0, 0), (0, tiles), (0, tiles // 2), (4, 0)):
        out = hip_ops.gemm_wide(x, w, shape, whole, fuse_swiglu=True, glu=glu)
        # half a step of the result's 8 bits; its exponential is the hardware's
        assert bool(((out.float() - act).abs() <= 2 ** -8 * act.abs() +
                     1e-6).all()), (shape, whole)


def test_gemm_wide_refuses(dev):
    """Sizes and shapes that the kernel has not, ahead of a launch."""
    from gridllm_amd.ops import hip_ops

    def t(*s):
        return torch.zeros(*s, dtype=torch.bfloat16, device=dev)
    for m, n, k, shape, kw in ((256, 256, 192, 0, {}), (256, 256, 288, 0, {}),
                               (256, 252, 256, 0, {}), (256, 256, 256, 5, {}),
                               (256, 256, 256, 4, {}), (256, 256, 256, -1, {}),
                               (256, 192, 256, 0, dict(fuse_swiglu=True)),
                               (256, 256, 256, 1, dict(f32=True))):
        with pytest.raises(RuntimeError):
            hip_ops.gemm_wide(t(m, k), t(n, k), shape, 1, **kw)
    with pytest.raises(RuntimeError):
        hip_ops.gemm_wide(t(256 * 256 + 1)[1:].view(256, 256), t(256, 256), 0, 1)


def test_linear_of_many_rows(dev):
    """What the rule runs products of more than 256 rows by, against F.linear."""
    import torch.nn.functional as F
    from gridllm_amd.ops import autotune
    g = torch.Generator().manual_seed(2)
    took = set()
    for m, n, k in ((257, 1152, 896), (300, 2048, 8192), (700, 896, 4864),
                    (1201, 1152, 896), (1500, 17920, 384), (3000, 512, 3072)):
        x = torch.randn(m, k, generator=g).to(dev, torch.bfloat16)
        w = torch.randn(n, k, generator=g).to(dev, torch.bfloat16)
        for fuse in (False, True):
            took.add(autotune._rule(m, n, k, fuse)[0])
            got = autotune.linear_gateup(x, w) if fuse else autotune.linear(x, w)
            want = F.linear(x, w)
            if fuse:
                a, b = want.float().view(m, -1, 2, 64).unbind(2)
                want = (F.silu(a) * b).reshape(m, -1)
            # two roundings of the products, up to two bf16 steps each
            err = (got.float() - want.float()).norm() / want.float().norm()
            assert err.item() < 2 ** -7, (m, n, k, fuse)
    assert took == {"blas", "tile", "wide"}


@pytest.mark.parametrize("m,n,k,way", [
    (350, 32000, 2048, "blas"), (2000, 1024, 896, "blas"),
    (700, 32064, 896, "wide"), (260, 512, 128, "tile"), (300, 520, 64, "blas")])
def test_scores_of_many_rows(dev, m, n, k, way):
    """linear_f32 of more than 256 rows: by the kernels that have such results, and
    by the library where a product in bf16 goes by a shape that has none."""
    import torch.nn.functional as F
    from gridllm_amd.ops import autotune
    assert autotune._rule(m, n, k, f32=True)[0] == way
    g = torch.Generator().manual_seed(5)
    x = torch.randn(m, k, generator=g).to(dev, torch.bfloat16)
    w = torch.randn(n, k, generator=g).to(dev, torch.bfloat16)
    got, want = autotune.linear_f32(x, w), F.linear(x, w).float()
    assert got.dtype == torch.float32 and got.shape == want.shape
    # f32 sums in another order: some results round to bf16's neighbour
    assert bool(((got - want).abs() <= 2 ** -7 * want.abs() +
                 k * 2e-7 * k ** 0.5).all())


def test_whole_products_are_nearly_all_the_librarys(dev):
    """Of products of more than 256 rows that are not in parts of K, 99.9 % and more
    of the results are the library's to the bit, and so are gated units those of the
    kernel behind it."""
    import torch.nn.functional as F
    from gridllm_amd.ops import autotune, hip_ops
    g = torch.Generator().manual_seed(2)
    took = set()
    for m, n, k in ((257, 1152, 896), (490, 3072, 8192), (490, 16384, 3072),
                    (700, 896, 4864), (1201, 1152, 896), (2731, 3072, 3072),
                    (2731, 16384, 3072)):
        x = torch.randn(m, k, generator=g).to(dev, torch.bfloat16)
        w = (torch.randn(n, k, generator=g) * 0.1).to(dev, torch.bfloat16)
        c = autotune._rule(m, n, k, False, True)
        took |= {c[0], autotune._rule(m, n, k, True, True)[0]}
        y = F.linear(x, w)
        same = autotune.linear(x, w, whole=True) == y
        # (where the library cuts K for some of its own tiles, which only it knows,
        # a few sums differ in their last bit)
        assert same.float().mean().item() > 0.999, (m, n, k)
        got = autotune.linear_gateup(x, w, whole=True)
        want = hip_ops.swiglu_il(y)
        assert (got == want).float().mean().item() > 0.999, (m, n, k)
    assert took == {"blas", "wide"}


@pytest.mark.parametrize("m,n,k,mt,sk", [
    (256, 5120, 3072, 2, 1),   # qkv m-tiled
    (256, 5120, 3072, 2, 3),   # + splitk compose
    (256, 16384, 3072, 4, 1),  # gateup, 64-row tiles (4-wave path)
    (192, 3072, 8192, 2, 4),   # down, ragged M
    (96, 3072, 3072, 2, 1),    # rpt<=64 with partial last tile
    (768, 5120, 3072, 6, 1),   # serving bucket ABOVE the plain-proj cap
    (1024, 3072, 8192, 8, 2),  # b1024 down, m-tiled + splitk
])
def test_gemm_proj_mtiled(dev, m, n, k, mt, sk):
    """M-tiled projection decomposition vs fp32 reference."""
    torch.manual_seed(m + mt)
    from gridllm_amd.ops import hip_ops
    x = (torch.randn(m, k, device=dev) * 0.1).to(torch.bfloat16)
    w = (torch.randn(n, k, device=dev) * 0.1).to(torch.bfloat16)
    ref = x.float() @ w.float().t()
    out = hip_ops.gemm_proj(x, w, splitk=sk, mtiles=mt)
    err = (out.float() - ref).abs().max().item()
    assert err < 0.02 * ref.abs().max().item() + 1e-6, err


def test_gemm_proj_mtiled_fused_swiglu(dev):
    """M-tiled + fused SwiGLU epilogue on an interleaved gate/up weight."""
    torch.manual_seed(9)
    from gridllm_amd.ops import hip_ops
    m, f, k = 256, 8192, 3072
    x = (torch.randn(m, k, device=dev) * 0.1).to(torch.bfloat16)
    wg = (torch.randn(f, k, device=dev) * 0.1).to(torch.bfloat16)
    wu = (torch.randn(f, k, device=dev) * 0.1).to(torch.bfloat16)
    # interleave rows into 128-row groups [64 gate | 64 up]
    g = torch.arange(f)
    perm = torch.empty(2 * f, dtype=torch.int64)
    perm[(g // 64) * 128 + g % 64] = g
    perm[(g // 64) * 128 + g % 64 + 64] = f + g
    w_il = torch.cat([wg, wu])[perm.to(dev)].contiguous()
    gate = (x.float() @ wg.float().t())
    up = (x.float() @ wu.float().t())
    ref = gate * torch.sigmoid(gate) * up
    for mt in (2, 4):
        out = hip_ops.gemm_proj(x, w_il, splitk=1, fuse_swiglu=True,
                                mtiles=mt)
        err = (out.float() - ref).abs().max().item()
        assert err < 0.03 * ref.abs().max().item() + 1e-5, (mt, err)


def test_slot_sampler_takes_host_slots(dev):
    """Slot numbers on the host, as torch's indexing takes them."""
    from gridllm_amd.engine.sampler import SlotSampler
    x = torch.randn(3, 5000, device=dev)

    class Row:
        class state:
            greedy = need_filter = False
    out = []
    for slots in (torch.tensor([4, 0, 2]), torch.tensor([4, 0, 2]).to(dev)):
        sm = SlotSampler(5, dev)
        sm.temps.fill_(0.7)
        sm.nongreedy.fill_(1)
        sm.seeds.copy_(torch.arange(5) + 3)
        out.append(sm.sample_ids(x, [Row] * 3, slots).tolist())
        assert sm.draws.tolist() == [1, 0, 1, 0, 1]
    assert out[0] == out[1]


def test_sampling_refuses_gpu(dev):
    """What the kernel would read beside its operands is an error ahead of the
    launch: host tensors, other types, vectors of other lengths."""
    from gridllm_amd.ops import hip_ops

    def i64(n):
        return torch.zeros(n, dtype=torch.int64, device=dev)

    def f32(*shape):
        return torch.ones(*shape, device=dev)
    good = (f32(3, 64), i64(3), f32(5), i64(5), i64(5), i64(5))
    assert hip_ops.sample_gumbel_slots(*good).tolist() == [0, 0, 0]
    for at, bad in ((0, good[0].cpu()), (0, good[0].double()),
                    (0, f32(3, 128)[:, ::2]), (1, i64(2)), (1, i64(3).int()),
                    (1, i64(3).cpu()), (2, f32(4)), (3, i64(4)),
                    (4, i64(10)[::2]), (5, f32(5))):
        with pytest.raises(ValueError):
            hip_ops.sample_gumbel_slots(*good[:at], bad, *good[at + 1:])
    for keys, temps in ((i64(2), f32(3)), (i64(3), f32(2)),
                        (i64(3).int(), f32(3)), (i64(3), f32(3).cpu())):
        with pytest.raises(ValueError):
            hip_ops.sample_gumbel(good[0], keys, temps)


@pytest.mark.parametrize("d", [64, 128])
def test_attn_prefill_without_keys(dev, d):
    """Queries that see nothing get nothing."""
    from gridllm_amd.ops import hip_ops
    q, kc, vc = (torch.randn(*s, device=dev).to(torch.bfloat16)
                 for s in ((130, 4, d), (2, 2, 64, d), (2, 2, 64, d)))
    assert not hip_ops.attn_prefill_cache(q, kc, vc, 1, 0, 0, 0.1).any()


@pytest.mark.parametrize("b", [2, 3, 16, 63, 64, 65, 255, 257, 1024])
def test_decode_rows_in_order_gpu(dev, b):
    """Rows by their keys, the longest first and equal ones in the batch's order; no
    order for one row, or for more than are put in one."""
    from gridllm_amd.ops import hip_ops
    g = torch.Generator().manual_seed(b)
    slots = torch.randperm(1500, generator=g)[:b].int()
    slots[b // 2] = slots[0]                  # (a slot may have several rows)
    lens = torch.randint(0, 9 if b % 2 else 4000, (1500,), generator=g).int()
    off = torch.randint(0, 50, (1500,), generator=g).int()
    got = hip_ops.decode_start(lens.to(dev), slots.to(dev), off.to(dev), 4096)
    for a, w in zip(got, R.decode_positions(lens, slots, off, 4096)):
        assert torch.equal(a.cpu(), w)
    n = lens[slots.long()]
    order = torch.sort(n, descending=True, stable=True).indices
    want = torch.stack([order.int(), n[order] + 1, slots[order],
                        n[order] + off[slots[order].long()]], 1)
    assert torch.equal(got[3].cpu(), want)
    want[:, 3] = n[order]
    assert torch.equal(hip_ops.decode_ordered(lens.to(dev), slots.to(dev))[1].cpu(),
                       want)
    many = torch.zeros(1025, dtype=torch.int32, device=dev)
    for few in (many[:1], many):
        assert hip_ops.decode_ordered(lens.to(dev), few)[1] is None


@pytest.mark.parametrize("nsplit", [0, 1, 3])
@pytest.mark.parametrize("hq,hk,d", [(6, 2, 64), (24, 8, 128)])
def test_attn_decode_in_order_gpu(dev, hq, hk, d, nsplit):
    """The order in which rows' blocks start changes no result."""
    from gridllm_amd.ops import hip_ops
    g = torch.Generator(device=dev).manual_seed(hq)
    b, smax = 37, 640
    q, kc, vc = (torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)
                 for s in ((b, hq, d), (b + 3, hk, smax, d), (b + 3, hk, smax, d)))
    slots = torch.randperm(b + 3, generator=g, device=dev)[:b].int()
    lens = torch.randint(0, smax, (b + 3,), generator=g, device=dev).int()
    _, _, seq, rows = hip_ops.decode_start(lens, slots, torch.zeros_like(lens), smax)
    want = hip_ops.attn_decode(q, kc, vc, seq, d ** -0.5, nsplit, slots)
    assert torch.equal(hip_ops.attn_decode(q, kc, vc, seq, d ** -0.5, nsplit, slots,
                                           rows=rows), want)


@pytest.mark.parametrize("nsplit", [0, 1, 5])
@pytest.mark.parametrize("hq,hk,d", [(6, 2, 64), (8, 1, 128), (24, 8, 128)])
@pytest.mark.parametrize("parts,biased,ordered", [
    (0, False, False), (3, False, True), (0, True, True), (3, True, False)])
def test_rope_attn_decode_gpu(dev, hq, hk, d, nsplit, parts, biased, ordered):
    """To the bit what rope_kv and attn_decode give, outputs and caches: one key, the
    edges of steps and splits, shifted positions, and a cache whose place for the new
    key is NaN."""
    from gridllm_amd.ops import hip_ops
    g = torch.Generator(device=dev).manual_seed(hq + parts)
    keys = [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 257, 640]
    b, smax, width = len(keys), 640, (hq + 2 * hk) * d

    def rand(*shape):
        return torch.randn(*shape, generator=g, device=dev)
    kc, vc = (rand(b + 2, hk, smax, d).to(torch.bfloat16) for _ in range(2))
    slots = torch.randperm(b + 2, generator=g, device=dev)[:b].int()
    lens = torch.zeros(b + 2, dtype=torch.int32, device=dev)
    lens[slots.long()] = torch.tensor(keys, dtype=torch.int32, device=dev) - 1
    for s, n in zip(slots.tolist(), keys):
        kc[s, :, n - 1:], vc[s, :, n - 1:] = float("nan"), float("nan")
    off = torch.randint(0, 90, (b + 2,), generator=g, device=dev).int()
    cos, sin = R.rope_tables(d, 800)
    cos, sin = cos.to(dev), sin.to(dev)
    place, pos, seq, rows = hip_ops.decode_start(lens, slots, off, smax)
    qkv = rand(parts, b, width) if parts else rand(b, width).to(torch.bfloat16)
    bias = rand(width).to(torch.bfloat16) if biased else None
    k2, v2 = kc.clone(), vc.clone()
    q = hip_ops.rope_kv(qkv, k2, v2, cos, sin, pos, place, hq, hk, d, bias)
    want = hip_ops.attn_decode(q, k2, v2, seq, d ** -0.5, nsplit, slots)
    got = hip_ops.rope_attn_decode(qkv, kc, vc, cos, sin, pos, place, seq, hq,
                                   d ** -0.5, slots, bias, rows if ordered else None,
                                   nsplit)
    assert want.isfinite().all() and torch.equal(got, want)
    for a, w in ((kc, k2), (vc, v2)):
        assert torch.equal(a.view(torch.int16), w.view(torch.int16))


@pytest.mark.parametrize("nsplit", [1, 5])
@pytest.mark.parametrize("ordered", [False, True])
def test_rope_attn_decode_without_keys_gpu(dev, ordered, nsplit):
    """A row of no keys gives zeros and writes nothing, into its own slot or ahead of
    it; the other rows are as without it."""
    from gridllm_amd.ops import hip_ops
    g = torch.Generator(device=dev).manual_seed(nsplit)
    hq, hk, d, smax, slots = 6, 2, 64, 256, 5

    def rand(*shape):
        return torch.randn(*shape, generator=g, device=dev)
    # (slot 0 is not taken by a row of no keys: there is memory ahead of each)
    kc, vc = (rand(slots, hk, smax, d).to(torch.bfloat16) for _ in range(2))
    slot = torch.tensor([3, 1, 4], dtype=torch.int32, device=dev)
    seq = torch.tensor([70, 0, 1], dtype=torch.int32, device=dev)
    pos = torch.tensor([69, 0, 0], dtype=torch.int32, device=dev)
    rows = torch.stack([torch.arange(3, device=dev, dtype=torch.int32), seq, slot,
                        pos], 1)[[0, 2, 1]].contiguous() if ordered else None
    cos, sin = (t.to(dev) for t in R.rope_tables(d, 128))
    qkv = rand(3, (hq + 2 * hk) * d).to(torch.bfloat16)
    k2, v2 = kc.clone(), vc.clone()
    some = [0, 2]
    place = (slot * smax + seq - 1)[some].contiguous()
    q = hip_ops.rope_kv(qkv[some], k2, v2, cos, sin, pos[some], place, hq, hk, d)
    want = hip_ops.attn_decode(q, k2, v2, seq[some], d ** -0.5, nsplit, slot[some])
    got = hip_ops.rope_attn_decode(qkv, kc, vc, cos, sin, pos, slot * smax + seq - 1,
                                   seq, hq, d ** -0.5, slot, None, rows, nsplit)
    assert torch.equal(got[some], want) and not got[1].any()
    assert torch.equal(kc, k2) and torch.equal(vc, v2)


@pytest.mark.parametrize("name", ["llama3.2:1b", "birepel:3b", "maferax:5b"])
def test_decode_of_fewer_tokens_than_slots_gpu(dev, name):
    """A slot without a token is as if it were not there (but for its length)."""
    from dataclasses import replace
    from gridllm_amd.models import model_class
    from gridllm_amd.models.registry import DenseFF, get_spec
    spec = get_spec(name)
    spec = replace(spec, layers=1 if isinstance(spec.layers, int) else tuple(
        replace(ly, ff=DenseFF(256, 7.0)) for ly in spec.layers[:2]))
    m = model_class(spec)(spec, device=dev, dtype="bf16", kv_slots=6, max_seq=256)
    slots = [m.cache.alloc(0) for _ in range(4)]
    for i, s in enumerate(slots):
        m.forward_prefill(torch.arange(5 + 40 * i, device=dev), s)
    toks = torch.tensor([3, 5, 7], device=dev)
    slot_map = torch.tensor(slots, dtype=torch.int32, device=dev)
    out = []
    kept = [m.cache.seq_lens] + [
        t for name in ("S", "m") for t in getattr(m.cache, name, []) if t is not None]
    were = [t.clone() for t in kept]
    for at in (slot_map[:3].contiguous(), slot_map):
        for t, was in zip(kept, were):
            t.copy_(was)
        if hasattr(m.cache, "prepare_decode"):
            m.cache.prepare_decode(slots)
        out.append(m.forward_decode(toks, at))
    assert torch.equal(*out)


@pytest.mark.parametrize("rows", [32, 64, 96, 128, 160])
@pytest.mark.parametrize("m,n,k,sk", [
    (1, 256, 64, 1),           # a stage, of four or three that are loaded ahead
    (33, 768, 192, 1), (160, 512, 256, 1),
    (95, 1280, 896, 4),        # the last part of K shorter, of fewer stages
    (161, 2304, 4096, 1),      # several blocks of rows, blocks that start further on
    (31, 69888, 128, 1),       # two tiles a block for some, one for others
    (200, 66048, 192, 2),      # up to eight, of unlike parts
    (75, 66048, 64, 1), (76, 66048, 64, 1),    # scores through the caches, and past them
])
def test_gemm_in_256_columns(dev, rows, m, n, k, sk):
    """Results as bf16, as f32 and in parts, at edges of rows, of K's parts and of the
    ring of stages, which runs on from one tile of a block to its next."""
    from gridllm_amd.ops import hip_ops
    g = torch.Generator(device=dev).manual_seed(m + k)
    x = torch.randn(m, k, generator=g, device=dev).to(torch.bfloat16)
    w = torch.randn(n, k, generator=g, device=dev).to(torch.bfloat16)
    ref = x.float() @ w.float().t()
    # bf16 result: 2^-9 of its size; K products' sums: k eps of their sizes' sum
    small = k * 2 ** -24 * (x.float().abs() @ w.float().abs().t()) + 1e-6
    out = torch.full((m, n), 9e9, dtype=torch.bfloat16, device=dev)
    hip_ops.gemm_tile(x, w, rows, 256, sk, out)
    assert bool(((out.float() - ref).abs() <= 2 ** -8 * ref.abs() + small).all())
    if sk == 1:
        assert torch.equal(hip_ops.gemm_tile_f32(x, w, rows, 256), out.float())
    else:
        parts = hip_ops.gemm_tile_parts(x, w, rows, 256, sk)
        assert bool(((parts.sum(0) - ref).abs() <= small).all())


@pytest.mark.parametrize("k", [1 << 20, (1 << 20) + 64])
def test_gemm_tile_of_long_rows(dev, k):
    """The longest rows of 32-bit offsets, and longer ones, which other kernels take for
    the same tilings. Products of -1, 0 and 1: sums of up to 2^24 are exact in any
    order."""
    from gridllm_amd.ops import hip_ops
    g = torch.Generator(device=dev).manual_seed(k)
    m, n = 70, 768
    x, w = (torch.randint(-1, 2, (r, k), generator=g, device=dev,
                          dtype=torch.int8).to(torch.bfloat16) for r in (m, n))
    want = sum(x[:, a:a + 65536].float() @ w[:, a:a + 65536].float().t()
               for a in range(0, k, 65536))
    assert float(want.abs().max()) < 2 ** 24
    for rows, cols, parts in ((32, 64, 1), (32, 96, 5), (64, 128, 3), (32, 256, 1),
                              (96, 256, 2), (96, 64, 1)):
        got = hip_ops.gemm_tile(x, w, rows, cols, parts)
        assert torch.equal(got, want.to(torch.bfloat16)), (rows, cols, parts)
        if parts > 1:
            assert torch.equal(hip_ops.gemm_tile_parts(x, w, rows, cols, parts).sum(0),
                               want)
        else:
            assert torch.equal(hip_ops.gemm_tile_f32(x, w, rows, cols), got.float())
    got = hip_ops.gemm_tile(x, w, 64, 64, 2, fuse_swiglu=True).double()
    gate, up = want.double().view(m, -1, 2, 64).unbind(2)
    ref = (torch.nn.functional.silu(gate) * up).reshape(m, -1)
    assert bool(((got - ref).abs() <= 2 ** -8 * ref.abs() + 1e-6).all())


@pytest.mark.parametrize("glu", [
    (1.0, float("inf"), 0.0, 0.0), (1.702, float("inf"), 0.0, 0.0),
    (1.702, 7.0, 1.0, 0.0),        # each constant alone leaves the short form
    (1.0, 7.0, 0.0, 0.0), (1.0, float("inf"), 1.0, 0.0),
    (1.6, float("inf"), 0.0, 0.044715)])
def test_gated_units_of_all_sizes(dev, glu):
    """Units of gates from 2^-20 to 2^10, both signs: where the exponential
    overflows, where it is nothing, and where an argument is not finite."""
    from gridllm_amd.ops import hip_ops
    from gridllm_amd.ops.reference import Glu
    alpha, limit, shift, cubic = glu
    a = torch.cat([s * 2.0 ** (torch.arange(-80, 40, device=dev) / 4)
                   for s in (1, -1)]).to(torch.bfloat16)
    b = torch.tensor([3.0, -0.37, 0.0, 60.0], device=dev, dtype=torch.bfloat16)
    gates, ups = (x.reshape(1, -1) for x in torch.meshgrid(a, b, indexing="ij"))
    out = hip_ops.swiglu(torch.cat([gates, ups], 1), glu=Glu(*glu)).double()
    g = gates.double().clamp(max=limit)
    u = ups.double().clamp(-limit, limit)
    z = alpha * g * (1 + cubic * g * g)
    ref = g * torch.sigmoid(z) * (u + shift)
    # bf16's half step; z and its multiple of log2 e, rounded, in the exponential;
    # and what f32 keeps of the smallest (2^-126, 1024 * 61 times)
    room = 2 ** -8 + 4 * 2 ** -24 * z.abs().clamp(max=128)
    assert bool(((out - ref).abs() <= room * ref.abs() + 2.0 ** -110).all())
    # a gate that is no number
    odd = torch.ones(1, 16, device=dev, dtype=torch.bfloat16)
    odd[0, 0] = float("nan")
    assert bool(hip_ops.swiglu(odd, glu=Glu(1.702, float("inf"), 0.0, 0.0))[
        0, 0].isnan())
