"""CPU tests of the reference ops (they are the numerics oracle, so they get
their own sanity checks against hand-computed values / torch built-ins)."""

import math

import pytest
import torch

from gridllm_amd.ops import reference as R


def test_rmsnorm_matches_manual():
    torch.manual_seed(0)
    x = torch.randn(4, 64)
    w = torch.randn(64)
    y, _ = R.rmsnorm(x, w, 1e-5)
    expected = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5) * w
    assert torch.allclose(y, expected, atol=1e-5)


def test_rmsnorm_residual_fused():
    torch.manual_seed(1)
    x = torch.randn(3, 32)
    r = torch.randn(3, 32)
    w = torch.ones(32)
    y, res_out = R.rmsnorm(x, w, 1e-6, residual=r)
    z = x + r
    assert torch.allclose(res_out, z, atol=1e-6)
    expected = z * torch.rsqrt(z.pow(2).mean(-1, keepdim=True) + 1e-6)
    assert torch.allclose(y, expected, atol=1e-5)


def test_rope_preserves_norm_and_rotates():
    torch.manual_seed(2)
    t, hq, hk, d = 5, 4, 2, 64
    q = torch.randn(t, hq, d)
    k = torch.randn(t, hk, d)
    cos, sin = R.rope_tables(d, 128)
    pos = torch.arange(t, dtype=torch.int32)
    q2, k2 = R.rope(q.clone(), k.clone(), cos, sin, pos)
    # rotation preserves per-pair norm
    def pair_norms(x):
        half = x.shape[-1] // 2
        return x[..., :half] ** 2 + x[..., half:] ** 2
    assert torch.allclose(pair_norms(q2), pair_norms(q), atol=1e-4)
    # position 0 is identity
    assert torch.allclose(q2[0], q[0], atol=1e-6)
    assert not torch.allclose(q2[1], q[1], atol=1e-3)


def test_swiglu():
    torch.manual_seed(3)
    gu = torch.randn(4, 16)
    out = R.swiglu(gu)
    g, u = gu[..., :8], gu[..., 8:]
    assert torch.allclose(out, torch.nn.functional.silu(g) * u, atol=1e-5)


def test_kv_append_and_decode_attention():
    torch.manual_seed(4)
    b, hk, hq, smax, d = 2, 2, 4, 16, 64
    kc = torch.zeros(b, hk, smax, d)
    vc = torch.zeros(b, hk, smax, d)
    n = 6
    for pos in range(n):
        kn = torch.randn(b, hk, d)
        vn = torch.randn(b, hk, d)
        slot = torch.tensor([i * smax + pos for i in range(b)], dtype=torch.int32)
        R.kv_append(kc, vc, kn, vn, slot)
    q = torch.randn(b, hq, d)
    seqlen = torch.tensor([n, n - 2], dtype=torch.int32)
    scale = 1.0 / math.sqrt(d)
    out = R.attn_decode(q, kc, vc, seqlen, scale)
    # row 0, compare vs direct softmax for head 0 (kv head 0)
    s = (q[0, 0].float() @ kc[0, 0, :n].float().T) * scale
    p = torch.softmax(s, dim=-1)
    expected = p @ vc[0, 0, :n].float()
    assert torch.allclose(out[0, 0], expected, atol=1e-4)


def test_attn_decode_slot_map():
    torch.manual_seed(5)
    hk, hq, smax, d = 2, 4, 8, 64
    kc = torch.randn(3, hk, smax, d)
    vc = torch.randn(3, hk, smax, d)
    q = torch.randn(1, hq, d)
    seqlen = torch.tensor([4], dtype=torch.int32)
    slot_map = torch.tensor([2], dtype=torch.int32)
    out = R.attn_decode(q, kc, vc, seqlen, 0.125, slot_map=slot_map)
    direct = R.attn_decode(q, kc[2:3], vc[2:3], seqlen, 0.125)
    assert torch.allclose(out, direct, atol=1e-6)


def test_attn_prefill_causal_matches_decode_chain():
    """Prefill of T tokens must equal running decode token by token."""
    torch.manual_seed(6)
    t, hq, hk, d, smax = 7, 4, 2, 64, 16
    scale = 1.0 / math.sqrt(d)
    q = torch.randn(1, t, hq, d)
    k = torch.randn(1, t, hk, d)
    v = torch.randn(1, t, hk, d)
    out = R.attn_prefill(q, k, v, scale)
    # last row: decode vs full cache
    kc = torch.zeros(1, hk, smax, d)
    vc = torch.zeros(1, hk, smax, d)
    kc[0, :, :t] = k[0].permute(1, 0, 2)
    vc[0, :, :t] = v[0].permute(1, 0, 2)
    dec = R.attn_decode(q[:, -1], kc, vc, torch.tensor([t], dtype=torch.int32),
                        scale)
    assert torch.allclose(out[0, -1], dec[0], atol=1e-4)


def test_attn_prefill_with_cached_prefix():
    torch.manual_seed(7)
    tpre, tnew, hq, hk, d = 4, 3, 2, 1, 64
    scale = 1.0 / math.sqrt(d)
    k = torch.randn(1, tpre + tnew, hk, d)
    v = torch.randn(1, tpre + tnew, hk, d)
    q = torch.randn(1, tpre + tnew, hq, d)
    full = R.attn_prefill(q, k, v, scale)
    part = R.attn_prefill(q[:, tpre:], k, v, scale, causal_offset=tpre)
    assert torch.allclose(full[:, tpre:], part, atol=1e-5)


def _mat(*shape, dtype=torch.bfloat16):
    return torch.zeros(*shape, dtype=dtype)


@pytest.mark.parametrize("m", [1, 16, 200])
def test_linear_takes_what_fits(m, monkeypatch):
    """Products whose operands F.linear refuses, or reads in a way of its own,
    are left to it."""
    from torch.autograd import forward_ad

    from gridllm_amd.ops import autotune
    ran = []
    monkeypatch.setattr(autotune, "_run", lambda c, x, *rest: ran.append(c))

    def choice(x, w):
        ran.clear()
        autotune.linear_gateup(x, w)
        return ran[0]
    x, w, blas = _mat(m, 256), _mat(512, 256), ("blas",)
    assert choice(x, w) != blas
    for bad in (_mat(m, 192), _mat(m, 320), _mat(m, 256, dtype=torch.float32),
                _mat(m, 256, dtype=torch.float16), _mat(256),
                _mat(m, 2, 256), _mat(m, 512)[:, ::2],
                _mat(m * 256 + 1)[1:].view(m, 256),
                torch.zeros(m, 256, dtype=torch.bfloat16, device="meta")):
        assert choice(bad, w) == blas
    for bad in (_mat(512, 128), _mat(512, 256, dtype=torch.float32),
                _mat(256, 512).t(), _mat(0, 256)):
        assert choice(x, bad) == blas
    assert choice(_mat(m, 0), _mat(512, 0)) == blas
    assert choice(_mat(0, 256), w) == blas
    # the same of sizes that were timed
    monkeypatch.setitem(autotune._CHOICE_GU, (m, 512, 256), ("rows",))
    assert choice(x, w) == ("rows",)
    assert choice(_mat(m, 192), w) == choice(_mat(m, 512)[:, ::2], w) == blas
    seen = []

    def look(a):
        seen.append(choice(a, w))
        return a
    torch.func.vmap(look)(_mat(2, m, 256))
    torch.func.jvp(look, (x,), (x,))
    with forward_ad.dual_level():
        look(forward_ad.make_dual(x, x))
    assert seen == [blas] * 3


def test_embed_norm_by_kernel_or_index(monkeypatch):
    """Indices and layouts that the fused kernel does not read are looked up by
    torch, which takes host indices of a table elsewhere, masks and strides."""
    from gridllm_amd import ops
    from gridllm_amd.ops import hip_ops
    fused = []

    def kernel(tokens, emb, weight, eps):
        fused.append(tokens)
        return emb[tokens], R.rmsnorm(emb[tokens], weight, eps)[0]
    monkeypatch.setattr(ops, "_on_gpu", lambda t: True)
    monkeypatch.setattr(hip_ops, "embed_norm", kernel)
    monkeypatch.setattr(ops, "rmsnorm", R.rmsnorm)
    g = torch.Generator().manual_seed(3)
    emb = torch.randn(10, 64, generator=g).to(torch.bfloat16)
    w, tok = torch.ones(64, dtype=torch.bfloat16), torch.tensor([3, -1, 0])
    off = torch.zeros(10 * 64 + 1, dtype=torch.bfloat16)[1:].view(10, 64)
    off.copy_(emb)
    for t, e, by_kernel in ((tok, emb, True), (tok.int(), emb, True),
                            (tok[[0, 0, 1, 1, 2, 2]][::2], emb, True),
                            (tok, emb.t().contiguous().t(), False),
                            (tok, off, False), (tok.view(3, 1), emb, False),
                            (torch.arange(10) % 3 == 0, emb, False)):
        fused.clear()
        x, y = ops.embed_norm(t, e, w, 1e-5)
        assert bool(fused) == by_kernel
        assert torch.equal(x, emb[t])
        assert torch.equal(y, R.rmsnorm(emb[t], w, 1e-5)[0])
    fused.clear()
    assert ops.embed_norm(tok, emb.to("meta"), w.to("meta"),
                          1e-5)[0].shape == (3, 64) and not fused


def test_embed_norm_refuses():
    from gridllm_amd.ops import hip_ops
    emb, w = _mat(10, 64), _mat(64)
    for tok in (torch.tensor([3]), torch.tensor([3], dtype=torch.int32)):
        with pytest.raises(ValueError):
            hip_ops.embed_norm(tok, emb, w, 1e-5)


def test_decode_positions_refuse():
    """Host tensors, other types and tables of other lengths are an error ahead of
    the launch; so is a step over no slots, rotary positions without their shifts, and
    an order of more rows than are put in one or at an address that is no int4's."""
    from gridllm_amd.ops import hip_ops
    i32 = torch.zeros(4, dtype=torch.int32)
    with pytest.raises(ValueError):
        hip_ops.decode_positions(i32, i32, i32, 64)
    with pytest.raises(ValueError):
        hip_ops.decode_lengths(i32, i32)
    meta = torch.zeros(4, dtype=torch.int32, device="meta")
    for bad in (meta.long(), meta[::2], meta.view(2, 2)):
        with pytest.raises(ValueError):
            hip_ops.decode_lengths(meta, bad)
    if hip_ops.available():
        call, at = hip_ops._load().gl_decode_start, 1 << 20
        assert call(*(None,) * 9, 1, 0, 64) == -100
        assert call(None, at, at, at, at, None, at, None, at, 1, 4, 64) == -100
        for rows, b in ((at, hip_ops._ROWS_ORDERED + 1), (at + 4, 8)):
            assert call(None, at, None, None, None, rows, at, None, at, b, 4, 64) == -100


def test_rope_attn_decode_refuses():
    """Operands by which the kernel would read or write behind others: caches of two
    shapes, fewer lengths, positions or slots than rows, and an order of other rows."""
    from gridllm_amd.ops import hip_ops
    hq, hk, d, b = 4, 2, 64, 3
    qkv, cos = _mat(b, (hq + 2 * hk) * d), torch.zeros(64, d // 2)
    kc, ids = _mat(5, hk, 64, d), torch.zeros(b, dtype=torch.int32)

    def call(vc=kc, pos=ids, seq=ids, slots=ids, rows=None):
        hip_ops.rope_attn_decode(qkv, kc, vc, cos, cos, pos, ids, seq, hq, 1.0, slots,
                                 None, rows)
    order = torch.zeros(b, 4, dtype=torch.int32)
    for bad in (dict(vc=kc[:4]), dict(vc=kc[:, :, :32]), dict(pos=ids[:2]),
                dict(seq=ids[:2]), dict(slots=ids[:2]), dict(seq=ids[0]),
                dict(rows=order[:2]), dict(rows=order[:, :3]),
                dict(rows=order.long()), dict(rows=order.t().contiguous().t())):
        with pytest.raises(ValueError):
            call(**bad)
    with pytest.raises(ValueError):
        hip_ops.attn_decode(_mat(b, hq, d), kc, kc, ids, 1.0, rows=order[:2])
    if hip_ops.available():
        lib = hip_ops._load()
        for tail in ((b, hq, 0, d, 64, 1, 1.0), (b, 0, hk, d, 64, 1, 1.0),
                     (b, hq, hk, d, 64, 3, 1.0)):   # (parts without a workspace)
            assert lib.gl_attn_decode(*(None,) * 9, *tail) == -100
            assert lib.gl_rope_attn_decode(*(None,) * 3, 0, *(None,) * 10,
                                           *tail) == -100


def test_tilings_of_long_rows():
    """Tilings are offered and picked for rows of any length, and the entry takes them
    (as far as it can be asked on the host: a wrong tile is refused ahead of a launch)."""
    from gridllm_amd.ops import hip_ops
    for k in (1 << 20, (1 << 20) + 64, 1 << 24):
        assert hip_ops.gemm_tilings(48, 1024, k) and hip_ops.gemm_tiling(48, 1024, k)
        assert hip_ops.gemm_tiling(200, 1024, k, True)
        if hip_ops.available():
            call = hip_ops._load().gl_gemm_tile
            tail = (32, 48, 0, 1.0, float("inf"), 0.0, 0.0)      # (no such tile)
            assert call(None, 64, None, None, None, 8, 96, k, 1, k, *tail) == -103


def test_decode_splits():
    """Odd numbers, which spread the first parts of all rows over the chip's
    engines; none of less than 128 keys; no more than the combining kernel has."""
    from gridllm_amd.ops.hip_ops import _MAX_SPLIT, decode_splits
    for blocks in range(0, 3100):
        for keys in (0, 1, 128, 129, 300, 513, 100_000):
            parts = decode_splits(blocks, keys)
            assert parts % 2 == 1 and parts <= _MAX_SPLIT
            assert parts == 1 or (parts - 1) * 128 < keys
            assert parts * blocks <= 1536 + blocks
    assert [decode_splits(b, 8192) for b in (8, 24, 192, 256, 512, 768, 1537)
            ] == [31, 15, 9, 7, 3, 3, 1]


def test_sampling_refuses():
    from gridllm_amd.ops import hip_ops
    if not hip_ops.available():
        pytest.skip("the HIP library is not built")
    x, k = torch.zeros(3, 64), torch.zeros(3, dtype=torch.int64)
    with pytest.raises(ValueError):                     # on the host
        hip_ops.sample_gumbel(x, k, torch.ones(3))
    with pytest.raises(ValueError):
        hip_ops.sample_gumbel_slots(x, k, torch.ones(3), k, k, k)
    call = hip_ops._load().gl_sample_gumbel
    assert call(*(None,) * 10, 1, 64, 1, 1) == -100     # neither keys nor slots
    assert call(*(None,) * 6, 1, 1, 1, 1, 1, 64, 1, 0) == -100


def test_tuner_skips_what_cannot_run(monkeypatch):
    """A candidate that fails is left out; the library is always there."""
    from gridllm_amd.ops import autotune
    took = {"blas": 3.0, "rows": 2.0, "tile": 1.0}
    tried = []

    def run(c, x, w, glu=None):
        tried.append(c)
        if c[0] == "tile":
            raise RuntimeError("no such tile")

    def timed(fn, ws, *rest):
        fn(ws[0])
        return took[tried[-1][0]]
    monkeypatch.setattr(autotune, "_run", run)
    monkeypatch.setattr(autotune, "_time_fn", timed)
    x = _mat(4, 256)
    assert autotune._tune(x, 512) == ("rows",)
    assert {c[0] for c in tried} == {"blas", "rows", "tile"}
    took["rows"] = 4.0
    assert autotune._tune(x, 512) == ("blas",)
    # sizes beyond the rules' are looked up once they have been timed
    monkeypatch.setattr(autotune, "_most_rows", 256)
    big, w = _mat(300, 256), _mat(512, 256)
    assert autotune._fit(big, w) is None
    autotune._tune(big, 512)
    assert autotune._fit(big, w) == (300, 512, 256)


def test_products_joined_by_the_next_kernel(monkeypatch):
    """The tuner times those with the norm behind them: each is one of the plain
    products, and not the vocabulary's; the others are timed alone."""
    from types import SimpleNamespace
    from gridllm_amd.models import model_class
    from gridllm_amd.models.registry import get_spec
    from gridllm_amd.ops import autotune
    for name, some in (("tiny", True), ("tiny-birepel", True),
                       ("tiny-vivepel", True), ("tiny-maferax", False)):
        spec = get_spec(name)
        model = model_class(spec)(spec, device="cpu", dtype="fp32", kv_slots=2,
                                  max_seq=64)
        plain, joined = model.gemm_shapes()[0], model.joined_shapes()
        assert joined <= set(plain) and bool(joined) == some
        timed = {}
        monkeypatch.setattr(autotune, "tune_shape", lambda m, n, k, dev, f32, j:
                            timed.update({(n, k): (f32, j)}))
        model.gateup_il = False
        autotune.tune_model_shapes(SimpleNamespace(
            spec=spec, device="cpu", gemm_shapes=lambda: (plain, []),
            joined_shapes=lambda: joined), [4])
        assert {s for s, (_, j) in timed.items() if j} == {
            s for s in joined if s[0] != spec.vocab}
        assert not any(f32 and j for f32, j in timed.values())


def test_scripts_call_what_there_is():
    """Every function that a script takes from the kernel layer is there."""
    import ast
    import pathlib

    from gridllm_amd.ops import autotune, hip_hybrid, hip_ops
    mods = {"hip_ops": hip_ops, "hip_hybrid": hip_hybrid, "autotune": autotune}
    seen = 0
    for path in sorted(pathlib.Path(__file__).parents[1].glob("scripts/*.py")):
        for node in ast.walk(ast.parse(path.read_text())):
            if isinstance(node, ast.Attribute) and \
                    isinstance(node.value, ast.Name) and node.value.id in mods:
                assert hasattr(mods[node.value.id], node.attr), \
                    (path.name, node.attr)
                seen += 1
    assert seen > 5


def test_tilings_by_rule():
    """Each is one that the kernel has; neighbouring sizes of weights are not left
    to another path than those around them; few columns have their K in parts."""
    from gridllm_amd.ops import hip_ops
    from gridllm_amd.ops.autotune import _rule
    for m in (1, 16, 17, 33, 64, 65, 96, 129, 160, 256):
        for n in (64, 128, 192, 896, 1024, 2048, 3072, 4096, 128256):
            for k in (64, 192, 896, 1024, 2048, 4096, 12288):
                for fuse in (False, True):
                    t = hip_ops.gemm_tiling(m, n, k, fuse)
                    if t is None:
                        continue
                    rows, cols, parts = t
                    assert rows in hip_ops._TILE_ROWS and n % cols == 0
                    assert cols in ((64, 128) if fuse else (64, 96, 128))
                    assert 1 <= parts <= max(1, k // 64)
    for fuse in (False, True):
        for m in (129, 160, 256):
            assert all(hip_ops.gemm_tiling(m, n, k, fuse)
                       for n in range(512, 4097, 128)
                       for k in range(512, 4097, 128))
    for m in (96, 160, 256):
        for n, k in ((256, 4096), (1024, 3072), (1024, 4096), (2048, 4096)):
            assert hip_ops.gemm_tiling(m, n, k)[2] > 1
    assert _rule(16, 1024, 6144)[0] == _rule(4, 1024, 8192)[0] == "tile"
    assert _rule(4, 1024, 4096)[0] == "rows"


def test_plans_of_many_rows():
    """Each is one that a kernel takes; gated units are not left to the library
    and another pass; what no kernel has is the library's."""
    from gridllm_amd.ops import hip_ops
    from gridllm_amd.ops.autotune import _rule
    kinds = set()
    for m in (257, 300, 512, 1000, 1200, 1201, 2731, 5000, 8000, 100000):
        for n in (8, 64, 100, 896, 1152, 3072, 5120, 16384, 128256):
            for k in (64, 100, 192, 256, 896, 3072, 4864, 8192):
                for fuse in (False, True):
                    plan = hip_ops.gemm_plan(m, n, k, fuse)
                    kinds.add(plan and plan[0])
                    if plan is None:
                        assert not fuse or n % 128 or k % 64 or k < 256
                        assert _rule(m, n, k, fuse) == ("blas",)
                    elif plan[0] == "tile":
                        rows, cols, parts = plan[1:]
                        assert rows in hip_ops._TILE_ROWS and n % cols == 0
                        assert cols in ((64, 128) if fuse else (64, 96, 128))
                        assert 1 <= parts <= k // 64 and k % 64 == 0
                    else:
                        shape, whole = plan[1:]
                        assert k % 64 == 0 and k >= 256
                        assert n % (128 if fuse else 8) == 0
                        assert shape in ((0, 4) if fuse else (0, 1, 2, 3))
                        rows, cols = hip_ops.WIDE_SHAPES[shape]
                        tiles = -(-m // rows) * -(-n // cols)
                        assert whole == tiles or (shape == 0 and
                                                  whole == tiles // 256 * 256)
    assert kinds == {None, "tile", "wide"}
    for bad in ((0, 256, 256), (300, 0, 256), (300, 256, 0), (-1, 256, 256),
                (1 << 40, 256, 256), (300, 256, 1 << 40)):
        assert hip_ops.gemm_plan(*bad) is None


@pytest.mark.parametrize("m,n,k,fuse,whole,plan", [
    # gated units of 256 x 256 with halves, 112 us, by 192 x 256 122; 125, 144
    (1053, 16384, 3072, True, False, ("wide", 0, 256)),
    (346, 37888, 3584, True, True, ("wide", 0, 256)),
    # 20.7 us, by the library 23.2
    (2159, 2048, 1536, False, False, ("wide", 3, 192)),
    # by the library 61 us, 192 x 128 73; 123, 142; 256 x 256 920, 1034; 414, 424
    # and of 192 x 192 whose last round is three quarters full 99, 91
    (2640, 6144, 3072, False, True, None),
    (1306, 8192, 3072, False, True, None), (2613, 9216, 3072, False, False, None),
    (2405, 8192, 28672, False, False, None), (7440, 12288, 3072, False, True, None),
    # by the library 491 us, 287; 212, 183; 78, by 192 x 128 94
    (2768, 8192, 8192, False, True, ("wide", 0, 256)),
    (4276, 8192, 3072, False, True, ("wide", 2, 731)),
    (2944, 4096, 4096, False, True, None)])
def test_plans_that_were_measured(m, n, k, fuse, whole, plan):
    """One of each kind of size on which the kernels here and the library are on
    different sides."""
    from gridllm_amd.ops import hip_ops
    assert hip_ops.gemm_plan(m, n, k, fuse, whole) == plan


def test_rmsnorm_of_a_residual_needs_a_place_for_the_sum():
    """(refused on the host: the kernel would store to address 0)"""
    from gridllm_amd.ops import hip_ops
    x = torch.zeros(2, 64, dtype=torch.bfloat16)
    lib = hip_ops._load()
    assert lib.gl_rmsnorm(None, x.data_ptr(), x.data_ptr(), x.data_ptr(),
                          x.data_ptr(), None, 2, 64, 1e-5) == -100


def test_rope_kv_refuses():
    """Rows of other types, and a bias of another type, size or stride, ahead of
    the launch."""
    from gridllm_amd.ops import hip_ops
    bf16 = torch.bfloat16
    kc = torch.zeros(1, 1, 8, 16, dtype=bf16)
    cos, sin = R.rope_tables(16, 8)
    at = torch.zeros(2, dtype=torch.int32)

    def call(rows, bias=None):
        hip_ops.rope_kv(rows, kc, kc, cos, sin, at, at, 2, 1, 16, bias)
    rows = torch.zeros(2, 64, dtype=bf16)
    for bad in (rows.float(), rows.half(), rows.expand(3, 2, 64)):
        with pytest.raises(ValueError):
            call(bad)
    for bias in (torch.zeros(64), torch.zeros(32, dtype=bf16),
                 torch.zeros(128, dtype=bf16)[::2]):
        with pytest.raises(ValueError):
            call(rows, bias)


def test_rope_kv_takes_any_bias_of_its_size(monkeypatch):
    """A bias that is a view at any place or stride reaches the kernel dense and
    aligned."""
    from gridllm_amd import ops
    from gridllm_amd.ops import hip_ops
    bf16, got = torch.bfloat16, []
    monkeypatch.setattr(ops, "_on_gpu", lambda t: True)
    monkeypatch.setattr(hip_ops, "rope_kv", lambda *a: got.append(a[-1]))
    want = torch.arange(64).to(bf16)
    flat, wide = torch.zeros(65, dtype=bf16), torch.zeros(64, 2, dtype=bf16)
    flat[1:], wide[:, 0] = want, want
    for bias in (want, flat[1:], wide[:, 0]):
        ops.rope_kv(torch.zeros(2, 64, dtype=bf16), *(None,) * 6, 2, 1, 16, bias)
        assert torch.equal(got[-1], want) and got[-1].is_contiguous()
        assert got[-1].data_ptr() % 16 == 0
    assert got[0] is want
    ops.rope_kv(torch.zeros(2, 64, dtype=bf16), *(None,) * 6, 2, 1, 16)
    assert got[-1] is None


def test_rope_attn_decode_takes_any_bias_of_its_size(monkeypatch):
    """As rope_kv does, in whose place it stands in a decode step."""
    from gridllm_amd import ops
    from gridllm_amd.ops import hip_ops
    bf16, got = torch.bfloat16, []
    monkeypatch.setattr(ops, "_on_gpu", lambda t: True)
    monkeypatch.setattr(hip_ops, "rope_attn_decode", lambda *a: got.append(a[-2]))
    want, rows = torch.arange(64).to(bf16), torch.zeros(2, 64, dtype=bf16)
    flat, wide = torch.zeros(65, dtype=bf16), torch.zeros(64, 2, dtype=bf16)
    flat[1:], wide[:, 0] = want, want
    slots = torch.zeros(2, dtype=torch.int32)
    for bias in (want, flat[1:], wide[:, 0], None):
        ops.rope_attn_decode(rows, *(None,) * 7, 2, 1.0, slots, bias)
    assert got[0] is want and got.pop() is None
    for b in got:
        assert torch.equal(b, want) and b.is_contiguous() and b.data_ptr() % 16 == 0


def test_plans_of_whole_products():
    """None is in parts of K, or by the kernel of which parts are."""
    from gridllm_amd.ops import hip_ops
    for m in (257, 300, 1200, 1201, 5000):
        for n in (896, 3072, 16384):
            for k in (896, 3072, 8192):
                for fuse in (False, True):
                    plan = hip_ops.gemm_plan(m, n, k, fuse, True)
                    assert plan is None or plan[0] == "wide"
                    assert plan is not None or not fuse


def test_scores_of_many_rows_by_shapes_that_have_them(monkeypatch):
    """A vocabulary's scores (f32) of more than 256 rows take no shape of tiles that
    has bf16 results alone, nor does a product in bf16 take one of theirs; by rule,
    and where the same sizes were timed as the other."""
    from gridllm_amd.ops import autotune, hip_ops

    class OnGpu(torch.Tensor):
        is_cuda = True
    ran = []

    def wide(x, w, shape, whole, fuse_swiglu=False, glu=None, f32=False):
        assert shape in ((0, 4) if f32 or fuse_swiglu else (0, 1, 2, 3))
        ran.append(("wide", f32))

    def others(c, x, w, glu=None):
        ran.append(c[:1])
        return wide(x, w, *c[1:]) if c[0] == "wide" else x
    monkeypatch.setattr(hip_ops, "gemm_wide", wide)
    monkeypatch.setattr(hip_ops, "gemm_tile_f32", lambda x, w, *c: ran.append("f32"))
    monkeypatch.setattr(autotune, "_run", others)
    for n, k in ((32000, 2048), (32064, 3072), (1024, 896), (128256, 2048)):
        w = torch.empty(n, k, dtype=torch.bfloat16)
        for m in (*range(257, 600, 9), 1201, 2000, 4096):
            x = torch.empty(m, k, dtype=torch.bfloat16).as_subclass(OnGpu)
            autotune.linear_f32(x, w)
            autotune.linear(x, w)
    assert ("wide", True) in ran and ("wide", False) in ran
    m, n, k = 350, 32000, 2048
    x = torch.empty(m, k, dtype=torch.bfloat16).as_subclass(OnGpu)
    w = torch.empty(n, k, dtype=torch.bfloat16)
    for f32, choice in ((True, ("wide", 4, 250)), (False, ("wide", 3, 500))):
        monkeypatch.setattr(autotune, "_tune", lambda *a, **kw: choice)
        assert autotune.tune_shape(m, n, k, "cpu", f32) == choice
    try:
        autotune.linear_f32(x, w)
        autotune.linear(x, w)
    finally:
        for table in (autotune._CHOICE, autotune._CHOICE_F32):
            table.pop((m, n, k), None)


def test_whole_products_of_sizes_that_were_timed(monkeypatch):
    """More than 256 rows whose sums over K are to stay whole do not take a choice
    with K in parts that a decode batch of as many rows was timed with."""
    from gridllm_amd.ops import autotune, hip_ops

    class OnGpu(torch.Tensor):
        is_cuda = True
    ran = []
    monkeypatch.setattr(autotune, "_run", lambda c, x, *rest: ran.append(c))
    monkeypatch.setattr(hip_ops, "gemm_tile_parts",
                        lambda x, w, *c: ran.append(("tile", *c)))
    n, k, cut = 3072, 8192, ("tile", 128, 128, 2)
    w = torch.empty(n, k, dtype=torch.bfloat16)
    for m, timed in ((512, cut), (512, ("ours", 2)), (512, ("blas",)),
                     (512, ("wide", 1, 48)), (256, cut)):
        x = torch.empty(m, k, dtype=torch.bfloat16).as_subclass(OnGpu)
        monkeypatch.setitem(autotune._CHOICE, (m, n, k), timed)
        monkeypatch.setitem(autotune._CHOICE_GU, (m, n, k), timed)
        for run in (autotune.linear, autotune.linear_parts,
                    lambda x, w, whole=False: autotune.linear_gateup(
                        x, w, whole=whole)):
            ran.clear()
            run(x, w)
            run(x, w, whole=True)
            assert ran[0] == timed
            assert ran[1] == timed if m == 256 or timed[0] in ("blas", "wide") \
                else ran[1][0] in ("blas", "wide")


def test_joined_choices_are_their_own(monkeypatch):
    """What was timed with the norm behind it, which adds up parts of K, is not what
    a product alone runs by, nor the other way round."""
    from gridllm_amd import ops
    from gridllm_amd.ops import autotune, hip_ops

    class OnGpu(torch.Tensor):
        is_cuda = True
    ran = []
    monkeypatch.setattr(autotune, "_run", lambda c, x, *rest: ran.append(c))
    monkeypatch.setattr(hip_ops, "gemm_tile_parts",
                        lambda x, w, *c: ran.append(("tile", *c)))
    monkeypatch.setattr(hip_ops, "gemm_tile_rmsnorm",
                        lambda x, w, *c: ran.append(("tile", *c[:3])))
    monkeypatch.setattr(ops, "rmsnorm", lambda *a, **kw: None)
    m, n, k = 24, 3072, 8192
    x = torch.empty(m, k, dtype=torch.bfloat16).as_subclass(OnGpu)
    w = torch.empty(n, k, dtype=torch.bfloat16)
    norm, resid = (torch.zeros(*s, dtype=torch.bfloat16) for s in ((n,), (m, n)))
    cut, alone = ("tile", 32, 64, 16), ("tile", 32, 64, 2)

    def both():
        ran.clear()
        autotune.linear(x, w)
        autotune.linear_parts(x, w)
        autotune.linear_rmsnorm(x, w, norm, 1e-5, resid)
        return [*ran, autotune.choice_of(m, w)]
    rule = both()[0]
    for order in ((True, False), (False, True)):
        with monkeypatch.context() as mp:
            for table in ("_CHOICE", "_CHOICE_JOINED"):
                mp.setattr(autotune, table, {}, raising=False)
            mp.setattr(autotune, "_tune", lambda x, n, f32, joined:
                       cut if joined else alone)
            autotune.tune_shape(m, n, k, "cpu", False, order[0])
            # of one kind alone: joined ones still take what was timed alone
            assert both() == ([rule, cut, cut, cut] if order[0] else [alone] * 4)
            autotune.tune_shape(m, n, k, "cpu", False, order[1])
            assert both() == [alone, cut, cut, cut]


@pytest.mark.parametrize("n,k", [(64, 64), (3072, 3072), (128256, 3072)])
def test_timings_fit_beside_a_full_cache(n, k):
    """An engine whose KV cache leaves little memory starts: the tuner takes no more
    than 24 copies of a weight, in 640 MB, or the two that it cannot do without."""
    from gridllm_amd.ops import autotune
    size = n * k * 2
    for room in (0, 1 << 30, (4 << 30) - 1):
        few = autotune._copies(size, room)
        assert few >= 2 and few <= 24 and (few == 2 or few * size <= 640 << 20)
    for room in (4 << 30, float("inf")):
        copies = autotune._copies(size, room)
        assert copies >= few and (copies == 2 or copies * size <= 2 << 30)


def test_tuner_asks_more_of_what_goes_through_the_cache(monkeypatch):
    """Tiles of several blocks of rows read weights through the Infinity Cache, but for
    few weights in short parts, and are taken if they are 5 % faster than one block's."""
    from gridllm_amd.ops import autotune, hip_ops
    once = hip_ops.gemm_tile_once
    assert once(96, 3072, 8192, 96, 1) and once(256, 128256, 3072, 256, 1)
    assert not once(97, 3072, 8192, 96, 1) and not once(90, 5120, 3072, 32, 4)
    assert once(48, 2048, 2048, 32, 4) and once(90, 1536, 1536, 32, 3)
    assert not once(48, 896, 4864, 32, 1) and not once(128, 2048, 2048, 32, 4)
    rows, ran = 96, []
    monkeypatch.setattr(hip_ops, "gemm_tilings", lambda *a: [(96, 64, 5), (64, 64, 5)])
    monkeypatch.setattr(hip_ops, "gemm_rows_supported", lambda *a: False)
    monkeypatch.setattr(autotune, "_weights", lambda *a: [None, None])
    monkeypatch.setattr(autotune, "_run", lambda c, *rest: ran.append(c))
    monkeypatch.setattr(autotune, "_most_rows", autotune._most_rows)

    def timed(fn, ws, *rest):
        fn(ws[0])
        return {"blas": 20.0, 96: 10.0, 64: cut}[ran[-1][1] if len(ran[-1]) > 1
                                                 else "blas"]
    monkeypatch.setattr(autotune, "_time_fn", timed)
    x = _mat(rows, 8960)
    for cut, best in ((9.6, 96), (9.2, 64)):
        assert autotune._tune(x, 1536)[1] == best


def test_plans_times_are_the_tilings():
    """What gl_gemm_plan says of a tiling's time is what _tile_us says: of the
    tilings that it looks at, the one it names takes the least by both."""
    from gridllm_amd.ops import hip_ops
    seen = 0
    for m in (257, 300, 384, 512, 700, 1000, 1200):
        for n in (64, 896, 1024, 1152, 2048, 3072):
            for k in (4096, 4864, 6144, 8192, 12288):
                plan = hip_ops.gemm_plan(m, n, k)
                if plan is None or plan[0] != "tile":
                    continue

                def us(rows, cols, parts):
                    return hip_ops._tile_us(m, n, k, rows, cols,
                                            -(-m // rows) * (n // cols), parts)
                least = float("inf")
                for rows in (96, 128, 160, 192, 256):
                    for cols in (64, 96, 128):
                        tiles = -(-m // rows) * (n // cols)
                        if n % cols or tiles > 512:
                            continue
                        most = max(1, min(256 // tiles, k // 384))
                        for parts in (1, (most + 1) // 2, most):
                            least = min(least, us(rows, cols, parts))
                # (the plan's sums are of 24 bits)
                assert abs(us(*plan[1:]) - least) < 1e-5 * least, (m, n, k)
                seen += 1
    assert seen > 50


@pytest.mark.parametrize("heads", [1, 3, 7, 8, 9, 14, 24, 33])
def test_prefill_blocks_have_each_tile_once(heads):
    """Blocks of prompt attention, by XCD: an eighth of the heads' tiles each, that of
    heads which follow each other, later tiles first."""
    import ctypes
    from gridllm_amd.ops import hip_ops
    call, place = hip_ops._load().gl_prefill_place, (ctypes.c_int * 2)()
    for tiles in (1, 2, 3, 5, 8, 31, 63):
        per = -(-tiles * heads // 8)
        seen = set()
        for xcd in range(8):
            last = tiles
            for at in range(per):
                if call(at * 8 + xcd, tiles, heads, place):
                    break
                tile, head = place
                assert 0 <= tile <= last
                last = tile
                # (head by head, later tiles first, it would be the same eighth)
                assert (head * tiles + tiles - 1 - tile) // per == xcd
                seen.add((tile, head))
        assert len(seen) == tiles * heads
