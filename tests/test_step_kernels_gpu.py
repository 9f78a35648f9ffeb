"""Work splits of the kernels around the projections and the attention, at the sizes
where a split can go wrong, against the plain references (ops/ref.py)."""
import pytest
import torch

from llm_mcp_amd import ops
from llm_mcp_amd.ops import encoder, mixers, ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(autouse=True)
def _native():
    ops.native()
    torch.manual_seed(0)


def _i32(x):
    return torch.as_tensor(x, dtype=torch.int32, device=DEV)


def _slots(T, NB):
    """A run from the middle of a page, a jump, a hole, a run that ends in a quad."""
    s = torch.cat([torch.arange(45, 45 + T // 2), torch.arange(NB * 16, NB * 16 + T - T // 2)])
    if T > 5:
        s[5] = -1
    return s.to(torch.int32)


# ------------------------------------------------- rotation and cache write --
@pytest.mark.parametrize("Hq,Hkv,D", [(5, 3, 16), (3, 2, 48), (9, 7, 64), (7, 5, 80), (32, 8, 128),
                                      (3, 3, 256)])
@pytest.mark.parametrize("T,skip_q", [(1, False), (31, True), (33, False), (96, True), (97, False)])
def test_rope_head_groups(Hq, Hkv, D, T, skip_q):
    """Head groups that do not divide the heads, one token over a tile."""
    NB = 10
    qkv = torch.randn(T, (Hq + 2 * Hkv) * D, device=DEV).bfloat16()
    pos, slots = _i32(torch.randint(0, 500, (T,))), _slots(T, NB).to(DEV)
    cs = ref.rope_cos_sin(512, D, 10000.0, DEV)
    kc = torch.zeros(NB, Hkv, 32, D, device=DEV, dtype=torch.bfloat16)
    vc = torch.zeros(NB, Hkv, 8, D, 4, device=DEV, dtype=torch.bfloat16)
    want, k0, v0 = qkv.cpu(), kc.cpu(), vc.cpu()
    ref.rope_cache(want, pos.cpu(), cs.cpu(), Hq, Hkv, D, slots.cpu(), k0, v0, False)
    if skip_q:
        want = qkv.cpu()
    ops.rope_and_cache(qkv, pos, cs, Hq, Hkv, D, slots, kc, vc, skip_q=skip_q)
    # two products and a sum in fp32, rounded to bf16 once: 2^-8 of the pair's length
    torch.testing.assert_close(qkv[:, :Hq * D].float().cpu(), want[:, :Hq * D].float(), atol=2e-2,
                               rtol=1e-2)
    torch.testing.assert_close(kc.float().cpu(), k0.float(), atol=2e-2, rtol=1e-2)
    assert torch.equal(vc.cpu(), v0)


@pytest.mark.parametrize("H,D", [(16, 64), (3, 128), (5, 48), (2, 256), (1, 8), (3, 20)])
@pytest.mark.parametrize("T", [1, 31, 32, 65])
@pytest.mark.parametrize("shift", [0, 1])
def test_kv_write(H, D, T, shift):
    """Few tokens, a workgroup each: aligned rows and rows that no 16-byte load reads."""
    NB = 6
    kv = torch.randn(T, 2 * H * D + 8, device=DEV).bfloat16()
    k = kv[:, shift:shift + H * D].view(T, H, D)
    v = kv[:, shift + H * D:shift + 2 * H * D].view(T, H, D)
    slots = _slots(T, NB).to(DEV)
    kc = torch.zeros(NB, H, 32, D, device=DEV, dtype=torch.bfloat16)
    vc = torch.zeros(NB, H, 8, D, 4, device=DEV, dtype=torch.bfloat16)
    k0, v0 = kc.cpu(), vc.cpu()
    ref.write_cache(k.cpu(), v.cpu(), slots.cpu(), k0, v0)
    ops.kv_write(k, v, slots, kc, vc)
    assert torch.equal(kc.cpu(), k0) and torch.equal(vc.cpu(), v0)


@pytest.mark.parametrize("H,D", [(16, 64), (3, 128), (5, 48), (2, 256), (1, 8), (3, 20)])
@pytest.mark.parametrize("T", [1601, 4096, 4097, 4127])
@pytest.mark.parametrize("shift", [0, 1])
def test_kv_write_of_many_tokens(H, D, T, shift):
    """Both sides of the line between a workgroup a token and 32-token tiles: tiles of 1, 31 and 32
    tokens, head groups that do not divide the heads, rows that no 16-byte load reads."""
    NB = T // 32 + 8
    kv = torch.randn(T, 2 * H * D + 8, device=DEV).bfloat16()
    k = kv[:, shift:shift + H * D].view(T, H, D)
    v = kv[:, shift + H * D:shift + 2 * H * D].view(T, H, D)
    slots = _slots(T, NB).to(DEV)
    kc = torch.zeros(NB, H, 32, D, device=DEV, dtype=torch.bfloat16)
    vc = torch.zeros(NB, H, 8, D, 4, device=DEV, dtype=torch.bfloat16)
    k0, v0 = kc.cpu(), vc.cpu()
    ref.write_cache(k.cpu(), v.cpu(), slots.cpu(), k0, v0)
    ops.kv_write(k, v, slots, kc, vc)
    assert torch.equal(kc.cpu(), k0) and torch.equal(vc.cpu(), v0)


# -------------------------------------------------------------- convolution --
@pytest.mark.parametrize("C", [40, 2056])
@pytest.mark.parametrize("taps", [2, 4, 9, 10, 32])
def test_conv_parts(C, taps):
    """Rows cut into parts: lengths around a part and a tile, fresh and continued
    sequences, more taps than the smallest part has tokens."""
    lens, old = [1, 7, 8, 9, 63, 64, 65, 130], [0, 3, 0, 70, 2, 0, 1, 200]
    S, T = len(lens), sum(lens)
    cu = torch.tensor([0] + lens).cumsum(0)
    ctx = torch.tensor(lens) + torch.tensor(old)
    slots = torch.randperm(S)
    u = torch.randn(T, C).bfloat16()
    w, bias = torch.randn(taps, C) * taps ** -0.5, torch.randn(C)
    state = torch.randn(S, taps - 1, C).bfloat16()
    st = state.to(DEV)
    y = ops.short_conv(u.to(DEV), w.to(DEV), st, _i32(cu), _i32(ctx), _i32(slots), bias=bias.to(DEV),
                       silu=True, tiles=_i32(mixers.conv_tiles(cu)))
    want = torch.empty(T, C)
    ref.short_conv(u, w, bias, state, cu, ctx, slots, want, True)
    torch.testing.assert_close(y.float().cpu(), want, atol=2e-2, rtol=1e-2)
    assert torch.equal(st.cpu(), state)


# ----------------------------------------------------------------- encoders --
def _values():
    """bf16 numbers over the range where gelu is neither 0 nor its argument, and far out."""
    v = torch.cat([torch.linspace(-14, 14, 3800), torch.logspace(-38, 38, 148),
                   -torch.logspace(-38, 38, 148)])
    return v.bfloat16()


@pytest.mark.parametrize("kernel", ["pgemm", "dgemm"])
def test_gelu_erf_epilogue(kernel):
    """gelu of given values (a product with a unit vector): the correctly rounded result
    or its neighbour -- at most 2.5e-6 of the value off before the rounding."""
    v, K = _values(), 256
    N = v.numel() // 256 * 256
    w = torch.zeros(N, K, dtype=torch.bfloat16)
    w[:, 3] = v[:N]
    a = torch.zeros(3, K, dtype=torch.bfloat16)
    a[:, 3] = 1
    a, w, b = a.to(DEV), w.to(DEV), torch.zeros(N, device=DEV, dtype=torch.bfloat16)
    if kernel == "pgemm":
        y = ops.pgemm(a, w, bias=b, act=ops.ACT_GELU_ERF)
    else:
        y = torch.empty(3, N, device=DEV, dtype=torch.bfloat16)
        ops.native().dgemm(y.data_ptr(), a.data_ptr(), w.data_ptr(), 0, 0, 0, 3, N, K, K, K, N, 31, 1,
                           6, torch.cuda.current_stream().cuda_stream, b.data_ptr())
    x = v[:N].double()
    want = torch.where(x < 0, 0.5 * x * torch.special.erfc(-x / 2 ** 0.5),
                       x - 0.5 * x * torch.special.erfc(x / 2 ** 0.5)).to(DEV)
    # half a unit in the last place and the 2.5e-6; below 2^-126 results flush to zero (z over 13)
    err = (y.double() - want).abs()
    assert bool((err <= want.abs() * (2.0 ** -8 + 3e-6) + 2.0 ** -125).all())


@pytest.mark.parametrize("cfg", [21, 31, 20, 22, 11])
@pytest.mark.parametrize("M", [1, 63, 64, 129, 300])
def test_dgemm_bias_epilogues(cfg, M):
    """Every tile of the encoders' rule: + bias, gelu(+ bias), edges of row tiles."""
    N, K = 512, 256
    a, w, b = (torch.randn(M, K, device=DEV).bfloat16(), torch.randn(N, K, device=DEV).bfloat16() * 0.1,
               torch.randn(N, device=DEV).bfloat16())
    z = a.float() @ w.float().t() + b.float()
    for epi, want in ((5, z), (6, torch.nn.functional.gelu(z))):
        y = torch.full((M, N), 7.0, device=DEV).bfloat16()
        ops.native().dgemm(y.data_ptr(), a.data_ptr(), w.data_ptr(), 0, 0, 0, M, N, K, K, K, N, cfg, 1,
                           epi, torch.cuda.current_stream().cuda_stream, b.data_ptr())
        # one bf16 rounding of an fp32 sum of 256 products
        torch.testing.assert_close(y.float(), want, atol=2e-3, rtol=2.0 ** -8)


@pytest.mark.parametrize("S", [1, 2, 3, 4, 6, 8, 12, 16])
@pytest.mark.parametrize("rows,cols,bias", [(1, 768, True), (17, 1024, False), (5, 2048, True),
                                            (3, 264, True)])
def test_layernorm_slabs(S, rows, cols, bias):
    p = torch.randn(S, rows, cols, device=DEV)
    r, w, b, c = (torch.randn(*s, device=DEV).bfloat16()
                  for s in ((rows, cols), (cols,), (cols,), (cols,)))
    y = torch.empty_like(r)
    ops.native().layernorm_slabs(y.data_ptr(), p.data_ptr(), S, rows * cols,
                                 c.data_ptr() if bias else 0, r.data_ptr(), w.data_ptr(), b.data_ptr(),
                                 rows, cols, 1e-12, torch.cuda.current_stream().cuda_stream)
    o = (p.double().sum(0) + (c.double() if bias else 0)).bfloat16()
    x = (o.float() + r.float()).bfloat16().double()
    want = torch.nn.functional.layer_norm(x, (cols,), w.double(), b.double(), 1e-12)
    # bf16 results; a sum on the edge of a rounding may fall to the other side (2^-8 of |x| to 8,
    # times 1 / sigma < 1 and a gain to 4) in one element of a thousand
    far = (y.double() - want).abs() > 1e-4 + 2.0 ** -8 * want.abs()
    assert float(far.double().mean()) < 2e-3
    torch.testing.assert_close(y.double(), want, atol=0.15, rtol=2.0 ** -8)


def test_embed_norm():
    from llm_mcp_amd.ops import encoder
    word, typ, pos = (torch.randn(s, 768, device=DEV).bfloat16() for s in (50, 2, 40))
    w, b = torch.randn(768, device=DEV).bfloat16(), torch.randn(768, device=DEV).bfloat16()
    ids, at = _i32([0, 49, 7, 50, -1]), _i32([0, 39, 3, 1, 2])       # two outside the table
    for p in (None, pos):
        y = encoder.embed_norm(ids, word, typ, w, b, 1e-12, p, at)
        x = torch.stack([word[i].float() if 0 <= i < 50 else torch.zeros(768, device=DEV)
                         for i in ids.tolist()])
        t = typ[0].float() if p is None else (pos[at.long()].float() + typ[0].float()).bfloat16().float()
        x = (x + t).bfloat16().double()
        want = torch.nn.functional.layer_norm(x, (768,), w.double(), b.double(), 1e-12)
        torch.testing.assert_close(y.double(), want, atol=1e-4, rtol=2.0 ** -8)


@pytest.mark.parametrize("model", ["nomic-embed-text", "mxbai-embed-large"])
def test_encoder_batches_agree(model):
    """One document alone, in a small batch and in a large one: other tiles, slices and
    kernels, the same vector to bf16 accuracy; and the models' own loop over single ops."""
    import dataclasses

    from llm_mcp_amd.models import config as mc
    from llm_mcp_amd.models.bert import BertModel
    from llm_mcp_amd.models.nomic_bert import NomicBertModel
    cfg = dataclasses.replace(mc.resolve(model), num_layers=2)
    m = (NomicBertModel if model.startswith("nomic") else BertModel)(cfg, "cuda", seed=2)
    g = torch.Generator().manual_seed(0)
    docs = [torch.randint(0, 30000, (n,), generator=g, dtype=torch.int32)
            for n in [1, 5, 16, 33] + [500] * 24]

    def run(which):
        lens = [len(docs[i]) for i in which]
        cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
        return m.forward(torch.cat([docs[i] for i in which]).to(DEV), cu.to(DEV), lens)

    whole = run(range(len(docs)))
    small = run([3, 0, 2, 1])
    from llm_mcp_amd.ops import encoder
    keep, encoder.layers_ok = encoder.layers_ok, lambda *a: False
    try:
        loop = run(range(len(docs)))
    finally:
        encoder.layers_ok = keep
    cos = torch.nn.functional.cosine_similarity
    assert float(cos(whole[:4], torch.stack([small[1], small[3], small[2], small[0]])).min()) > 0.9995
    assert float(cos(whole[4:5], run([4])).min()) > 0.9995
    assert float(cos(whole, loop).min()) > 0.9995


# ----------------------------------------------------- products left to a norm --
@pytest.mark.parametrize("N,K", [(4096, 4096), (4096, 14336)])
def test_two_deferred_products_keep_their_slabs(N, K):
    """Two products of one shape whose K reduction waits for the same norm: each has slabs
    of its own."""
    x, y = (torch.randn(4, K, device=DEV).bfloat16() for _ in range(2))
    w = torch.randn(N, K, device=DEV).bfloat16() * K ** -0.5
    a, b = ops.linear(x, w, defer=True), ops.linear(y, w, defer=True)
    assert isinstance(a, ops.Partials) and isinstance(b, ops.Partials)
    for p, r in ((a, x), (b, y)):
        torch.testing.assert_close(p.sum().double(), r.double() @ w.double().t(), atol=1e-4, rtol=1e-4)


# ------------------------------------------------- K23: few rows, small weights --
@pytest.mark.parametrize("M", [1, 15, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(32, 32), (96, 64), (768, 800), (8224, 96), (160, 2080)])
def test_sgemm(M, N, K):
    """Every epilogue: row tiles, one and two column tiles per workgroup, fewer K steps
    than waves, strided rows."""
    a = torch.randn(M, K + 8, device=DEV).bfloat16()[:, :K]
    w = torch.randn(N, K, device=DEV).bfloat16() * K ** -0.5
    b = torch.randn(N, device=DEV).bfloat16()
    y = a.double() @ w.double().t()
    # fp32 sums of K products of bf16 numbers of order one; one rounding to bf16
    tol = dict(atol=2e-3, rtol=2.0 ** -8)
    torch.testing.assert_close(ops.sgemm(a, w).double(), y, **tol)
    torch.testing.assert_close(ops.sgemm(a, w, bias=b).double(), y + b.double(), **tol)
    g, u = y.view(M, N // 32, 2, 16).unbind(2)
    for epi, f in ((3, torch.nn.functional.silu), (4, torch.relu)):
        torch.testing.assert_close(ops.sgemm(a, w, epi).double(), (f(g) * u).reshape(M, -1), **tol)
    for s in (1, 2, 4):
        if K // 32 % s == 0:
            p = ops.sgemm(a, w, 2, s)
            assert tuple(p.slabs.shape) == (s, M, N)
            torch.testing.assert_close(p.slabs.double().sum(0), y, atol=2e-5, rtol=2e-5)


@pytest.mark.parametrize("M", [2, 3, 8, 9, 32, 33])
def test_linear_of_few_rows(M):
    """The rule of ops.linear: both sides of its lines, with bias, deferred, strided rows."""
    for N, K in ((2048, 2048), (4096, 4096)):
        x = torch.randn(M, K + 8, device=DEV).bfloat16()
        w, b = torch.randn(N, K, device=DEV).bfloat16() * K ** -0.5, torch.randn(N, device=DEV).bfloat16()
        y = x[:, :K].double() @ w.double().t()
        for xs in (x[:, :K], x[:, :K].contiguous()):
            n = ops.SGEMM_CALLS[0]
            got = ops.linear(xs, w, defer=True)
            got = got.sum() if isinstance(got, ops.Partials) else got
            torch.testing.assert_close(got.double(), y, atol=2e-2, rtol=1e-2)
            assert ops.SGEMM_CALLS[0] - n == int(2 < M <= (32 if N == 2048 else 8))
            torch.testing.assert_close(ops.linear(xs, w, bias=b).double(), y + b.double(), atol=2e-2,
                                       rtol=1e-2)


# --------------------------------------------- K13: the last round in pieces --
def _k13(M, N, K, **kw):
    a = torch.randn(M, K, device=DEV).bfloat16()
    w = torch.randn(N, K, device=DEV).bfloat16() * K ** -0.5
    return a, w


@pytest.mark.parametrize("M,N,K,cut", [
    (2048, 4096, 4096, True),      # half a round: two pieces a tile, one a workgroup
    (2300, 4096, 14336, True),     # 144 tiles: pieces that end inside tiles, ragged rows
    (257, 512, 6144, True),        # four tiles of four pieces each
    (100, 256, 8192, True),        # one tile
    (6500, 3328, 4160, True),      # a whole round, then 82 tiles
    (7000, 4864, 832, False),      # 532 tiles: 20 of 13 steps
    (2048, 8192, 512, False)])     # one round, whole
def test_k13_last_round(M, N, K, cut):
    """Every form of the epilogue on row-major W where the last round of tiles is cut along K: the
    numbers of a product in fp32, the same bits each time, nothing left in the counters."""
    assert (ops.native().pgemm_tail_floats(M, N, K) > 0) == cut
    a, w = _k13(M, N, K)
    z = a.float() @ w.float().t()
    tol = dict(atol=4e-3, rtol=2.0 ** -7)
    y = ops.pgemm(a, w)
    torch.testing.assert_close(y.float(), z, **tol)
    for _ in range(3):
        assert torch.equal(ops.pgemm(a, w), y)
    b = torch.randn(N, device=DEV).bfloat16()
    torch.testing.assert_close(ops.pgemm(a, w, bias=b).float(), z + b.float(), **tol)
    torch.testing.assert_close(ops.pgemm(a, w, bias=b, act=ops.ACT_GELU_ERF).float(),
                               torch.nn.functional.gelu(z + b.float()), **tol)
    g, u = z.view(M, N // 32, 2, 16).unbind(2)
    torch.testing.assert_close(ops.pgemm(a, w, act=ops.ACT_SWIGLU).float(),
                               (torch.nn.functional.silu(g) * u).reshape(M, -1), **tol)
    r = torch.randn(M, N, device=DEV).bfloat16()
    want = (r.float() + z.bfloat16().float())
    ssq = torch.empty(M, N // 64, device=DEV)
    ops.pgemm(a, w, residual=r, ssq=ssq)
    torch.testing.assert_close(r.float(), want, atol=4e-2, rtol=2.0 ** -7)
    torch.testing.assert_close(ssq, r.float().pow(2).view(M, N // 64, 64).sum(-1), atol=1e-3, rtol=1e-5)
    s = torch.rand(M, device=DEV) + 0.5
    torch.testing.assert_close(ops.pgemm(a, w, row_scale=s).float(), z * s[:, None], **tol)
    assert not any(int(c.abs().sum()) for c in ops._PG_COUNTERS.values())


@pytest.mark.parametrize("M,N,K", [(1, 256, 192), (300, 256, 256), (513, 512, 768), (257, 768, 832)])
def test_k13_on_fewer_workgroups_than_xcds(M, N, K):
    """1 to 6 whole tiles, a workgroup each."""
    assert ops.native().pgemm_tail_floats(M, N, K) == 0 and -(-M // 256) * (N // 256) < 8
    a, w = _k13(M, N, K)
    torch.testing.assert_close(ops.pgemm(a, w).float(), a.float() @ w.float().t(), atol=4e-3, rtol=2.0 ** -7)


def test_k13_under_capture():
    """A captured product runs whole tiles and replays beside eager ones."""
    a, w = _k13(2048, 4096, 4096)
    y, st = ops.pgemm(a, w), torch.cuda.Stream()
    out = torch.empty_like(y)
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        ops.pgemm(a, w, out=out)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=st):
            ops.pgemm(a, w, out=out)
    for _ in range(3):
        out.zero_()
        g.replay()
        assert torch.equal(ops.pgemm(a, w), y)
        torch.cuda.synchronize()
        torch.testing.assert_close(out.float(), y.float(), atol=4e-3, rtol=2.0 ** -7)


# ------------------------------------------------- K24: the encoders' attention --
@pytest.mark.parametrize("lens", [[1], [16], [33, 1, 2], [64, 65, 63], [127, 128, 129, 5], [700, 31, 32, 256],
                                  [1, 1024, 3]])
@pytest.mark.parametrize("H,rope,thr", [(12, True, 8.0), (3, False, 8.0), (16, True, 0.0), (2, False, 0.0)])
def test_k24_attention(lens, H, rope, thr):
    """Against softmax(q k^T) v in 64 bits on the same rounded operands; the weights enter the
    second product as bf16 and the output is bf16: 2^-8 each of sum p |v| and of the output.
    One sequence is NaN and must not be seen by the others."""
    D, T = 64, sum(lens)
    wide = torch.randn(T, 3 * H * D + 8, device=DEV).bfloat16()
    qkv = wide[:, :3 * H * D]                                   # rows wider than q, k, v
    qkv[:, :2 * H * D] *= 3                                     # wide scores
    cu = torch.tensor([0] + lens, device=DEV).cumsum(0).int()
    cs = None
    if rope:
        a = torch.arange(max(lens), device=DEV)[:, None] * 1e4 ** (-torch.arange(32, device=DEV) / 32)
        cs = torch.cat([a.cos(), a.sin()], 1).float().contiguous()
    bad = len(lens) // 2 if len(lens) > 1 else -1
    if bad >= 0:
        qkv[cu[bad]:cu[bad + 1]] = float("nan")
    got = encoder.attention(qkv, cu, encoder.batch(lens, torch.device(DEV)), H, D ** -0.5, cs, thr)
    for i, n in enumerate(lens):
        lo, o = int(cu[i]), got[int(cu[i]):int(cu[i + 1])]
        if i == bad:
            assert o.isnan().all()
            continue
        q, k, v = qkv[lo:lo + n].float().view(n, 3, H, D).unbind(1)
        if rope:
            c, s = cs[:n, None, :32], cs[:n, None, 32:]
            q, k = (torch.cat([x[..., :32] * c - x[..., 32:] * s, x[..., 32:] * c + x[..., :32] * s], -1)
                    .bfloat16().float() for x in (q, k))
        q, k, v = (x.double().transpose(0, 1) for x in (q, k, v))
        p = (q @ k.transpose(1, 2) * D ** -0.5).softmax(-1)
        want, bound = p @ v, 2.0 ** -8 * (p @ v.abs())
        bound = 1.05 * (bound + 2.0 ** -8 * (want.abs() + bound)) + 1e-4      # fp32 sums and exponents
        err = (o.double().view(n, H, D).transpose(0, 1) - want).abs()
        assert (err <= bound).all(), (err - bound).max()


# ---------------------------------------- K4: short partitions and their sum --
@pytest.mark.parametrize("ctxs,parts", [([255, 256, 257], 16), ([1, 513, 2049], 8), ([2304], 9), ([6000], 40),
                                        ([300] * 8, 4), ([700] * 9, 4), ([3000, 40], 17)])
@pytest.mark.parametrize("Hq,Hkv,D", [(32, 8, 128), (8, 8, 64)])
def test_k4_partitions(ctxs, parts, Hq, Hkv, D):
    """Few rows, cut to 256 tokens, up to 24 partitions (sums of 8 at a time): the softmax in
    64 bits; weights as bf16 and a bf16 output, 2^-8 each of sum p |v| and of the output."""
    B, pages = len(ctxs), [-(-c // 32) for c in ctxs]
    NB = sum(pages) + 1
    kc = torch.randn(NB, Hkv, 32, D, device=DEV).bfloat16() * 2
    vc = torch.randn(NB, Hkv, 8, D, 4, device=DEV).bfloat16()           # key quads
    bt = torch.zeros(B, max(pages), dtype=torch.int32, device=DEV)
    perm = torch.randperm(NB, device=DEV).int()
    for b in range(B):
        bt[b, :pages[b]] = perm[sum(pages[:b]):sum(pages[:b + 1])]
    ctx = torch.tensor(ctxs, dtype=torch.int32, device=DEV)
    q = torch.randn(B, Hq * D, device=DEV).bfloat16()
    out = torch.empty(B, Hq * D, dtype=torch.bfloat16, device=DEV)
    ws = ops.DecodeWorkspace(B, Hq, D, parts, DEV)
    ws.part_o.fill_(float("nan"))                                       # unused partitions are not read
    ws.part_ml.fill_(float("nan"))
    ops.paged_decode_attention(q, kc, vc, bt, ctx, D ** -0.5, out, ws, Hq=Hq)
    for b, n in enumerate(ctxs):
        t = bt[b, :pages[b]].long()
        k = kc[t].transpose(1, 2).reshape(-1, Hkv, D)[:n].double()
        v = vc[t].permute(0, 2, 4, 1, 3).reshape(-1, Hkv, D)[:n].double()
        k, v = (x.repeat_interleave(Hq // Hkv, 1).transpose(0, 1) for x in (k, v))
        p = (q[b].double().view(Hq, 1, D) @ k.transpose(1, 2) * D ** -0.5).softmax(-1)
        want, bound = p @ v, 2.0 ** -8 * (p @ v.abs())
        bound = 1.05 * (bound + 2.0 ** -8 * (want.abs() + bound)) + 1e-4
        assert ((out[b].double().view(Hq, 1, D) - want).abs() <= bound).all()


# ------------------------------------------------------------ K25: one or two rows --
@pytest.mark.parametrize("M", [1, 2])
@pytest.mark.parametrize("N,K", [(32, 1024), (96, 3072), (3072, 2048), (2048, 8192), (4128, 14336)])
def test_k25(M, N, K):
    """Every epilogue against 64 bits: fp32 sums of K products (K / 64 in turn, then 64 by halves:
    an error of K / 64 + 6 roundings of sum |a w| at most), bf16 results."""
    a = torch.randn(M, K + 8, device=DEV).bfloat16()[:, :K]              # rows wider than K
    w = torch.randn(N, K, device=DEV).bfloat16() * K ** -0.5
    z, size = a.double() @ w.double().t(), a.double().abs() @ w.double().abs().t()
    slack = (K / 64 + 6) * 2.0 ** -24 * size
    calls = ops.GEMV_CALLS[0]

    def close(got, want, bound):
        assert ((got.double() - want).abs() <= bound + 2.0 ** -8 * want.abs() + 1e-30).all()

    close(ops.linear(a, w), z, slack)
    b = torch.randn(N, device=DEV).bfloat16()
    close(ops.linear(a, w, bias=b), z + b.double(), slack + 2.0 ** -23 * (z + b.double()).abs())
    p = ops.linear(a, w, defer=True)
    assert p.slabs.numel() == (2 if N < 4096 and K // 1024 % 2 == 0 else 1) * M * N
    assert ((p.slabs.view(-1, M, N).double().sum(0) - z).abs() <= slack).all()
    g, u = z.view(M, N // 32, 2, 16).unbind(2)
    gs, us = slack.view(M, N // 32, 2, 16).unbind(2)
    for got, act in ((ops.linear_swiglu(a, w, ops.SWIGLU16), torch.nn.functional.silu),
                     (ops.linear_relu_glu(a, w), torch.relu)):
        bound = 1.1 * gs * u.abs() + act(g).abs() * us + 2.0 ** -20 * (act(g) * u).abs() + 2 * gs * us
        close(got, (act(g) * u).reshape(M, -1), bound.reshape(M, -1))
    out = torch.zeros(M, N + 2, device=DEV).bfloat16()[:, :N]            # any even row stride
    close(ops.linear(a, w, out=out), z, slack)
    assert ops.GEMV_CALLS[0] == calls + 6
    a[0, 5] = float("inf")
    assert not ops.linear(a, w)[0].isfinite().any()


@pytest.mark.parametrize("M,N,K", [(1, 96, 1024), (2, 96, 1024), (3, 96, 1024), (32, 96, 96), (4, 96, 160)])
def test_few_rows_destinations(M, N, K):
    """Any destination that torch writes: odd rows and offsets, other types, the operands' own memory;
    gradients; empty products.  Two roundings to bf16 at most (product, sum with a bias)."""
    a, w = torch.randn(M, K, device=DEV).bfloat16(), torch.randn(N, K, device=DEV).bfloat16() * K ** -0.5
    y, tol = a.double() @ w.double().t(), dict(atol=4e-3, rtol=2.0 ** -8)
    buf = torch.zeros(M, N + 3, device=DEV).bfloat16()
    wide = torch.zeros(M, 2 * N, device=DEV).bfloat16()
    for out in (buf[:, 1:N + 1], buf[:, :N], buf[:, 2:N + 2], wide[:, ::2], torch.zeros(M, N, device=DEV),
                torch.zeros(N, M, device=DEV).bfloat16().t()):
        got = ops.linear(a, w, out=out)
        torch.testing.assert_close(got.double(), y, **tol)
        torch.testing.assert_close(out.double(), y, **tol)
    both = torch.cat([a, torch.zeros(M, N, device=DEV).bfloat16()], 1)
    at = both.clone()
    ops.linear(at[:, :K], w, out=at[:, :N])                        # over its own rows
    torch.testing.assert_close(at[:, :N].double(), y, **tol)
    g = torch.zeros(M, N // 2 + 1, device=DEV).bfloat16()[:, 1:]
    p, q = y.view(M, N // 32, 2, 16).unbind(2)
    ops.linear_swiglu(a, w, ops.SWIGLU16, out=g)
    torch.testing.assert_close(g.double(), (torch.nn.functional.silu(p) * q).reshape(M, -1), atol=2e-2,
                               rtol=2.0 ** -6)
    v = w.clone().requires_grad_()
    ops.linear(a, v).float().sum().backward()
    torch.testing.assert_close(v.grad.double(), a.double().sum(0).expand(N, K), atol=1e-2 * M, rtol=1e-2)
    assert ops.linear(a, w[:0]).shape == (M, 0)
    assert not ops.linear(a[:, :0], w[:, :0]).any()
