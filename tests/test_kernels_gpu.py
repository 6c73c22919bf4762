"""HIP kernels at the sizes where their tiles, splits and dispatch rules
meet, against float64 on the same bfloat16 inputs."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def lib():
    from fei_amd import ops
    ops.require_lib()
    return ops


def randbf(*shape, seed=0, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * scale).bfloat16()


def row_err(got, want):
    """Largest error of a row, relative to the row."""
    d = (got.double() - want).norm(dim=-1)
    return float((d / want.norm(dim=-1).clamp_min(1e-30)).max())


# -- prompt attention ----------------------------------------------------------

def attend64(q, k, v, pos0, scale, kv_len=None):
    S, T = q.shape[1], k.shape[2]
    G = q.shape[2] // k.shape[1]
    k, v = (t.double().repeat_interleave(G, 1) for t in (k, v))
    s = torch.matmul(q.transpose(1, 2).double(),
                     k.transpose(2, 3).contiguous()) * scale
    key = torch.arange(T, device=DEV).view(1, 1, 1, T)
    last = (pos0.view(-1, 1, 1, 1) + torch.arange(S, device=DEV).view(1, 1, S, 1)
            if kv_len is None else kv_len.view(-1, 1, 1, 1) - 1)
    p = torch.softmax(s.masked_fill(key > last, float("-inf")), -1)
    return torch.matmul(p.nan_to_num(0.0), v).transpose(1, 2)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S,Hq,Hkv,T,pos0,kv_len,scale", [
    (1, 8, 2, 64, [0], None, None),             # one key
    (33, 4, 1, 128, [31, 0], None, None),       # 132 rows: a block and a bit
    (63, 5, 1, 700, [637], None, None),         # groups of 5, splits
    (32, 12, 3, 1400, [1368, 2], None, None),   # one split used, or all
    (257, 3, 3, 257, [0], None, -0.2),          # groups of 1; scale < 0
    (40, 4, 2, 64, [10], None, 0.0),            # all keys alike
    (65, 3, 3, 65, [0, 0, 0], [65, 1, 0], None),   # no key at all
    (70, 2, 2, 4000, [0, 0], [4000, 129], None),
    # rows of a batch that are cut and not: one long one, as many as make none
    # worth it, more than a wave's lanes
    (150, 12, 3, 1400, [900, 0, 20, 300], None, None),
    (150, 12, 3, 1400, [900, 950, 800, 960], None, None),
    (3, 4, 1, 1300, [1200] * 3 + [0, 700] * 33 + [1000], None, None),
])
def test_attn_prefill_geometries(lib, D, S, Hq, Hkv, T, pos0, kv_len, scale):
    B, W = len(pos0), (Hq + 2 * Hkv) * D
    qkv = randbf(B, S, W, seed=S)
    q = qkv.as_strided((B, S, Hq, D), (S * W, W, D, 1))
    k, v = randbf(B, Hkv, T, D, seed=1), randbf(B, Hkv, T, D, seed=2)
    # what lies past the keys is never used
    ends = kv_len or [p + S for p in pos0]
    kn, vn = k.clone(), v.clone()
    for b, n in enumerate(ends):
        kn[b, :, n:] = vn[b, :, n:] = float("nan")
    p0 = torch.tensor(pos0, dtype=torch.int32, device=DEV)
    kl = None if kv_len is None else torch.tensor(kv_len, dtype=torch.int32,
                                                  device=DEV)
    got = lib.attn_prefill(q, kn, vn, p0, scale=scale, causal=kv_len is None,
                           kv_len=kl)
    want = attend64(q, k, v, p0, D ** -0.5 if scale is None else scale, kl)
    # weights and results are each rounded to bfloat16 once: 2^-9 of each
    # weight times its value, and 2^-9 of the result
    assert row_err(got, want) < 2 ** -7


# -- decode GEMVs ----------------------------------------------------------------

def rms64(x, g, eps):
    x = x.double()
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * g.double()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("M,N,K", [
    (1, 8, 16),            # less than one load a lane
    (1, 9, 2064),          # odd rows, a few loads past the full ones
    (2, 2048, 4096),       # rows shared by four waves
    (2, 33, 8208),         # the same with a remainder
    (3, 2050, 4112),
    (1, 130, 14336),
    (3, 17, 14336),        # more activations than 64 KB
    (4, 24, 4096),
    (8, 11, 2048),
    (8, 10, 4096),
    (8, 6, 8192),          # 128 KB of LDS
])
def test_gemv_geometries(lib, M, N, K, fp8):
    """Norm inside or not, plain, residual and SwiGLU sums, both kinds of
    weights. Sums are float32 and rounded to bfloat16 once: 2^-9 of a value,
    2^-8 allowed. Normed rows are rounded once more, for a SwiGLU before both
    products: 3 * 2^-9 in all, 2^-7 allowed."""
    if fp8 and M * K * 2 > 65536:
        pytest.skip("the fp8 products refuse rows of this size")
    x, g = randbf(M, K, seed=M), randbf(K, seed=3) * 0.2 + 1
    w = randbf(2 * N, K, seed=N, scale=K ** -0.5)
    res = randbf(M, N, seed=5)
    w64, w1 = w.double(), w
    if fp8:
        w1, sc = lib.quant_fp8(w)
        w64 = w1.view(torch.float8_e4m3fn).double() * sc.double()[:, None]
    half = (lambda t: t[:N].contiguous())
    xn = rms64(x, g, 1e-5)
    x64 = x.double()
    r = res.clone()
    if fp8:
        got = lib.gemv_norm_fp8(x, g, half(w1), half(sc))
        sw = lib.gemv_swiglu_norm_fp8(x, g, w1, sc)
        lib.gemv_res_fp8(x, half(w1), half(sc), r)
    else:
        # the kernel itself: most rows of these sizes go to another
        def run(out, gain, w, epi):
            lib._launch_gemv(out, x, gain, w, None, N, 1e-5, epi)
            return out
        new = lambda: torch.full_like(r, float("nan"))
        got = run(new(), g, half(w), lib._BF16)
        sw = run(new(), g, w, lib._SWIGLU)
        run(r, None, half(w), lib._RES)
        assert row_err(run(new(), None, half(w), lib._BF16),
                       x64 @ w64[:N].T) < 2 ** -8
        y = x64 @ w64.T
        assert row_err(run(new(), None, w, lib._SWIGLU),
                       torch.nn.functional.silu(y[:, :N]) * y[:, N:]) < 2 ** -8
    tol = 2 ** -7
    assert row_err(got, xn @ w64[:N].T) < tol
    assert row_err(r, res.double() + x64 @ w64[:N].T) < 2 ** -8
    y = xn @ w64.T
    assert row_err(sw, torch.nn.functional.silu(y[:, :N]) * y[:, N:]) < tol


# -- decode attention --------------------------------------------------------------

def rope64(x, pos, theta=500000.0):
    D = x.shape[-1]
    inv = theta ** (-torch.arange(0, D, 2, dtype=torch.float64, device=DEV) / D)
    a = (pos.double().view(-1, 1) * inv).unsqueeze(1)
    u, w = x[..., :D // 2].double(), x[..., D // 2:].double()
    return torch.cat([u * a.cos() - w * a.sin(), w * a.cos() + u * a.sin()], -1)


def test_attn_prefill_rows_far_apart(lib):
    """Cache rows so far from each other that a tile's offsets have more than 32
    bits."""
    n, S, D, far = 70, 40, 64, 1 << 25
    room = torch.empty(n * far, dtype=torch.bfloat16, device=DEV)
    k, v = (room[i * D:].as_strided((1, 1, n, D), (n * far, n * far, far, 1))
            for i in range(2))
    k.copy_(randbf(1, 1, n, D, seed=1))
    v.copy_(randbf(1, 1, n, D, seed=2))
    q = randbf(1, S, 2, D, seed=3)
    p0 = torch.tensor([n - S], dtype=torch.int32, device=DEV)
    assert torch.equal(lib.attn_prefill(q, k, v, p0),
                       lib.attn_prefill(q, k.contiguous(), v.contiguous(), p0))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("Hq,Hkv,splits,lens", [
    (8, 2, 4, [1, 2]),               # the new token alone
    (3, 1, 32, [31, 32, 33]),        # around a wave's 32 keys, groups of 3
    (8, 1, 16, [128, 129, 300]),     # one split, two
    (16, 1, 2, [700]),               # more keys than one round of the splits
    (4, 4, 64, [2000, 15, 1]),
    (8, 2, 1, [257, 500]),
])
def test_attn_decode_geometries(lib, D, paged, rope, Hq, Hkv, splits, lens):
    """Against float64, over caches whose rows past each length are NaN, with
    the step's RoPE and cache row made inside or before."""
    from fei_amd.ops import reference as ref
    B, BS, T = len(lens), 16, max(lens) + 5
    W = (Hq + 2 * Hkv) * D
    qkv = randbf(B, W, seed=sum(lens))
    q, k, v = (qkv[:, a * D:b * D].view(B, -1, D) for a, b in
               ((0, Hq), (Hq, Hq + Hkv), (Hq + Hkv, Hq + 2 * Hkv)))
    pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device=DEV)
    kc, vc = randbf(B, Hkv, T, D, seed=1), randbf(B, Hkv, T, D, seed=2)
    for b, n in enumerate(lens):
        kc[b, :, n - rope:] = vc[b, :, n - rope:] = float("nan")
    args = dict(splits=splits)
    if rope:
        table = ref.rope_table(T, D, device=DEV)
        args.update(k=k, v=v, table=table)
    if paged:
        nb = -(-T // BS)
        perm = torch.randperm(B * nb, generator=torch.Generator().manual_seed(3))
        bt = perm.view(B, nb).int().to(DEV)
        pools = []
        for c in (kc, vc):
            pad = torch.full((B, Hkv, nb * BS, D), float("nan"), device=DEV,
                             dtype=torch.bfloat16)
            pad[:, :, :T] = c
            p = torch.empty(B * nb, Hkv, BS, D, device=DEV, dtype=torch.bfloat16)
            p[bt.view(-1).long()] = pad.view(B, Hkv, nb, BS, D).transpose(1, 2) \
                .reshape(B * nb, Hkv, BS, D)
            pools.append(p)
        got = lib.attn_decode_paged(q, *pools, bt, pos, **args)
        kn, vn = (p[bt.long()].transpose(1, 2).reshape(B, Hkv, nb * BS, D)[:, :, :T]
                  for p in pools)
    else:
        got = lib.attn_decode(q, kc, vc, pos, **args)
        kn, vn = kc, vc
    q64 = rope64(q, pos) if rope else q.double()
    k64 = rope64(k, pos)
    for b, n in enumerate(lens):
        if rope:                     # the row is in the cache now, rounded once
            assert row_err(kn[b, :, n - 1], k64[b]) < 2 ** -8
            assert torch.equal(vn[b, :, n - 1], v[b])
        kk, vv = (t[b, :, :n].double().repeat_interleave(Hq // Hkv, 0)
                  for t in (kn, vn))
        p = torch.softmax((kk * q64[b].unsqueeze(1)).sum(-1) * D ** -0.5, -1)
        # the result is rounded once: 2^-9
        assert row_err(got[b], (p.unsqueeze(-1) * vv).sum(1)) < 2 ** -8


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("T,splits", [(64, 4), (512, 1), (512, 8)])
def test_attn_decode_without_keys(lib, paged, T, splits):
    """A position before the first: zeros, whether one block or several would
    have the keys, and no cache row."""
    from fei_amd.ops import reference as ref
    B, Hq, Hkv, D, BS = 3, 4, 2, 64, 16
    q, k, v = (randbf(B, H, D, seed=H) for H in (Hq, Hkv, Hkv + 5))
    v = v[:, :Hkv].contiguous()
    pos = torch.tensor([-1, 5, -200], dtype=torch.int32, device=DEV)
    shape = (B * (T // BS), Hkv, BS, D) if paged else (B, Hkv, T, D)
    kc, vc = (torch.zeros(shape, device=DEV, dtype=torch.bfloat16)
              for _ in range(2))
    out = torch.full((B, Hq, D), float("nan"), device=DEV, dtype=torch.bfloat16)
    args = dict(splits=splits, k=k, v=v, out=out,
                table=ref.rope_table(T, D, device=DEV))
    if paged:
        bt = torch.arange(shape[0], device=DEV, dtype=torch.int32).view(B, -1)
        lib.attn_decode_paged(q, kc, vc, bt, pos, **args)
        kc, vc = (c.view(B, T // BS, Hkv, BS, D) for c in (kc, vc))
    else:
        lib.attn_decode(q, kc, vc, pos, **args)
    assert not out[0].any() and not out[2].any() and out[1].isfinite().all()
    for c in (kc, vc):
        assert not c[0].any() and not c[2].any() and c[1].any()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("Hq,Hkv,lens", [
    (8, 2, [1, 129, 251]),           # little room
    (32, 2, [250]),                  # groups of 16: the most LDS
    (12, 4, [31, 33, 63, 257, 288] * 4),         # 64 heads and more
    (8, 8, [700, 511, 513, 1, 97, 300, 400, 512]),
    (8, 8, list(range(960, 1160, 10))),          # 160 heads: several rounds
    (8, 8, [60] * 19 + [1019]),      # one long one among short ones, the most in one
    (8, 8, [1020] + [60] * 20),      # block and the fewest in several
])
def test_attn_decode_in_one_block(lib, D, paged, rope, Hq, Hkv, lens):
    """Where a block takes all keys of a head."""
    test_attn_decode_geometries(lib, D, paged, rope, Hq, Hkv, 8, lens)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("Hq,Hkv,lens", [
    (16, 8, [1500, 1, 700, 129, 128, 900] * 3),  # 144 heads: fewer splits than asked
    (10, 10, list(range(1200, 1350, 10))),       # 150
])
def test_attn_decode_as_many_blocks_as_places(lib, D, paged, Hq, Hkv, lens):
    test_attn_decode_geometries(lib, D, paged, True, Hq, Hkv, 16, lens)


@pytest.mark.parametrize("paged", [False, True])
def test_attn_decode_in_one_block_without_keys(lib, paged):
    test_attn_decode_without_keys(lib, paged, 192, 4)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("Hq,Hkv,n,size", [(8, 2, 700, 1), (4, 4, 300, 4),
                                           (16, 1, 1000, 1)])
def test_attn_decode_sums_are_float32(lib, D, rope, Hq, Hkv, n, size):
    """The splits' sums, which are not rounded to bfloat16: queries under RoPE
    and weights keep float32's 24 bits. Scores are of size ``size`` squared; D
    roundings of 2^-24 make theirs, and what comes of it is relative to the
    result: 1e-6. Weights or queries of 16 bits are 2e-6 and more off."""
    from fei_amd.ops import reference as ref
    W, T, splits = (Hq + 2 * Hkv) * D, n + 3, 8
    qkv = randbf(1, W, seed=n) * size
    q, k, v = (qkv[:, a * D:b * D].view(1, -1, D) for a, b in
               ((0, Hq), (Hq, Hq + Hkv), (Hq + Hkv, Hq + 2 * Hkv)))
    kc, vc = randbf(1, Hkv, T, D, seed=1), randbf(1, Hkv, T, D, seed=2)
    pos = torch.tensor([n - 1], dtype=torch.int32, device=DEV)
    table = ref.rope_table(T, D, device=DEV)
    po = torch.zeros(1, Hq, splits, D, device=DEV)
    ml = torch.zeros(1, Hq, splits, 2, device=DEV)
    ml[..., 0] = -3e38
    lib.attn_decode(q, kc, vc, pos, splits=splits, workspace=(po, ml),
                    **(dict(k=k, v=v, table=table) if rope else {}))
    used = min(splits, -(-n // 128))
    assert used > 1 and not ml[:, :, used:, 1].any()
    top = ml[0, ..., 0].double().amax(-1, keepdim=True)
    w = torch.exp2(ml[0, ..., 0].double() - top)
    got = (po[0].double() * w.unsqueeze(-1)).sum(1) \
        / (ml[0, ..., 1].double() * w).sum(-1, keepdim=True)
    q64 = q[0].double()
    if rope:                           # by the same float32 angles
        c, s = table.view(T, D // 2, 2)[n - 1].double().unbind(-1)
        a, b = q64.split(D // 2, -1)
        q64 = torch.cat([a * c - b * s, b * c + a * s], -1)
    kk, vv = (t[0, :, :n].double().repeat_interleave(Hq // Hkv, 0)
              for t in (kc, vc))
    p = torch.softmax((kk * q64.unsqueeze(1)).sum(-1) * D ** -0.5, -1)
    assert row_err(got, (p.unsqueeze(-1) * vv).sum(1)) < 1e-6


# -- products of few rows on the matrix units ------------------------------------

@pytest.mark.parametrize("M", [2, 3, 4, 8, 9, 17, 25, 32, 40, 64])
@pytest.mark.parametrize("N,K", [
    (16, 64),              # one stage, three waves without any
    (20, 320),             # five stages for four waves, a part of a tile
    (5120, 192),           # tiles of 32 rows
    (8200, 64),            # SwiGLU: tiles of 64 rows, the last in part
    (2048, 4160),
])
def test_skinny_geometries(lib, M, N, K):
    """Each kind of result, against float64: float32 sums, rounded to
    bfloat16 once where the result is (2^-9; 2^-8 allowed)."""
    from fei_amd.ops import mixers as mx
    x, w = randbf(M, K, seed=M), randbf(2 * N, K, seed=N, scale=K ** -0.5)
    assert mx.skinny_ok(M, K, x, w) == (3 <= M <= 32)
    assert mx.skinny_ok(M, K, x, w, 2) == (M <= 32)
    y = x.double() @ w.double().T
    a, b = y[:, :N], y[:, N:]
    w1 = w[:N].contiguous()
    out = torch.full((M, N), float("nan"), device=DEV, dtype=torch.bfloat16)
    mx.skinny(out, x, w1, N, mx.EPI_BF16)
    assert row_err(out, a) < 2 ** -8
    b16 = randbf(N, seed=2)
    mx.skinny(out, x, w1, N, mx.EPI_BF16, bias16=b16)
    assert row_err(out, a + b16.double()) < 2 ** -8
    mx.skinny(out, x, w1, N, mx.EPI_GELU, bias16=b16)
    assert row_err(out, torch.nn.functional.gelu(a + b16.double())) < 2 ** -8
    res = randbf(M, N, seed=1)
    want = res.double() + a
    mx.skinny(res, x, w1, N, mx.EPI_RES_BF16)
    assert row_err(res, want) < 2 ** -8
    wide = torch.zeros(M, N + 24, device=DEV, dtype=torch.bfloat16)
    mx.skinny(None, x, w, N, mx.EPI_SWIGLU, act=wide[:, 8:], stride=N + 24)
    assert row_err(wide[:, 8:8 + N], torch.nn.functional.silu(a) * b) < 2 ** -8
    assert not wide[:, :8].any() and not wide[:, 8 + N:].any()
    bias = torch.randn(N, device=DEV)
    f = torch.empty(M, N, device=DEV)
    mx.skinny(f, x, w1, N, mx.EPI_F32, bias=bias, scale=0.5, cap=3.0)
    assert row_err(f, 3 * torch.tanh(a * 0.5 / 3) + bias.double()) < 1e-5
    mx.skinny(f.copy_(want), x, w1, N, mx.EPI_RES, scale=0.25)
    assert row_err(f, want.float().double() + 0.25 * a) < 1e-5
    n_mix, n_r = N - 12, 4
    proj = torch.empty(M, n_mix, device=DEV, dtype=torch.bfloat16)
    router = torch.empty(M, n_r, device=DEV)
    act = torch.zeros(M, 16, device=DEV, dtype=torch.bfloat16)
    mx.skinny(proj, x, w1, N, mx.EPI_PARALLEL, n_mix=n_mix, router=router,
              act=act[:, 4:], stride=16)
    assert row_err(proj, a[:, :n_mix]) < 2 ** -8
    assert row_err(router, a[:, n_mix:n_mix + n_r]) < 1e-5
    assert (act[:, 4:12].double() - a[:, -8:].clamp(min=0) ** 2).abs().max() \
        < 2 ** -8 * (a[:, -8:] ** 2).max()
    if M > 32:
        return
    # a residual's next product under a norm: the sums of squares of its tiles
    h = randbf(M, N, seed=6)
    sums = lib.add_product(x, w1, h)
    assert row_err(sums, (h.double() ** 2 @ torch.nn.functional.pad(
        torch.eye(-(-N // 16), device=DEV, dtype=torch.float64)
        .repeat_interleave(16, 0)[:N], (0, 0)))) < 1e-5
    if N % 64 == 0:
        g, w2 = randbf(N, seed=7), randbf(48, N, seed=8, scale=N ** -0.5)
        # inputs rounded under their gains: 2^-9 of each product, up to twice
        # that of a row of few results; a SwiGLU takes two of them with slopes
        # of up to 1.1, 2.2 * 2^-8, and is rounded: under 2^-6
        y2 = rms64(h, g, 1e-5) @ w2.double().T
        assert row_err(lib.gemv_norm(h, g, w2, 1e-5, sums=sums), y2) < 2 ** -7
        assert row_err(lib.gemv_swiglu_norm(h, g, w2, 1e-5, sums=sums),
                       torch.nn.functional.silu(y2[:, :24]) * y2[:, 24:]) \
            < 2 ** -6


@pytest.mark.parametrize("M", [2, 8, 9, 24, 32])
@pytest.mark.parametrize("N,K", [(16, 64), (200, 320), (2048, 192), (2056, 64),
                                 (4000, 128)])
def test_skinny_blocks_of_8_columns(lib, M, N, K):
    """Up to 2048 columns and past them: sums of squares by blocks, a last block in
    part, waves without steps; the products that read the rows under a norm."""
    x, w = randbf(M, K, seed=1), randbf(N, K, seed=2, scale=K ** -0.5)
    h, res = randbf(M, N, seed=3), randbf(M, N, seed=3)
    want = h.double() + x.double() @ w.double().T
    sums = lib.add_product(x, w, h, any_tiles=True)
    # rounded once, by 2^-9 at most; the sums of squares are of what is written
    assert row_err(h, want) < 2 ** -8
    cols = 8 if N <= 2048 else 16
    sq = torch.nn.functional.pad(h.double() ** 2, (0, -N % cols))
    assert row_err(sums, sq.view(M, -1, cols).sum(-1)) < 1e-5
    assert row_err(lib.add_product(x, w, res),
                   torch.nn.functional.pad(res.double() ** 2, (0, -N % 16))
                   .view(M, -1, 16).sum(-1)) < 1e-5
    if N % 64 == 0:
        g, w2 = randbf(N, seed=4), randbf(48, N, seed=5, scale=N ** -0.5)
        # 2^-9 of each product, up to twice that of a row of few results
        assert row_err(lib.gemv_norm(h, g, w2, 1e-5, sums=sums),
                       rms64(h, g, 1e-5) @ w2.double().T) < 2 ** -7


@pytest.mark.parametrize("M", [2, 8, 9, 24, 32])
@pytest.mark.parametrize("N,K", [(128, 1024), (2048, 8192), (1000, 320)])
def test_skinny_blocks_of_8_and_16_columns_agree(lib, M, N, K):
    """To the last bit: the encoder has both in front of the same rows."""
    x, w = randbf(M, K, seed=1), randbf(N, K, seed=2, scale=K ** -0.5)
    h = [randbf(M, N, seed=3) for _ in range(2)]
    for any_tiles in (False, True):
        lib.add_product(x, w, h[any_tiles], any_tiles)
    assert torch.equal(*h)


# -- RoPE of a prompt --------------------------------------------------------------

@pytest.mark.parametrize("B,S,Hq,Hkv,D,pad", [
    (1, 1, 1, 1, 64, 0), (2, 33, 5, 1, 128, 0), (1, 7, 4, 2, 24, 0),
    (1, 9, 3, 3, 64, 3),         # rows that start at no multiple of 16 bytes
])
def test_rope_prefill_geometries(lib, B, S, Hq, Hkv, D, pad):
    from fei_amd.ops import reference as ref
    W, T = (Hq + 2 * Hkv) * D + pad, S + 9
    buf = randbf(B * S * W + 8, seed=S)
    parts = [buf.as_strided((B, S, H, D), (S * W, W, D, 1), o * D + (pad and 1))
             for H, o in ((Hq, 0), (Hkv, Hq), (Hkv, Hq + Hkv))]
    q, k, v = parts
    q0 = q.clone()
    pos0 = torch.arange(B, dtype=torch.int32, device=DEV) * 4 + 3
    kc, vc = (torch.zeros(B, Hkv, T, D, device=DEV, dtype=torch.bfloat16)
              for _ in range(2))
    lib.rope_kv_prefill(q, k, v, kc, vc, pos0, ref.rope_table(T, D, device=DEV))
    for b in range(B):
        p = torch.arange(S, device=DEV) + pos0[b]
        # angles are float32, results rounded once
        assert row_err(q[b], rope64(q0[b], p)) < 2 ** -8
        assert row_err(kc[b, :, p].transpose(0, 1), rope64(k[b], p)) < 2 ** -8
        assert torch.equal(vc[b, :, p].transpose(0, 1), v[b])
    rest = torch.ones(T, dtype=torch.bool, device=DEV)
    rest[p] = False
    assert not kc[-1][:, rest].any() and not vc[-1][:, rest].any()


# -- encoder ---------------------------------------------------------------------

@pytest.mark.parametrize("cols", [8, 512, 520, 768, 1032, 2048, 2056])
@pytest.mark.parametrize("rows", [1, 5])
def test_layernorm_widths(lib, rows, cols):
    """Float32 statistics; the result is rounded once (2^-9)."""
    x, r = randbf(rows, cols, seed=1) + 3, randbf(rows, cols, seed=2)
    w, b = randbf(cols, seed=3), randbf(cols, seed=4)
    for res in (None, r):
        y = x.double() + (0 if res is None else r.double())
        want = torch.nn.functional.layer_norm(y, (cols,), w.double(),
                                              b.double(), 1e-6)
        assert row_err(lib.layernorm(x, w, b, 1e-6, residual=res), want) < 2 ** -8


def test_gelu_all_bfloat16(lib):
    """Every bfloat16 but -inf."""
    x = torch.arange(1 << 16, device=DEV, dtype=torch.int32).to(torch.int16) \
        .view(torch.bfloat16)
    got = lib.gelu(x)
    # torch's loses its digits below -7, in float64 too
    want = x.double() * torch.special.erfc(x.double() * -0.5 ** 0.5) / 2
    ok = x.isfinite()
    err = (got.double() - want).abs()[ok]
    # rounded once: 2^-9 of the value, in the far tail too; what an exponential
    # below float32's normal numbers makes of it is zero
    most = 2 ** -8 * want[ok].abs() + 2.0 ** -126
    assert (err <= most).all()
    assert got[x == float("inf")].eq(float("inf")).all()
    assert got[x.isnan()].isnan().all()


def test_encoder_attention_reads_views(lib):
    """Queries, keys and values as they lie in one projection, aligned or
    not, give what contiguous copies give."""
    B, S, H, D = 2, 70, 3, 64
    lens = torch.tensor([70, 9], dtype=torch.int32, device=DEV)
    zero = torch.zeros(B, dtype=torch.int32, device=DEV)
    buf = randbf(B * S * 3 * H * D + 8, seed=4)
    for shift in (0, 1):
        qkv = buf[shift:shift + B * S * 3 * H * D].view(B, S, 3, H, D)
        q, k, v = qkv.unbind(2)
        got = lib.attn_prefill(q, k.transpose(1, 2), v.transpose(1, 2), zero,
                               causal=False, kv_len=lens)
        want = lib.attn_prefill(q.contiguous(), k.transpose(1, 2).contiguous(),
                                v.transpose(1, 2).contiguous(), zero,
                                causal=False, kv_len=lens)
        assert torch.equal(got, want)


# -- prompt attention over windows ---------------------------------------------

@pytest.mark.parametrize("dims", [(128, 64, 128), (64, 0, 64), (64, 64, 128),
                                  (192, 64, 64), (64, 0, 192), (96, 32, 64)])
@pytest.mark.parametrize("window,parts,scale", [
    (0, [(1, 1, 0), (2, 129, 0), (131, 33, 70)], 0.1),
    (64, [(0, 200, 300), (200, 64, 0)], 0.1),
    (65, [(0, 128, 63), (130, 31, 1000)], -0.1),
    (1, [(0, 66, 5)], 0.1),
    (1024, [(0, 300, 1100)], 0.0),
])
def test_window_prefill_geometries(lib, dims, window, parts, scale):
    """Panels of 64 (the first four) and the general path, whose only
    difference is the width of the heads."""
    from fei_amd.ops import mixers as mx
    (dim, rot, vdim), H, kr = dims, 3, 64
    rows = max(r + n for r, n, _ in parts)
    q_w = H * (dim + rot)
    proj = randbf(rows, q_w + kr + rot + H * vdim, seed=rows)
    spans, tiles, at = [], [], 0
    for i, (r, n, pos0) in enumerate(parts):
        k0 = max(0, pos0 - window + 1) if window else 0
        spans.append([r, n, pos0, k0, at])
        tiles += [[i, q] for q in range(0, n, 128)]
        at += pos0 + n - k0
    kv = randbf(at, H * (dim + vdim), seed=1)
    krot = randbf(at, rot, seed=2)
    out = torch.full((rows, H * vdim), 7.0, dtype=torch.bfloat16, device=DEV)
    sp, tl = (torch.tensor(x, dtype=torch.int32, device=DEV)
              for x in (spans, tiles))
    p = mx._p
    mx._lib().fei_window_prefill(
        p(out), out.stride(0), p(proj), proj.stride(0), p(kv), p(krot), p(sp),
        p(tl), len(tiles), H, dim, rot, vdim, kr, scale, window, 0,
        mx._stream())
    used = torch.zeros(rows, dtype=torch.bool)
    for (r, n, pos0), (_, _, _, k0, a) in zip(parts, spans):
        used[r:r + n] = True
        m = pos0 + n - k0
        q = proj[r:r + n, :q_w].double().view(n, H, dim + rot).transpose(0, 1)
        keys = torch.cat(
            [kv[a:a + m, :H * dim].double().view(m, H, dim),
             krot[a:a + m].double()[:, None].expand(m, H, rot)], 2)
        s = torch.matmul(q, keys.permute(1, 2, 0).contiguous()) * scale
        qp = pos0 + torch.arange(n, device=DEV)[:, None]
        kp = k0 + torch.arange(m, device=DEV)[None]
        hide = kp > qp
        if window:
            hide |= qp - kp >= window
        w = torch.softmax(s.masked_fill(hide, float("-inf")), -1)
        v = kv[a:a + m, H * dim:].double().view(m, H, vdim).transpose(0, 1)
        o = torch.matmul(w, v.contiguous()).transpose(0, 1).reshape(n, -1)
        o = o * proj[r:r + n, q_w + kr + rot:].double().sigmoid()
        # weights keep 16 bits, sums are float32: the rounding of the result
        # (2^-9 an element, less in a row's norm) is what shows
        assert row_err(out[r:r + n], o) < 2.0 ** -8
    assert bool((out[~used.to(DEV)] == 7.0).all())


# -- products of tens of rows ----------------------------------------------------

@pytest.mark.parametrize("M,N,K", [
    (33, 64, 64), (64, 72, 128), (65, 200, 192), (96, 128, 1024),
    (97, 2048, 2048), (128, 4096, 4096), (129, 1000, 1088), (256, 136, 8192),
    (75, 6144, 4096),
])
def test_product_parts(lib, M, N, K):
    x, w = randbf(M, K + 64, seed=M)[:, :K], randbf(N, K, seed=N)
    assert lib.rows_ok(M, w)
    parts = lib.product_parts(x, w)
    want = x.double() @ w.double().t()
    # float32 sums of K products
    assert row_err(parts.sum(0), want) < 2.0 ** -22 * K ** 0.5
    h, gain = randbf(M, N, seed=3, scale=K ** 0.5), randbf(N, seed=4)
    res = h.clone()
    y = lib.add_norm_parts(parts, res, gain, 1e-5)
    new = (h.double() + want)
    assert row_err(res, new) < 2.0 ** -8
    inv = (res.double().pow(2).mean(-1, keepdim=True) + 1e-5).rsqrt()
    assert row_err(y, res.double() * inv * gain.double()) < 2.0 ** -8
    if N >= 64 and K >= 4096:
        from fei_amd.ops import rows
        acc = torch.randn(M, N, device=DEV)
        want = acc.double() + 0.3 * want
        assert rows.add_ok(acc, x, w)
        rows.add_product(acc, x, w, 0.3)
        assert row_err(acc, want) < 2.0 ** -22 * K ** 0.5


@pytest.mark.parametrize("M,I,K", [
    (33, 8, 64), (64, 64, 256), (75, 1000, 512), (128, 14336, 128),
    (256, 8192, 192), (200, 72, 1024),
])
def test_rows_swiglu(lib, M, I, K):
    from fei_amd.ops import rows
    x, w = randbf(M, K, seed=M), randbf(2 * I, K, seed=I, scale=K ** -0.5)
    assert rows.swiglu_ok(M, x, w)
    gu = x.double() @ w.double().t()
    want = torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]
    assert row_err(lib.gemv_swiglu(x, w), want) < 2.0 ** -8


@pytest.mark.parametrize("B,S,Hq,Hkv,D", [(1, 33, 4, 2, 128), (3, 17, 3, 1, 64),
                                          (2, 40, 2, 2, 16), (1, 75, 32, 8, 128)])
def test_rope_kv_parts(lib, B, S, Hq, Hkv, D):
    """Against the kernel for whole products."""
    T, W = B * S, (Hq + 2 * Hkv) * D
    parts = torch.randn(3, T, W, device=DEV)
    table = torch.randn(200, D // 2, 2, device=DEV)
    pos0 = torch.arange(B, device=DEV, dtype=torch.int32) * 7
    kc, vc = (torch.zeros(B, Hkv, 200, D, dtype=torch.bfloat16, device=DEV)
              for _ in range(2))
    kr, vr = kc.clone(), vc.clone()
    q = lib.rope_kv_parts(parts, S, Hq, kc, vc, pos0, table)
    qkv = parts.sum(0).bfloat16()
    q0, k0, v0 = (qkv[:, a * D:b * D].view(B, S, b - a, D) for a, b in (
        (0, Hq), (Hq, Hq + Hkv), (Hq + Hkv, Hq + 2 * Hkv)))
    lib.rope_kv_prefill(q0, k0, v0, kr, vr, pos0, table)
    # there the sums are rounded before they are turned, here only after
    for a, b in ((q, q0), (kc, kr), (vc, vr)):
        d = (a.double() - b.double()).abs().amax()
        assert d <= 2.0 ** -7 * b.double().abs().amax()
    assert torch.equal(vc, vr)


@pytest.mark.parametrize("B,S", [(1, 33), (2, 20), (1, 128), (2, 65), (1, 200)])
def test_prompt_in_parts_matches_whole_products(lib, B, S):
    import dataclasses
    from fei_amd.engine.config import get_spec
    from fei_amd.models.llama import LlamaModel
    spec = dataclasses.replace(get_spec("llama3-1b"), num_layers=2,
                               vocab_size=512)
    m = LlamaModel(spec, torch.device(DEV), torch.bfloat16, seed=1,
                   max_seq_len=256)
    toks = torch.randint(0, 512, (B, S), device=DEV)
    pos0 = torch.arange(B, dtype=torch.int32, device=DEV) * 3

    def run(parts):
        if not parts:
            m.rows_in_parts = lambda T, caches: False
        kc, vc = ([torch.zeros(B, spec.num_kv_heads, 256, m.D,
                               dtype=torch.bfloat16, device=DEV)
                   for _ in range(2)] for _ in range(2))
        return m.forward_prefill(toks, pos0, kc, vc, all_positions=True), kc, vc
    assert m.rows_in_parts(B * S, [])
    (a, ka, va), (b, kb, vb) = run(True), run(False)
    # a rounding of 2^-9 here and there, through two layers
    assert row_err(a, b.double()) < 2.0 ** -5
    for x, y in zip(ka + va, kb + vb):
        assert row_err(x.flatten(), y.double().flatten()) < 2.0 ** -6


# as many splits as the product sums itself, and one more, with keys for one split, for
# all, at their edges, and none
@pytest.mark.parametrize("Hq,Hkv,D", [(32, 8, 64), (16, 4, 128), (32, 8, 128), (6, 2, 64)])
@pytest.mark.parametrize("room", [128, 256, 320, 512, 640, 1024, 2048, 2112])
@pytest.mark.parametrize("fp8", [False, True])
def test_output_product_sums_the_splits(lib, Hq, Hkv, D, room, fp8):
    W, N = (Hq + 2 * Hkv) * D, 2056
    w = randbf(N, Hq * D, seed=1, scale=(Hq * D) ** -0.5)
    w, ws = lib.quant_fp8(w) if fp8 else (w, None)
    table = torch.randn(room, D // 2, 2, device=DEV)
    kc, vc = (randbf(1, Hkv, room, D, seed=i) for i in (2, 3))
    for n in sorted({0, 1, 127, 128, 129, room // 2, room - 1, room}):
        qkv = randbf(1, W, seed=n + 9)
        q, k, v = (qkv[:, a * D:b * D].view(1, -1, D) for a, b in (
            (0, Hq), (Hq, Hq + Hkv), (Hq + Hkv, Hq + 2 * Hkv)))
        # without RoPE where there is no key to turn
        rope = dict(k=k, v=v, table=table) if n else {}
        args = dict(splits=32, scale=D ** -0.5, **rope)
        pos = torch.tensor([n - 1], dtype=torch.int32, device=DEV)
        res = randbf(1, N, seed=5)
        got, want = res.clone(), res.clone()
        att = lib.attn_decode(q, kc.clone(), vc.clone(), pos, **args)
        # what no split has written is not read
        room_for = tuple(torch.full((1, Hq, 32, x), float("nan"), device=DEV)
                         for x in (D, 2))
        if fp8:
            lib.gemv_res_fp8(att.view(1, -1), w, ws, want)
            lib.attn_decode_product_fp8(q, kc.clone(), vc.clone(), pos, w, ws, got,
                                        workspace=room_for, **args)
        else:
            lib.gemv_res(att.view(1, -1), w, want)
            lib._launch_attn_decode(q, kc.clone(), vc.clone(), None, room, 0, Hkv, pos,
                                    32, D ** -0.5, room_for, None, rope.get("k"),
                                    rope.get("v"), rope.get("table"), (w, None, got))
        # the attention's sums are rounded to bfloat16 once, in another order here
        assert row_err(got, want.double()) < 2.0 ** -8, n


# one row, one and more groups of 8, prompts and decoding steps; ``odd``: a layer whose
# weights the kernels for few rows do not read as they lie, from which on the operations
# run one by one
@pytest.mark.parametrize("name", ["llama3-1b", "wide"])
@pytest.mark.parametrize("B,S", [(1, 0), (2, 0), (9, 0), (32, 0), (1, 1), (1, 32),
                                 (3, 7), (33, 0)])
@pytest.mark.parametrize("odd", [None, 0, 1])
def test_layers_of_few_rows_from_one_call(lib, name, B, S, odd, monkeypatch):
    import dataclasses
    from fei_amd.engine.config import get_spec
    from fei_amd.models.llama import LlamaModel
    sizes = dict(hidden_size=2112, num_heads=8, num_kv_heads=4, head_dim=128,
                 intermediate_size=448) if name == "wide" else {}
    spec = dataclasses.replace(get_spec("llama3-1b"), num_layers=3, vocab_size=512,
                               **sizes)
    m = LlamaModel(spec, torch.device(DEV), torch.bfloat16, seed=1,
                   max_seq_len=640)
    if odd is not None:
        w = m.layers[odd].wdown
        m.layers[odd].wdown = torch.cat([w, w], 1)[:, :w.shape[1]]
    toks = torch.randint(0, 512, (B, S) if S else (B,), device=DEV)
    pos = torch.arange(B, dtype=torch.int32, device=DEV) * 13 % 500
    new = randbf(3, B, spec.num_kv_heads, 640, m.D, seed=2)
    done, few = [], lib.llama_few

    def run(one_call):
        monkeypatch.setattr(lib, "llama_few", lambda *a, **k: done.append(
            few(*a, **k) if one_call else (0, None)) or done[-1])
        kc, vc = new.clone(), -new
        if S:
            return m.forward_prefill(toks, pos, list(kc), list(vc)), kc, vc
        return m.forward_decode(toks, pos, list(kc), list(vc)), kc, vc
    for a, b in zip(run(True), run(False)):
        assert torch.equal(a, b)
    # the layers before the odd one; none where it is the first, whose weights say
    # whether this chain is taken at all
    assert [d for d, _ in done] == ([] if B > 32 or odd == 0
                                    else [3 if odd is None else odd, 0])


# splits that one kernel sums, and that the output product does, in contiguous caches and in
# pages, which lie as they happen to
@pytest.mark.parametrize("B", [1, 3])
@pytest.mark.parametrize("last", [130, 300, 639])
@pytest.mark.parametrize("paged", [False, True])
def test_few_rows_over_many_keys(lib, B, last, paged):
    import dataclasses
    from fei_amd.engine.config import get_spec
    from fei_amd.models.llama import LlamaModel
    spec = dataclasses.replace(get_spec("llama3-1b"), num_layers=3, vocab_size=512)
    m = LlamaModel(spec, torch.device(DEV), torch.bfloat16, seed=1, max_seq_len=640)
    pos = torch.arange(last, last - 13 * B, -13, dtype=torch.int32, device=DEV)
    shape = (B * 40, spec.num_kv_heads, 16, m.D) if paged else \
        (B, spec.num_kv_heads, 640, m.D)
    table = torch.randperm(B * 40, device=DEV).int().view(B, 40) if paged else None
    k, v = (randbf(3, *shape, seed=i) for i in (2, 3))
    h = randbf(B, spec.hidden_size, seed=4)
    eps = spec.norm_eps
    got, kc, vc = h.clone(), list(k.clone()), list(v.clone())
    # what no split has written is not read
    ws = [torch.full((B, spec.num_heads, 16, n), float("nan"), device=DEV)
          for n in (m.D, 2)]
    done, sums = lib.llama_few(got, m.layers, kc, vc, m.hq_l, eps, pos, m.rope, 16, ws,
                               table)
    assert done == 3 and got.isfinite().all()
    want, k1, v1 = h.clone(), list(k.clone()), list(v.clone())

    def attend(li, qkv):
        q, kn, vn = m._qkv_views(qkv, B)
        args = dict(splits=16, scale=m.D ** -0.5, k=kn, v=vn, table=m.rope)
        if paged:
            return lib.attn_decode_paged(q, k1[li], v1[li], table, pos, **args)
        return lib.attn_decode(q, k1[li], v1[li], pos, **args)
    want_sums = m.fused_layers(want, attend)
    if B > 1:
        assert torch.equal(got, want) and torch.equal(sums, want_sums)
        assert all(torch.equal(a, b) for a, b in zip(kc + vc, k1 + v1))
        return
    # the splits' sums are rounded once, by 2^-9, but in another order: a layer's
    # attention and the two residuals behind it, three times
    assert row_err(got, want.double()) < 3 * 3 ** 0.5 * 2.0 ** -9
    for a, b in zip(kc + vc, k1 + v1):
        assert row_err(a.flatten(), b.double().flatten()) < 2.0 ** -9
    assert torch.equal(kc[0], k1[0]) and torch.equal(vc[0], v1[0])


@pytest.mark.parametrize("B,S", [(1, 1), (1, 8), (2, 9), (1, 32)])
def test_few_prompt_rows_over_many_keys(lib, B, S, monkeypatch):
    """So many that they are cut, into what llama_few makes room for."""
    import dataclasses
    from fei_amd.engine.config import get_spec
    from fei_amd.models.llama import LlamaModel
    spec = dataclasses.replace(get_spec("llama3-1b"), num_layers=2, vocab_size=512)
    m = LlamaModel(spec, torch.device(DEV), torch.bfloat16, seed=1, max_seq_len=2048)
    assert lib._prefill_splits(B, spec.num_kv_heads, 4 * S, 2048) > 1
    toks = torch.randint(0, 512, (B, S), device=DEV)
    pos0 = 1900 - 300 * torch.arange(B, dtype=torch.int32, device=DEV)
    k, v = (randbf(2, B, spec.num_kv_heads, 2048, m.D, seed=i) for i in (2, 3))
    few = lib.llama_few

    def run(one_call):
        kc, vc, done = list(k.clone()), list(v.clone()), []
        monkeypatch.setattr(lib, "llama_few", lambda *a, **b: done.append(
            few(*a, **b) if one_call else (0, None)) or done[-1])
        y = m.forward_prefill(toks, pos0, kc, vc)
        assert [d for d, _ in done] == [2 if one_call else 0]
        return [y, *kc, *vc]
    for a, b in zip(run(True), run(False)):
        assert a.isfinite().all() and torch.equal(a, b)


@pytest.mark.parametrize("B", [1, 3])
def test_workspace_of_a_decoding_step(lib, B):
    """More entries than the two that attention takes make no difference, nor does
    what lies there; too small a one is refused."""
    import dataclasses
    from fei_amd.engine.config import get_spec
    from fei_amd.models.llama import LlamaModel
    spec = dataclasses.replace(get_spec("llama3-1b"), num_layers=2, vocab_size=512)
    m = LlamaModel(spec, torch.device(DEV), torch.bfloat16, seed=1, max_seq_len=640)
    toks = torch.randint(0, 512, (B,), device=DEV)
    pos = torch.arange(B, dtype=torch.int32, device=DEV) * 90 + 300
    k, v = (randbf(2, B, spec.num_kv_heads, 640, m.D, seed=i) for i in (2, 3))

    def run(ws, splits=16):
        return m.forward_decode(toks, pos, list(k.clone()), list(v.clone()),
                                attn_splits=splits, workspace=ws)
    ws = [torch.full((B, spec.num_heads, 16, n), float("nan"), device=DEV)
          for n in (m.D, 2)]
    more = torch.zeros(7, dtype=torch.int32, device=DEV)
    want = run(None)
    assert want.isfinite().all()
    for w in (ws, (*ws, more), [*ws, more, None]):
        assert torch.equal(run(w), want)
    with pytest.raises(AssertionError):
        run(ws, 32)


# in parts and by whole products, up to the rows that the last layer's kernels for few
# take, and one more
@pytest.mark.parametrize("layers", [1, 2])
@pytest.mark.parametrize("B,S", [(1, 33), (2, 65), (1, 300), (3, 257), (32, 2), (32, 9),
                                 (33, 9), (5, 1)])
def test_last_layer_of_a_prompt(lib, B, S, layers):
    import dataclasses
    from fei_amd.engine.config import get_spec
    from fei_amd.models.llama import LlamaModel
    spec = dataclasses.replace(get_spec("llama3-1b"), num_layers=layers,
                               vocab_size=512)
    m = LlamaModel(spec, torch.device(DEV), torch.bfloat16, seed=1,
                   max_seq_len=640)
    toks = torch.randint(0, 512, (B, S), device=DEV)
    pos0 = torch.arange(B, dtype=torch.int32, device=DEV) * 3
    new = randbf(layers, B, spec.num_kv_heads, 640, m.D, seed=2)

    def run(everything):
        kc, vc = new.clone(), -new
        y = m.forward_prefill(toks, pos0, list(kc), list(vc),
                              all_positions=everything)
        return y[:, -1] if everything else y, kc, vc
    (a, ka, va), (b, kb, vb) = run(False), run(True)
    assert a.shape == b.shape
    # one layer's roundings, 2^-9 each, fall otherwise
    assert row_err(a, b.double()) < 2.0 ** -6
    assert torch.equal(ka, kb) and torch.equal(va, vb)


@pytest.mark.parametrize("B,S,taken", [(1, 64, False), (1, 65, True), (2, 32, False),
                                       (32, 7, False), (9, 8, True), (1, 300, True),
                                       (33, 9, False), (4, 8, False)])
def test_when_a_prompts_last_rows_are_taken_out(lib, B, S, taken, monkeypatch):
    """Of enough rows for the launches that it costs."""
    import dataclasses
    from fei_amd.engine.config import get_spec
    from fei_amd.models.llama import LlamaModel
    spec = dataclasses.replace(get_spec("llama3-1b"), num_layers=2, vocab_size=512)
    m = LlamaModel(spec, torch.device(DEV), torch.bfloat16, seed=1, max_seq_len=320)
    called, finish = [], m._finish
    monkeypatch.setattr(m, "_finish", lambda *a: called.append(1) or finish(*a))
    toks = torch.randint(0, 512, (B, S), device=DEV)
    pos0 = torch.zeros(B, dtype=torch.int32, device=DEV)
    kc, vc = (list(randbf(2, B, spec.num_kv_heads, 320, m.D, seed=i)) for i in (2, 3))
    got = m.forward_prefill(toks, pos0, kc, vc)
    assert bool(called) == taken
    if not taken and B * S > 64:
        # the head's product of the last rows alone may take another kernel
        want = m.forward_prefill(toks, pos0, kc, vc, all_positions=True)[:, -1]
        assert row_err(got, want.double()) < 2.0 ** -7


@pytest.mark.parametrize("B,S,lengths", [(1, 4, None), (1, 24, None),
                                         (4, 8, [8, 1, 3, 5]), (2, 16, [16, 9]),
                                         (32, 1, None), (1, 33, None),
                                         (3, 50, [50, 1, 20]), (1, 300, None),
                                         # tiles enough without parts of K
                                         (2, 350, [350, 17]), (2, 512, None),
                                         (5, 205, None)])   # layer by layer
def test_encoder_layers_from_one_call(lib, B, S, lengths, monkeypatch):
    from fei_amd.models.bge import BgeEncoder
    m = BgeEncoder(device=torch.device(DEV))
    ids = torch.randint(0, 1000, (B, S), device=DEV)
    n = None if lengths is None else torch.tensor(lengths, device=DEV)
    # what one launch, or the rows that texts have, would run
    monkeypatch.setattr(lib, "encoder_one", lambda *a: None)
    monkeypatch.setattr(lib, "encoder_packed", lambda *a: None)
    ran, layers = [], lib.encoder_layers
    monkeypatch.setattr(lib, "encoder_layers", lambda *a: ran.append(layers(*a)) or ran[-1])
    got = m.encode_ids(ids, n)
    assert [r is not None for r in ran] == [B * S <= lib.ENCODER_ROWS]
    monkeypatch.setattr(lib, "encoder_layers", lambda *a: None)
    want = m.encode_ids(ids, n)
    if not 32 < B * S <= lib.ENCODER_ROWS:   # the same kernels in the same order
        assert torch.equal(got, want)
    else:
        # 8 roundings a layer, 2^-9 / sqrt(3) each, that differ on either side:
        # sqrt(2 * 96) of them make 0.016; twice that
        assert row_err(got, want.double()) < 2.0 ** -5


@pytest.mark.parametrize("B,S", [(3, 1), (1, 8), (1, 9), (2, 8), (1, 17), (5, 5)])
@pytest.mark.parametrize("heads,inner", [(12, 3072), (1, 64), (16, 128)])
def test_encoder_norms_inside_products(lib, B, S, heads, inner, monkeypatch):
    """Up to 24 rows: the same sums in the same order as with a launch for each
    norm, at the edges of the rows, and of widths that leave lanes without columns
    or a wave without steps."""
    import dataclasses
    from fei_amd.engine.config import get_spec
    from fei_amd.models.bge import BgeEncoder
    C = heads * 64
    spec = dataclasses.replace(get_spec("bge-base"), num_layers=3, num_heads=heads,
                               num_kv_heads=heads, hidden_size=C,
                               intermediate_size=inner)
    m = BgeEncoder(spec, device=torch.device(DEV))
    for i, lw in enumerate(m.layers):
        for n in ("ln1_w", "ln2_w"):
            lw[n].copy_(1 + randbf(C, seed=i) * 0.2)
        for n in ("bqkv", "bo", "bi", "bo2", "ln1_b", "ln2_b"):
            lw[n].copy_(randbf(lw[n].numel(), seed=i + 9) * 0.1)
    ids = torch.randint(0, 1000, (B, S), device=DEV)
    monkeypatch.setattr(lib, "encoder_one", lambda *a: None)
    ran, layers = [], lib.encoder_layers
    monkeypatch.setattr(lib, "encoder_layers", lambda *a: ran.append(layers(*a)) or ran[-1])
    got = m.encode_ids(ids)
    assert len(ran) == 1 and ran[0] is not None
    monkeypatch.setattr(lib, "encoder_layers", lambda *a: None)
    want = m.encode_ids(ids)
    assert got.isfinite().all() and torch.equal(got, want)


@pytest.mark.parametrize("B,S,C", [(1, 1, 8), (2, 3, 512), (5, 7, 520), (3, 9, 768),
                                   (1, 512, 1032), (2, 2, 2048)])
def test_embedding_and_its_norm(lib, B, S, C):
    """The bits of a look-up, a sum and a norm; what it does not read as it lies goes
    there, and positions that there are not are refused as they were."""
    ids = torch.randint(0, 100, (B, S), device=DEV)
    ids[0, 0], ids[-1, -1] = 99, 0
    tok, pos = randbf(100, C, seed=1), randbf(512, C, seed=2)
    w, b = 1 + 0.1 * randbf(C, seed=3), randbf(C, seed=4)
    want = lib.layernorm(torch.nn.functional.embedding(ids, tok) + pos[:S], w, b, 1e-6)
    args = (w, b, 1e-6, torch.bfloat16)
    assert lib._embedding_ok(ids, tok, pos, w, b)
    assert torch.equal(lib.embed_layernorm(ids, tok, pos, *args), want)
    wide = torch.cat([tok, tok], 1)[:, :C]
    assert not lib._embedding_ok(ids, wide, pos, w, b)
    assert torch.equal(lib.embed_layernorm(ids, wide, pos, *args), want)
    if S > 1:
        with pytest.raises(RuntimeError):
            lib.embed_layernorm(ids, tok, pos[:S - 1] if S > 2 else pos[:0], *args)


@pytest.mark.parametrize("B,S,lengths", [
    (3, 214, [214, 0, 1]), (9, 77, [77, 76, 64, 65, 1, 0, 13, 500, -3]),
    (2, 512, [1, 512]), (1500, 2, None),         # tiles of 64 x 64
    (64, 50, None), (40, 200, None), (7, 512, [512, 0, 0, 0, 0, 0, 129])])
def test_encoder_of_the_rows_that_texts_have(lib, B, S, lengths):
    """Against all rows with padding; a length is taken at 0 and S where it is less
    or more, and nobody is asked for the rows behind it."""
    from fei_amd.models.bge import BgeEncoder
    m = BgeEncoder(device=torch.device(DEV))
    g = torch.Generator().manual_seed(B)
    if lengths is None:
        lengths = torch.randint(0, S + 1, (B,), generator=g).tolist()
    ids = torch.randint(0, 1000, (B, S), generator=g).to(DEV)
    n = torch.tensor(lengths, device=DEV)
    called = []
    packed, lib.encoder_packed = lib.encoder_packed, \
        lambda *a: called.append(packed(*a)) or called[-1]
    try:
        got = m.encode_ids(ids, n)
        lib.encoder_packed = lambda *a: None
        want = m.encode_ids(ids, n.clamp(0, S))
    finally:
        lib.encoder_packed = packed
    assert called[0] is not None
    empty = n <= 0
    assert not got[empty].any()
    # as between the paths for all rows
    assert row_err(got[~empty], want[~empty].double()) < 2.0 ** -5
    assert got.isfinite().all()


@pytest.mark.parametrize("B,S", [(20, 40), (64, 60)])    # both kinds of tiles
@pytest.mark.parametrize("heads,inner", [(1, 64), (2, 192), (3, 128)])
def test_narrow_encoder_of_the_rows_that_texts_have(lib, B, S, heads, inner):
    """A K of one to three steps, which no part of K is cut from."""
    import dataclasses
    from fei_amd.engine.config import get_spec
    from fei_amd.models.bge import BgeEncoder
    spec = dataclasses.replace(get_spec("bge-base"), num_layers=3, num_heads=heads,
                               num_kv_heads=heads, hidden_size=heads * 64,
                               intermediate_size=inner)
    m = BgeEncoder(spec, device=torch.device(DEV))
    ids = torch.randint(0, 1000, (B, S), device=DEV)
    n = torch.arange(B, device=DEV) * 7 % S + 1
    called = []
    packed, lib.encoder_packed = lib.encoder_packed, \
        lambda *a: called.append(packed(*a)) or called[-1]
    try:
        got = m.encode_ids(ids, n)
        lib.encoder_packed = lambda *a: None
        want = m.encode_ids(ids, n)
    finally:
        lib.encoder_packed = packed
    assert called[0] is not None
    # as between the paths for all rows
    assert row_err(got, want.double()) < 2.0 ** -5


@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("M,N,K", [(33, 4, 64), (64, 768, 3072), (65, 100, 128),
                                   (500, 2304, 768)])
def test_rows_bias(lib, gelu, M, N, K):
    from fei_amd.ops import rows
    x, w, b = randbf(M, K, seed=M), randbf(N, K, seed=N, scale=K ** -0.5), \
        randbf(N, seed=1)
    out = torch.full((M, N), float("nan"), device=DEV, dtype=torch.bfloat16)
    rows._lib().fei_rows_bias(*(t.data_ptr() for t in (out, x, w, b)), M, N, K,
                              int(gelu), rows._stream())
    want = x.double() @ w.double().t() + b.double()
    if gelu:
        want = torch.nn.functional.gelu(want)
    assert row_err(out, want) < 2.0 ** -8


# -- grouped products ------------------------------------------------------------

@pytest.mark.parametrize("T,E,top,N,K", [
    (300, 4, 2, 512, 256),       # 128 columns, three buffers
    (2000, 16, 4, 768, 128),     # 192, three
    (2000, 16, 4, 2048, 64),     # 128, two
    (2000, 16, 4, 1344, 192),    # 192, two
    (400, 3, 1, 20, 320),        # a part of a block, steps that do not divide
])
def test_moe_gemm_blocks(lib, T, E, top, N, K):
    """Each size of block of the grouped product, with experts that have more
    and fewer rows than their share."""
    from fei_amd.ops import mixers as mx
    n = T * top
    x, w = randbf(T, K, seed=T), randbf(E, N, K, seed=N, scale=K ** -0.5)
    g = torch.Generator(device=DEV).manual_seed(2)
    score = torch.randn(T, E, generator=g, device=DEV)
    score[:, 0] += 0.3
    ids = score.topk(top, 1).indices.int().contiguous()
    most = min(n, n // 128 + E)
    likely = min(most, E * -(-n // (E * 128)))
    order, place = (torch.empty(n, dtype=torch.int32, device=DEV)
                    for _ in range(2))
    tiles = torch.empty(most, 3, dtype=torch.int32, device=DEV)
    count = torch.empty(1, dtype=torch.int32, device=DEV)
    p, st, lb = mx._p, mx._stream(), mx._lib()
    lb.fei_moe_plan(p(order), p(place), p(tiles), p(count), p(ids), n, E, top,
                    128, most, st)
    out = torch.full((n, N), float("nan"), device=DEV, dtype=torch.bfloat16)
    lb.fei_moe_gemm(p(out), p(x), p(w), p(order), p(tiles), p(count), most,
                    likely, N, K, 0, 2, st)
    want = torch.empty(T, top, N, dtype=torch.float64, device=DEV)
    for e in range(E):
        t, k = (ids == e).nonzero(as_tuple=True)
        want[t, k] = x[t].double() @ w[e].double().t()
    got = out[place.view(T, top).long()]
    assert row_err(got.view(n, N), want.view(n, N)) < 2.0 ** -8


# -- gated linear attention over prompts ---------------------------------------------

@pytest.mark.parametrize("dim,vdim", [
    (16, 40), (32, 100), (64, 256), (128, 300), (128, 33), (136, 64),
    (200, 256), (256, 512), (30, 510), (128, 256),
])
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2e-5),
                                       (torch.bfloat16, 2.0 ** -8)])
def test_gla_prompt_tiles(lib, dim, vdim, dtype, tol):
    """Each count of column tiles a block takes at once, the last ones in part,
    against the recurrence token by token on the CPU. float32: sums of 256
    terms and 16 ulp of the exponentials; bfloat16: one rounding."""
    from types import SimpleNamespace as NS
    from fei_amd.ops import mixers as mx
    H, rank = 2, 8
    parts = [(0, 70, 0), (70, 64, 0), (134, 1, 0)]
    T = 135
    g = torch.Generator().manual_seed(dim + vdim)
    rand = lambda *s: torch.randn(*s, generator=g)
    m = NS(heads=H, dim=dim, vdim=vdim, gate_rank=rank, tau=8.0)
    w = NS(a2=rand(H * dim, rank) * 0.3, bias=rand(H * dim),
           norm=rand(vdim).abs() + 0.5, eps=1e-5)
    proj = rand(T, 2 * H * dim + 2 * H * vdim + rank).to(dtype)
    chunks, spans = [], []
    for i, (row, n, pos0) in enumerate(parts):
        spans.append([len(chunks), -(-n // 64), pos0, i])
        chunks += [[i, row + a, min(64, n - a)] for a in range(0, n, 64)]

    def run(dev):
        up = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)
        batch = NS(portions=parts, n_dec=0, slots=up([2, 0, 1]),
                   chunk_plan=lambda: (up(chunks), up(spans)))
        out = torch.zeros(T, H * vdim, dtype=dtype, device=dev)
        states = torch.ones(4, H, vdim, dim, device=dev)
        mx.gla_prefill(proj.to(dev), out, m,
                       NS(**{k: v.to(dev) if torch.is_tensor(v) else v
                             for k, v in vars(w).items()}), batch, states)
        return out.cpu(), states.cpu()
    (got, s), (want, s0) = run(DEV), run("cpu")
    assert row_err(got, want.double()) < tol * (1 if dtype == torch.float32 else 2)
    assert row_err(s[:3].flatten(1), s0[:3].double().flatten(1)) < 2e-5
    assert bool((s[3] == 1).all())


@pytest.mark.parametrize("B", [1, 3, 70])
@pytest.mark.parametrize("H,dim,vdim,rank", [(1, 16, 40, 8), (3, 30, 33, 16),
                                             (8, 128, 256, 16), (2, 256, 512, 32)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gla_tokens_beside_prompts(lib, B, H, dim, vdim, rank, dtype):
    """One call for both gives the bits of a call for each."""
    from types import SimpleNamespace as NS
    from fei_amd.ops import mixers as mx
    parts = [(B, 70, 0), (B + 70, 2, 5), (B + 72, 64, 9)]
    T = B + 136
    g = torch.Generator(device=DEV).manual_seed(dim + B)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    up = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    m = NS(heads=H, dim=dim, vdim=vdim, gate_rank=rank, tau=8.0)
    w = NS(a2=rand(H * dim, rank) * 0.3, bias=rand(H * dim), norm=rand(vdim), eps=1e-5)
    proj = rand(T, 2 * H * dim + 2 * H * vdim + rank).to(dtype)
    chunks, spans = [], []
    for i, (row, n, pos0) in enumerate(parts):
        spans.append([len(chunks), -(-n // 64), pos0, B + i])
        chunks += [[i, row + a, min(64, n - a)] for a in range(0, n, 64)]
    slots = torch.randperm(B + 4, generator=g, device=DEV)[:B + 3].int()
    pos = torch.arange(T, device=DEV).int()      # the first token starts its sequence
    batch = NS(portions=parts, n_dec=B, slots=slots, pos=pos,
               chunk_plan=lambda: (up(chunks), up(spans)))
    states = rand(B + 4, H, vdim, dim)
    outs, mems = ([x.clone() for _ in range(2)]
                  for x in (torch.zeros(T, H * vdim, dtype=dtype, device=DEV), states))
    mx.gla_mixed(proj, outs[0], m, w, batch, mems[0])
    mx.gla_decode(proj[:B], outs[1][:B], m, w, batch, mems[1])
    mx.gla_prefill(proj, outs[1], m, w, batch, mems[1])
    assert torch.equal(*outs) and torch.equal(*mems)
    assert not torch.equal(mems[0], states)


# -- latent attention of tokens and prompts --------------------------------------------

@pytest.mark.parametrize("B", [1, 5, 600])
@pytest.mark.parametrize("H,dim,rot,vdim,rank,window", [
    (1, 24, 8, 20, 40, None), (3, 30, 6, 33, 67, 50), (16, 128, 64, 128, 512, 100),
    (20, 64, 32, 64, 256, None)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_latent_tokens_beside_prompts(lib, B, H, dim, rot, vdim, rank, window, dtype):
    """One call for both gives the bits of a call for each."""
    from types import SimpleNamespace as NS
    from fei_amd.engine.step import RaggedBatch
    from fei_amd.ops import mixers as mx
    g = torch.Generator(device=DEV).manual_seed(dim + B)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    up = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    new = [1] * B + [70, 2, 130]
    lens = [1 + 37 * i % 160 for i in range(B)] + [70, 159, 150]
    row = [sum(new[:i]) for i in range(B, B + 3)]
    T, S, W = sum(new), B + 3, 10
    m = NS(heads=H, dim=dim, rot_dim=rot, vdim=vdim, kv_rank=rank, window=window,
           scale=dim ** -0.5, row_width=rank + rot)
    ukv = (rand(H * (dim + vdim), rank) * rank ** -0.5).to(dtype)
    w = NS(uk=ukv[:H * dim], uv=ukv[H * dim:], ukv=ukv, norm=rand(rank), eps=1e-5)
    angles = rand(160, rot // 2)
    rotab = torch.stack([angles.cos(), angles.sin()], -1).flatten(1).contiguous()
    batch = RaggedBatch(
        tokens=torch.zeros(T, dtype=torch.int64, device=DEV),
        pos=up([p for n, c in zip(lens, new) for p in range(n - c, n)]),
        row_seq=up([i for i, c in enumerate(new) for _ in range(c)]),
        table=torch.randperm(S * W, generator=g, device=DEV).int().view(S, W),
        slots=up(list(range(S))), n_dec=B,
        portions=[(r, new[B + i], lens[B + i] - new[B + i]) for i, r in enumerate(row)])
    proj = rand(T, H * (dim + rot) + rank + rot + H * vdim).to(dtype)
    cache = rand(S * W * 16, rank + rot).to(dtype)
    outs, mems, projs = ([x.clone() for _ in range(2)] for x in (
        torch.zeros(T, H * vdim, dtype=dtype, device=DEV), cache, proj))
    mx.latent_attn_mixed(projs[0], outs[0], m, w, rotab, batch, mems[0], 16)
    args = (m, w, rotab, batch, mems[1], 16)
    mx.latent_attn_decode(projs[1][:B], outs[1][:B], *args)
    mx.latent_attn_prefill(projs[1], outs[1], *args)
    assert torch.equal(*mems) and torch.equal(*projs) and torch.equal(*outs)
    assert not torch.equal(mems[0], cache) and bool(outs[0].isfinite().all())


# -- largest values ----------------------------------------------------------------

@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,V", [(1, 1), (3, 7), (20, 128256), (2, 2049),
                                 (600, 64), (5, 50257), (65535, 3), (65536, 3)])
def test_argmax_is_the_first(lib, dtype, B, V):
    """Ties, infinities, NaN and zeros of both signs."""
    g = torch.Generator(device=DEV).manual_seed(V)
    x = torch.randn(B, V, generator=g, device=DEV).to(dtype)
    rows = [x, (x * 2).round(), -x.abs() * 0.0, torch.full_like(x, -float("inf"))]
    y = x.clone()
    y[:, V // 2:] = float("nan")
    z = x.clone()
    z[:, V // 3] = float("inf")
    for t in (*rows, y, z):
        got = lib.argmax(t)
        assert got.dtype == torch.int64
        # argmax of the CPU: the first of equals, NaN above all
        assert torch.equal(got.cpu(), t.float().cpu().argmax(-1))


@pytest.mark.parametrize("M,C,p", [(1, 8, 1), (5, 512, 3), (70, 768, 8),
                                   (66, 1024, 2), (9, 1032, 5), (6, 2048, 4)])
def test_parts_layernorm(lib, M, C, p):
    from fei_amd.ops import rows
    parts = torch.randn(p, M, C, device=DEV)
    bias, res, gain, shift = (randbf(*s, seed=i) for i, s in enumerate(
        ((C,), (M, C), (C,), (C,))))
    out = torch.full((M + 1, C), float("nan"), device=DEV, dtype=torch.bfloat16)
    rows._lib().fei_parts_layernorm(
        out.data_ptr(), parts.data_ptr(), p, bias.data_ptr(), res.data_ptr(),
        gain.data_ptr(), shift.data_ptr(), M, C, 1e-6, rows._stream())
    x = parts.double().sum(0) + bias.double() + res.double()
    want = torch.nn.functional.layer_norm(x, (C,), gain.double(),
                                          shift.double(), 1e-6)
    assert row_err(out[:M], want) < 2.0 ** -8
    assert bool(out[M].isnan().all())


@pytest.mark.parametrize("B,S,C,lens", [
    (1, 1, 8, [1]), (3, 7, 768, [7, 0, 3]), (2, 513, 768, [513, 200]),
    (2, 40, 2048, [40, 99]), (5, 9, 1032, [9, 1, 2, -3, 5]), (1, 300, 64, [300]),
])
def test_pool_unit(lib, B, S, C, lens):
    """Rows past a length, or past the text, do not count; no row: zeros."""
    h = randbf(B, S, C, seed=S)
    got = lib.pool_unit(h, torch.tensor(lens, dtype=torch.int32, device=DEV))
    for b, n in enumerate(lens):
        x = h[b, :max(n, 0)].double()
        want = torch.nn.functional.normalize(
            x.sum(0) / max(x.shape[0], 1), dim=0)
        # float32 sums of up to 513 terms, the partial ones short
        assert float((got[b] - want).norm()) < 1e-5
        assert n > 0 or not got[b].any()


def test_pool_unit_keeps_nan_and_inf(lib):
    """As in torch: a NaN in one column makes a text's whole result NaN, an
    infinity the others zero; texts beside it are as without."""
    h = randbf(4, 9, 768, seed=1)
    h[1, 3, 5], h[2, 8, 700] = float("nan"), float("inf")
    h[3, 4, 0] = float("nan")                       # past the length
    lens = torch.tensor([9, 9, 9, 4], dtype=torch.int32, device=DEV)
    got = lib.pool_unit(h, lens)
    assert got[1].isnan().all()
    assert got[2, 700].isnan() and not got[2, :700].any() \
        and not got[2, 701:].any()
    for b in (0, 3):
        want = torch.nn.functional.normalize(
            h[b, :lens[b]].double().mean(0), dim=0)
        assert float((got[b] - want).norm()) < 1e-5
