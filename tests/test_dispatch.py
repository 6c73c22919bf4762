"""Which calls the kernels for few rows take: those whose tensors are what the
kernels read through a bare pointer. The others get what the library gives."""

import subprocess
import sys

import pytest
import torch

from fei_amd import ops
from fei_amd.ops import mixers as mx
from fei_amd.ops import rows

DEV = "cuda:0"


def rand(*shape, seed=0, dev="cpu", dtype=torch.bfloat16, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dev, dtype)


def row_err(got, want):
    d = (got.double() - want).norm(dim=-1)
    return float((d / want.norm(dim=-1).clamp_min(1e-30)).max())


@pytest.mark.parametrize("T", [3, 9, 32])
def test_few_rows_want_plain_tensors(T):
    K, N = 128, 64
    x, w = rand(T, K), rand(N, K)
    assert mx.plain(x, w) and mx.skinny_ok(T, K, x, w)
    assert mx._gemv_rows(8, K, rand(8, K), w)
    wide = rand(T, 2 * K)
    leaf = rand(N, K).requires_grad_()
    for a, b in [(wide[:, K:], w),                  # columns of a wider buffer
                 (x.t().contiguous().t(), w),       # columns first
                 (x, rand(N, 2 * K)[:, :K]),
                 (x, rand(K, N).t()),
                 (x.float(), w), (x, w.half()), (x.float(), w.float()),
                 (x, rand(N, K + 64)), (x, w[0]),   # sizes that do not fit
                 (x, leaf)]:                        # a gradient is asked for
        assert not mx.plain(a, b)
        assert not mx.skinny_ok(T, K, a, b)
        assert not mx._gemv_rows(8, K, a, b)
    with torch.no_grad():
        assert mx.plain(x, leaf)


@pytest.mark.parametrize("M", [1, 3, 5, 8, 32])
def test_products_want_plain_weights(M):
    """Which kernel, if any; it needs no GPU to say so."""
    for K, how in ((128, "gemv" if M == 1 else "skinny"),
                   (72, "gemv" if M in (1, 3, 8) else None), (70, None)):
        x, w = rand(M, K), rand(48, K)
        assert ops._kernel_for(x, w, M, K) == how
        assert ops._kernel_for(rand(M, 2 * K)[:, K:], w, M, K) == how
        leaf = rand(48, K).requires_grad_()
        for a, b in [(x.float(), w.float()), (x.half(), w.half()),
                     (x.float(), w), (x, rand(K, 48).t()), (x, leaf),
                     (x, rand(48, 2 * K)[:, :K]), (x, rand(48, K + 8)),
                     (x, w[0])]:
            assert ops._kernel_for(a, b, M, K) is None
        with torch.no_grad():
            assert ops._kernel_for(x, leaf, M, K) == how
    out = rand(M, 48)
    assert ops._fits(None, x, M * 48) and ops._fits(out, x, M * 48)
    for bad in (out.float(), rand(M, 49), rand(M, 96)[:, :48] if M > 1 else rand(2, 48)):
        assert not ops._fits(bad, x, M * 48)


def test_gains_in_lds_are_aligned():
    K, sums = 128, torch.zeros(4, 8)
    buf = torch.zeros(K + 8, dtype=torch.bfloat16)
    assert buf.data_ptr() % 16 == 0
    for at, inside in ((0, True), (1, False), (2, False), (4, False), (8, True)):
        assert ops._norm_inside("skinny", 4, K, sums, buf[at:at + K]) == inside
        assert ops._norm_inside("gemv", 4, K, None, buf[at:at + K])
    assert not ops._norm_inside("skinny", 4, K, None, buf[:K])


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 3, 8, 32])
@pytest.mark.parametrize("shift", [0, 1, 4])
def test_gains_anywhere(M, shift):
    K, N = 256, 64
    x, h = rand(M, K, seed=1, dev=DEV), rand(M, K, seed=2, dev=DEV)
    w0 = rand(K, K, seed=3, dev=DEV, scale=K ** -0.5)
    w = rand(N, K, seed=4, dev=DEV, scale=K ** -0.5)
    gain = (1 + 0.2 * rand(K + 8, seed=5, dev=DEV))[shift:shift + K]
    sums = ops.add_product(x, w0, h)
    h64 = h.double()
    y = (h64 * (h64.pow(2).mean(-1, keepdim=True) + 1e-5).rsqrt()
         * gain.double()) @ w.double().t()
    # rows rounded under their gains, results once more
    assert row_err(ops.gemv_norm(h, gain, w, 1e-5, sums=sums), y) < 2 ** -7
    want = torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:]
    assert row_err(ops.gemv_swiglu_norm(h, gain, w, 1e-5, sums=sums),
                   want) < 2 ** -6


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 3, 5, 8, 9, 32, 40])
def test_products_of_other_types_and_layouts(M):
    F = torch.nn.functional
    K, N = 128, 96
    for dtype, tol in ((torch.float32, 1e-5), (torch.float16, 2 ** -10),
                       (torch.bfloat16, 2 ** -8)):
        make = dict(dev=DEV, dtype=dtype, scale=K ** -0.5)
        x = rand(M, K, seed=1, dev=DEV, dtype=dtype)
        for w in (rand(N, K, seed=2, **make), rand(K, N, seed=2, **make).t(),
                  rand(N, 2 * K, seed=2, **make)[:, K:]):
            y = x.double() @ w.double().t()
            assert row_err(ops.linear_decode(x, w), y) < tol
            wide = rand(M, 2 * N, seed=3, dev=DEV, dtype=dtype)
            for res in (wide[:, N:], wide[:, N:].contiguous()):
                left, want = wide[:, :N].clone(), res.double() + y
                # sums rounded before they are added, in the library
                ops.gemv_res(x, w, res)
                assert row_err(res, want) < 2 * tol
                assert torch.equal(wide[:, :N], left)
            b = rand(2 * N, seed=4, dev=DEV, dtype=dtype)
            for bias in (b[:N], b[::2]):
                got = ops.linear_bias(x, w, bias)
                assert row_err(got, y + bias.double()) < tol
            if dtype == torch.bfloat16:
                want = F.silu(y[:, :N // 2]) * y[:, N // 2:]
                # rounded once, in the library twice before
                assert row_err(ops.gemv_swiglu(x, w), want) < 2 ** -6
        for w in (w[:, :64].contiguous(), w.cpu().contiguous()):
            for call in (lambda: ops.linear_decode(x, w),
                         lambda: ops.linear_bias(x, w, b[:N]),
                         lambda: ops.gemv_swiglu(x, w)):
                with pytest.raises(RuntimeError):
                    call()
    leaf = w.to(DEV).requires_grad_()
    ops.linear_decode(x, leaf).sum().backward()
    assert row_err(leaf.grad, x.double().sum(0).expand(N, K)) < 2 ** -7


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 3, 4, 8, 9, 32, 40])
def test_views_of_few_rows(T):
    """Activations, weights and residuals that are column ranges of wider
    buffers: what contiguous copies give, nothing written beside them."""
    K, N, ff = 256, 96, 32
    wide = rand(T, 2 * K + 8, seed=1, dev=DEV)
    a = wide[:, 8:K + 8]
    w = rand(N, K, seed=2, dev=DEV, scale=K ** -0.5)
    ws = rand(N, 2 * K, seed=2, dev=DEV, scale=K ** -0.5)[:, K:]
    bias = rand(2 * N, seed=3, dev=DEV, dtype=torch.float32)
    for aa, ww in ((a, w), (a.contiguous(), ws), (a, ws),
                   (a.contiguous(), w)):
        y = aa.double() @ ww.double().t()
        buf = rand(T, 2 * N, seed=4, dev=DEV, dtype=torch.float32)
        for res in (buf[:, N:], buf[:, N:].contiguous()):
            left, want = buf[:, :N].clone(), res.double() + 0.5 * y
            got = mx.residual_linear(res, aa, ww, 0.5)
            # float32 sums of K products
            assert row_err(got, want) < 1e-5
            assert torch.equal(buf[:, :N], left)
        for b in (bias[:N], bias[::2]):
            assert row_err(mx.linear_f32(aa, ww, b), y + b.double()) < 1e-5
        assert row_err(mx.logits_head(aa, ww, 0.25, 3.0),
                       3 * torch.tanh(y * 0.25 / 3)) < 1e-5
        act = torch.zeros(T, 3 * ff, dtype=torch.bfloat16, device=DEV)
        n_mix = N - 2 * ff
        proj = mx.mix_in(aa, a, ww, n_mix, ff, act[:, ff:2 * ff])
        # rounded once (2^-9), a SwiGLU's sums before it too in the library
        assert row_err(proj, y[:, :n_mix]) < 2 ** -8
        g, u = (a.double() @ ww.double().t())[:, n_mix:].split(ff, 1)
        assert row_err(act[:, ff:2 * ff],
                       torch.nn.functional.silu(g) * u) < 2 ** -6
        assert not act[:, :ff].any() and not act[:, 2 * ff:].any()


@pytest.mark.parametrize("E,top,rows", [(16, 4, 128), (8, 2, 128), (4, 1, 32),
                                        (64, 8, 128)])
def test_tiles_to_expect(E, top, rows):
    """Against experts drawn by chance."""
    from fei_amd.ops.moe import likely_tiles
    g = torch.Generator().manual_seed(E)
    for T in (300, 500, 800, 900, 1000, 1500, 1908, 2048, 4000):
        n = T * top
        if n < 32 * E:
            continue
        seen = []
        for _ in range(30):
            ids = torch.rand(T, E, generator=g).topk(top, 1).indices.flatten()
            seen.append(int((-(-ids.bincount(minlength=E) // rows)).sum()))
        # the mean of 30, and that top choices of a row are never the same
        assert abs(likely_tiles(n, E, rows) - sum(seen) / 30) < 1 + 0.05 * E


@pytest.mark.parametrize("T", [64, 192, 1024])
@pytest.mark.parametrize("D", [64, 128])
def test_attn_decode_of_no_sequences_returns(D, T):
    """Whichever way as many positions would go; in a process of its own, which it
    would end. Nothing is launched, so it needs no GPU."""
    if not ops.kernels_available():
        pytest.skip("the kernels are not built")
    call = ("from fei_amd import ops; ops.require_lib().fei_attn_decode("
            "*[None] * 8, 0, 8, 2, {}, {}, 0, 0, 4, 1.0, 0, None, None, None, 0, "
            "None)").format(D, T)
    done = subprocess.run([sys.executable, "-c", call], capture_output=True,
                          text=True, timeout=300)
    assert done.returncode == 0, done


@pytest.mark.gpu
@pytest.mark.parametrize("T", [64, 192, 1024])
def test_attn_decode_of_an_empty_batch(T):
    q = rand(0, 8, 64, dev=DEV)
    pos = torch.zeros(0, dtype=torch.int32, device=DEV)
    kc = rand(0, 2, T, 64, dev=DEV)
    assert ops.attn_decode(q, kc, kc, pos, splits=4).shape == (0, 8, 64)
    pool = rand(4, 2, 16, 64, dev=DEV)
    table = torch.zeros(0, T // 16, dtype=torch.int32, device=DEV)
    assert ops.attn_decode_paged(q, pool, pool, table, pos,
                                 splits=4).shape == (0, 8, 64)
    torch.cuda.synchronize()
    with pytest.raises(AssertionError):      # what is refused stays so
        ops.attn_decode(q, kc, kc, pos, splits=65)


def encoder_shapes(C, HD, inner):
    return [(3 * HD, C), (3 * HD,), (C, HD), (C,), (C,), (C,),
            (inner, C), (inner,), (C, inner), (C,), (C,), (C,)]


def test_encoder_weights_have_their_sizes():
    """A kernel reads as much of them as the encoder's sizes say."""
    C, HD, inner = 128, 64, 192
    good = [rand(*s) for s in encoder_shapes(C, HD, inner) * 2]
    assert ops._encoder_weights(good, C, HD, inner) == [t.data_ptr() for t in good]
    for i, t in enumerate(good):
        for other in (t[..., :-8].contiguous(), t[:-8].contiguous(), t.float(),
                      torch.cat([t, t], -1)[..., :t.shape[-1]] if t.dim() == 2
                      else torch.stack([t, t], 1)[:, 0],
                      t.t().contiguous() if t.dim() == 2 else t[None],
                      rand(t.numel() + 1)[1:].view(t.shape)):
            bad = good[:i] + [other] + good[i + 1:]
            assert ops._encoder_weights(bad, C, HD, inner) is None, i
    assert ops._encoder_weights(good[:-1], C, HD, inner) is None


# with all rows in one native call, packed in both kinds of tiles, and layer by layer
@pytest.mark.gpu
@pytest.mark.parametrize("B,S,lengths", [(2, 30, True), (10, 80, True), (40, 80, True),
                                         (40, 80, False)])
@pytest.mark.parametrize("name", ["wqkv", "wo", "wi", "wo2"])
def test_encoder_weights_of_other_sizes_are_refused(B, S, lengths, name):
    from fei_amd.models.bge import BgeEncoder
    m = BgeEncoder(device=torch.device(DEV))
    ids = torch.zeros(B, S, dtype=torch.long, device=DEV)
    n = torch.full((B,), S, device=DEV) if lengths else None
    w = m.layers[-1][name]
    m.layers[-1][name] = w[:, :-64].contiguous()
    with pytest.raises(RuntimeError):
        m.encode_ids(ids, n)
    m.layers[-1][name] = w
    assert m.encode_ids(ids, n).isfinite().all()


def test_keys_beside_tokens_are_few():
    """What the tokens' launches prepare of the portions beside them: by bytes, by how
    many keys a block takes and by how long the tokens take; never past a grid."""
    from types import SimpleNamespace as NS
    m, wide = NS(heads=16, row_width=576), NS(heads=32, row_width=576)
    for spec, tokens, keys, pays in (
            (m, 1, 12000, True), (m, 4, 8000, True), (m, 4, 16000, False),
            (m, 5, 4000, True), (m, 64, 4000, True), (m, 8, 8000, False),
            (wide, 4, 16000, True), (wide, 4, 64000, False), (wide, 8, 8000, True),
            (wide, 256, 12000, False), (m, 0, 100, False), (m, 1024, 100, False),
            (NS(heads=16, row_width=320), 32, 8000, True),
            (NS(heads=16, row_width=1088), 32, 4000, False),
            (NS(heads=1, row_width=9), 1, 1 << 17, False)):
        assert mx._keys_beside(spec, tokens, 600, keys, 2) == pays, (spec, tokens, keys)
    assert not mx._keys_beside(m, 4, 600, 8000, 4)
    assert not mx._keys_beside(NS(heads=1, row_width=9), 1, 1 << 16, 100, 2)


def test_when_leaving_out_padding_pays():
    for M, texts, pays in (
            (1024, 1024, False), (900, 850, False), (900, 700, True),
            (1025, 1025, True), (2560, 2560, True),
            (3600, 3600, False), (4096, 3700, False), (6144, 5000, True),
            (8192, 8192, False), (9000, 9000, True), (12800, 12800, True),
            (16384, 16384, False), (16384, 15900, True), (32768, 32768, False),
            (32768, 0, True)):
        assert ops.encoder_packing_pays(M, texts, 3072) == pays, (M, texts)


@pytest.mark.gpu
@pytest.mark.parametrize("alike", [True, False])
def test_texts_of_one_length_are_not_packed(alike, monkeypatch):
    """The host knows the texts' lengths; either way they are the same embeddings."""
    from fei_amd.models.bge import BgeEncoder
    m = BgeEncoder(device=torch.device(DEV))
    texts = ["ab" * (45 if alike else 1 + i * 11 % 45) for i in range(40)]
    called, packed = [], ops.encoder_packed
    monkeypatch.setattr(ops, "encoder_packed",
                        lambda *a: called.append(1) or packed(*a))
    got = m.encode_texts(texts, batch_size=40)
    assert bool(called) != alike
    monkeypatch.setattr(ops, "encoder_packing_pays", lambda *a: alike)
    want = m.encode_texts(texts, batch_size=40)
    assert len(called) == 1
    # as between the paths for all rows
    assert row_err(got, want.double()) < 2.0 ** -5
