"""Which calls the kernels for few rows take: those whose tensors are what the
kernels read through a bare pointer. The others get what the library gives."""

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
