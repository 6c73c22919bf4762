"""Products of hundreds of rows (csrc/tile.hip) against float64."""

import pytest
import torch

from fei_amd import ops
from fei_amd.ops import mixers as mx
from fei_amd.ops import tiles

DEV = "cuda:0"
F = torch.nn.functional


def rand(*shape, seed=0, dev=DEV, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dev, torch.bfloat16)


def err(got, want):
    return float((got.double() - want).norm() / want.norm())


def test_what_tiles_take():
    """It needs no GPU to say so; CPU tensors are for torch."""
    x, w = rand(300, 128, dev="cpu"), rand(64, 128, dev="cpu")
    assert not tiles.tile_ok(300, x, w)
    for M in (129, 257, 300, 1301, 2048, 6006, 16384):
        for N, K in ((64, 64), (768, 768), (4096, 14336), (28672, 4096)):
            assert tiles.size_for(M, N, K) in [t[:2] for t in tiles.TILES]
            size, p = tiles.parts_for(M, N, K)
            assert size in [t[:2] for t in tiles.TILES] and 1 <= p <= 8
    # one full round of the CUs in tiles of 192 columns, not 3/4 of one of 256
    assert tiles.size_for(16384, 768, 768) == (256, 192)


@pytest.mark.parametrize("K", [64, 128, 192, 256, 320, 768, 3072])
def test_parts_of_any_k(K):
    """A part has 256 steps or all that there are."""
    for M, N in ((2, 64), (3073, 128), (4096, 192), (16384, 768), (131072, 2048)):
        assert 1 <= tiles.parts_up_to(M, N, K) <= max(1, min(8, K // 256))


def test_host_and_device_rank_tiles_by_the_same_times():
    """Parts of K are chosen on the host, the tiles that they run in on the device."""
    import os
    import re
    source = open(os.path.join(os.path.dirname(ops.__file__), "csrc", "tile.hip")).read()
    times = re.findall(r"= time\((\d+), (\d+), ([\d.]+)f, ([\d.]+)f\)", source)
    assert [tuple(map(float, t)) for t in times] == [
        t for t in tiles.TILES if t[1] > 128]
    # of a round, beside its steps
    assert "steps * alone + 3.f" in source
    assert tiles._time(1, 1, 64, 1, 256, 256, 0.0, 0.0) == 3.0


def test_when_activations_go_into_tiles():
    """Where those fill the CUs: not of few rows and results, whatever K."""
    for M, N, K in ((129, 8, 64), (300, 256, 4096), (1000, 1024, 1024), (8192, 64, 256),
                    (1000, 2048, 2048), (512, 6144, 4096), (700, 512, 8192),
                    (2048, 2048, 8192), (1301, 4096, 14336), (129, 28672, 4096)):
        assert tiles._rate(M, N, K) < (0.7 if K <= 8192 else 0.86)
    for M, N, K in ((16384, 3072, 768), (2048, 28672, 4096), (6006, 16384, 2048),
                    (1301, 12288, 2048), (1000, 6144, 4096), (4096, 4096, 14336)):
        assert tiles._rate(M, N, K) > (0.7 if K <= 8192 else 0.86)


def test_when_plain_products_pay():
    """Not where the library's own tiles fill the CUs."""
    for M, N, K, pays in ((8192, 16384, 1280, False), (4000, 8192, 2048, False),
                          (2048, 6144, 1024, False), (2048, 3072, 2048, False),
                          (3000, 6144, 1536, False), (300, 512, 2048, False),
                          (6006, 3072, 2048, True), (2600, 5000, 1024, True),
                          (1301, 5704, 2048, True), (4096, 2560, 1024, True)):
        assert tiles._plain_pays(M, N, K) == pays


def test_when_parts_of_k_pay():
    for M, N, K, pays in ((257, 992, 8192, False), (257, 1000, 8192, True),
                          (300, 4096, 14336, True), (8192, 1024, 8192, False),
                          (8192, 1024, 10240, True), (8191, 960, 14336, False),
                          (4096, 2048, 8192, False), (4096, 1792, 8192, True)):
        w = torch.empty(N, K, device="meta")
        assert tiles.parts_pay(M, w) == pays


def test_how_far_apart_rows_may_lie():
    """A lane's offset in bytes from a tile's first row has 32 bits, for up to 127 rows
    and 128 bytes."""
    w = torch.empty(64, 64, device="meta")
    for far in (64, 72, tiles.FAR - 8, tiles.FAR, tiles.FAR + 8, 1 << 26):
        x = torch.empty_strided((129, 64), (far, 1), device="meta")
        assert tiles._near(x, w) == (far < tiles.FAR)
        assert not tiles._near(x, w) or 127 * far * 2 + 128 < 1 << 32
    wide = torch.empty(8, tiles.FAR, device="meta")
    assert not tiles._near(wide[:129], wide)


@pytest.mark.gpu
def test_rows_far_apart():
    """Rows as far apart as tiles take them and further, which are the library's."""
    M, N, K = 257, 1024, 8192
    w = rand(N, K, seed=2, scale=K ** -0.5)
    near, res = rand(M, K, seed=1), rand(M, N, seed=3).float()
    y = near.double() @ w.double().t()
    for far in (tiles.FAR - 8, tiles.FAR):
        x = torch.empty_strided((M, K), (far, 1), device=DEV,
                                dtype=torch.bfloat16).copy_(near)
        assert tiles.tile_ok(M, x, w) == (far < tiles.FAR)
        # float32 sums of K products and one addition; a result rounded once
        assert err(mx.residual_linear(res.clone(), x, w),
                   res.double() + y) < 2 ** -24 * K ** 0.5
        assert err(mx.mix_in(x, None, w, N, 0, x), y) < 2 ** -9
        del x


# one step of K, an odd and an even number of them; one row and one 8 columns past a
# tile, and short of it; more tiles than CUs, with few steps each
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (256, 256, 64), (257, 264, 128), (191, 248, 192), (385, 776, 320),
    (1000, 1536, 1088), (5000, 4104, 64), (4100, 3080, 192)])
@pytest.mark.parametrize("size", [t[:2] for t in tiles.TILES])
def test_tile(M, N, K, size):
    # rows of x and out are ranges of wider ones; nothing is written beside them
    x = rand(M, K + 8, seed=1)[:, :K]
    w, b = rand(2 * N, K, seed=2, scale=K ** -0.5), rand(N, seed=3)
    y = x.double() @ w.double().t()
    u, g = y[:, N:], y[:, :N]
    # a result is rounded once, by 2^-9 at most, 0.3 of that in the mean; GELU's and
    # SwiGLU's own errors are float32's
    for epi, bias, want in (
            (tiles.TILE_BF16, None, g), (tiles.TILE_SWIGLU, None, F.silu(g) * u),
            (tiles.TILE_GELU, b, F.gelu(g + b.double())),
            (tiles.TILE_RELU2, None, g.clamp_min(0) ** 2)):
        wide = torch.full((M, N + 16), 7.0, device=DEV, dtype=torch.bfloat16)
        ww = w if epi == tiles.TILE_SWIGLU else w[:N]
        tiles._launch(wide[:, 8:N + 8], x, ww, N, epi, size, bias)
        assert err(wide[:, 8:N + 8], want) < 2 ** -9
        assert bool((wide[:, :8] == 7).all() and (wide[:, N + 8:] == 7).all())
    for p in (1, 2, 3, 5):
        if K // 64 < p:
            continue
        parts = torch.full((p, M, N), 7.0, device=DEV)
        tiles._launch(parts, x, w[:N], N, tiles.TILE_PARTS, size, None, p)
        # float32 sums of K terms in any order: 2^-24 sqrt(K) of their size and
        # less; 4e-7 seen
        assert err(parts.double().sum(0), g) < 2 ** -24 * max(K ** 0.5, 16)


# a few tiles more than the CUs have in whole rounds, which are run in halves: of rows
# where the last tile has rows for one half alone, and for more; of columns
@pytest.mark.gpu
@pytest.mark.parametrize("size,M,N", [((256, 256), 2400, 6664), ((256, 256), 2500, 6664),
                                      ((256, 192), 2400, 5192), ((192, 256), 2500, 4872),
                                      ((192, 256), 2500, 5000)])
@pytest.mark.parametrize("K", [64, 192, 1088])
def test_last_round_in_halves(size, M, N, K):
    x, w = rand(M, K, seed=1), rand(2 * N, K, seed=2, scale=K ** -0.5)
    y = x.double() @ w.double().t()
    for epi, want in ((tiles.TILE_BF16, y[:, :N]),
                      (tiles.TILE_SWIGLU, F.silu(y[:, :N]) * y[:, N:])):
        out = torch.full((M, N), 7.0, device=DEV, dtype=torch.bfloat16)
        tiles._launch(out, x, w if epi == tiles.TILE_SWIGLU else w[:N], N, epi, size)
        assert err(out, want) < 2 ** -9               # a result is rounded once


# each of the tiles that the device chooses from, short of the last row and past it
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(2500, 768, 192), (10336, 768, 64), (9000, 2304, 64),
                                   (10400, 3080, 128), (16000, 776, 1088)])
@pytest.mark.parametrize("count", [0, 1, 129, 0.4, 0.63, 1.0, 99999])
def test_rows_that_the_device_counts(M, N, K, count):
    x, w, b = rand(M, K, seed=1), rand(N, K, seed=2, scale=K ** -0.5), rand(N, seed=3)
    count = int(M * count) if isinstance(count, float) else count
    n, rows = min(count, M), torch.tensor([count], dtype=torch.int32, device=DEV)
    y = x[:n].double() @ w.double().t()

    def run(out, epi, parts=1):
        ops.require_lib().fei_tile_counted(
            out.data_ptr(), N, x.data_ptr(), K, w.data_ptr(), b.data_ptr(), M, N, K,
            epi, parts, rows.data_ptr(), ops._stream())
        assert bool((out[..., n:, :] == 7).all())
        return out[..., :n, :]
    for epi, want in ((tiles.TILE_BIAS, y + b.double()),
                      (tiles.TILE_GELU, F.gelu(y + b.double()))):
        got = run(torch.full((M, N), 7.0, device=DEV, dtype=torch.bfloat16), epi)
        assert n == 0 or err(got, want) < 2 ** -9     # a result is rounded once
    for p in (1, 2, 3):
        if K // 64 >= p:
            got = run(torch.full((p, M, N), 7.0, device=DEV), tiles.TILE_PARTS, p)
            # float32 sums in any order, as above
            assert n == 0 or err(got.double().sum(0), y) < 2 ** -24 * max(K ** 0.5, 16)


@pytest.mark.gpu
def test_activations_of_every_value():
    """All of bfloat16, and infinities and NaN that sums come to (as no factor, which
    would meet zeros): the bits of the library's product and the pass behind it, which
    divides."""
    every = torch.arange(1 << 16, dtype=torch.int32, device=DEV).to(torch.int16)
    every = every.view(torch.bfloat16)
    every = every[every.isfinite()]
    big = every.abs().max()
    M, K, N = len(every) + 4, 64, 16
    x = torch.zeros(M, K, device=DEV, dtype=torch.bfloat16)
    x[:-4, 0], x[:, 2] = every, 1.0
    x[-4, 0], x[-3, 0], x[-2, :2], x[-1, :2] = big, -big, big, -big
    w = torch.zeros(2 * N, K, device=DEV, dtype=torch.bfloat16)
    w[:N, 0] = 1.0
    w[8:N, 0], w[8:N, 1] = 2.0, -2.0         # infinities, and their difference
    w[N:, 2] = torch.tensor([1, -1, 0.5, 3, 1e30, 1e-30, 2.0 ** 100, 0] * 2)
    y = F.linear(x, w)
    assert y[-4, 8].isinf() and y[-2, 8].isnan() and y[-2, N:].isfinite().all()
    none = torch.zeros(N, device=DEV, dtype=torch.bfloat16)
    for epi, ww, want in (
            (tiles.TILE_BF16, w[:N], y[:, :N]),
            (tiles.TILE_SWIGLU, w, ops.swiglu(y)),
            (tiles.TILE_GELU, w[:N], ops.gelu(y[:, :N].contiguous())),
            (tiles.TILE_RELU2, w[:N], mx.ref.square_relu(y[:, :N]).bfloat16())):
        out = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
        tiles._launch(out, x, ww, N, epi, (256, 256), none)
        if epi == tiles.TILE_RELU2:          # a NaN is not above 0
            want = want.where(~y[:, :N].isnan(), torch.zeros_like(want))
        assert torch.equal(out.isnan(), want.isnan())
        ok = ~want.isnan()
        differ = out[ok] != want[ok]
        assert not differ.any(), (epi, out[ok][differ][:8], want[ok][differ][:8])


@pytest.mark.gpu
@pytest.mark.parametrize("M,I,K", [(129, 64, 128), (300, 100, 192),
                                   (700, 1024, 256), (300, 64, 72)])
def test_swiglu_of_many_rows(M, I, K):
    """Through the public op; sizes that tiles do not take go to the library."""
    x, w = rand(M, 2 * K, seed=1), rand(2 * I, K, seed=2, scale=K ** -0.5)
    for a in (x[:, :K].contiguous(), x[:, K:]):
        y = a.double() @ w.double().t()
        want = F.silu(y[:, :I]) * y[:, I:]
        if I % 8:      # beyond 32 rows the SwiGLU pass takes whole vectors
            assert not tiles.tile_ok(M, a, w[:I])
            continue
        # rounded once, in the library and its pass twice before
        assert err(ops.gemv_swiglu(a, w), want) < 2 ** -8
        out = torch.full((M, 2 * I), 7.0, device=DEV, dtype=torch.bfloat16)
        n2 = a.contiguous()
        mx.mix_in(n2, n2, torch.cat([w[:8], w]), 8, I, out[:, I:])
        assert err(out[:, I:], want) < 2 ** -8
        assert bool((out[:, :I] == 7).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,I,K", [(2600, 2056, 1088), (2049, 2048, 512),
                                   (2600, 2056, 1080)])
def test_activations_of_many_rows(M, I, K):
    """Through the public ops, where tiles take them; the last is the library's."""
    x, w = rand(M, K, seed=1), rand(2 * I, K, seed=2, scale=K ** -0.5)
    b = rand(2 * I, seed=3)
    assert (ops._many_rows(M, x, w) == "tile") == (K % 64 == 0)
    y = x.double() @ w.double().t()
    # rounded once, in the library and its pass twice before
    assert err(ops.gemv_swiglu(x, w), F.silu(y[:, :I]) * y[:, I:]) < 2 ** -8
    assert err(ops.linear_bias(x.view(1, M, K), w, b, True)[0],
               F.gelu(y + b.double())) < 2 ** -8
    out = torch.full((M, 3 * I), 7.0, device=DEV, dtype=torch.bfloat16)
    h = mx.GainNormed(x.float(), None, torch.bfloat16, x)
    mx.parallel_in(h, w, 0, 2 * I, 0, out[:, I:])
    assert err(out[:, I:], y.clamp_min(0) ** 2) < 2 ** -8
    assert bool((out[:, :I] == 7).all())


@pytest.mark.gpu
def test_swiglu_of_many_rows_to_a_place_between():
    """Results that start on any 2 bytes: nothing is written beside them."""
    M, I, K = 2048, 2048, 512
    x, w = rand(M, K, seed=1), rand(2 * I, K, seed=2, scale=K ** -0.5)
    assert ops._many_rows(M, x, w) == "tile"
    y = x.double() @ w.double().t()
    for at in (0, 1, 4, 8):
        room = torch.full((M * I + 16,), 7.0, device=DEV, dtype=torch.bfloat16)
        got = ops.gemv_swiglu(x, w, room[at:at + M * I].view(M, I))
        # rounded once, in the library and its pass twice before
        assert err(got, F.silu(y[:, :I]) * y[:, I:]) < 2 ** -8
        assert bool((room[:at] == 7).all() and (room[at + M * I:] == 7).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(257, 256, 8192), (600, 2048, 8256),
                                   (1500, 1024, 10240)])
def test_parts_and_their_norm(M, N, K):
    x, w = rand(M, K, seed=1), rand(N, K, seed=2, scale=K ** -0.5)
    h, gain = rand(M, N, seed=3), rand(N, seed=4)
    assert ops.tile_parts_ok(M, x, w)
    assert not ops.tile_parts_ok(M, x.float(), w)
    assert not ops.tile_parts_ok(M, x[:, 64:], w)
    want = h.double() + x.double() @ w.double().t()
    out = ops.add_norm_parts(ops.tile_parts(x, w), h, gain, 1e-5)
    assert err(h, want) < 2 ** -9
    norm = want * (want.pow(2).mean(-1, keepdim=True) + 1e-5).rsqrt()
    assert err(out, norm * gain.double()) < 2 ** -8


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(257, 8, 8192), (300, 2048, 10240),
                                   (1706, 1000, 8256), (300, 2048, 8128)])
def test_residual_of_many_rows(M, N, K):
    """In parts of K, or (short K, a residual between others') in the library."""
    a, w = rand(M, K, seed=1), rand(N, K, seed=2, scale=K ** -0.5)
    x = rand(M, N + 2, seed=3).float()
    for res in (x[:, :N].contiguous(), x[:, 2:]):
        assert tiles.add_ok(res, a, w) == (K >= 8192 and N % 8 == 0
                                           and res.data_ptr() % 16 == 0)
        want = res.double() + 0.5 * (a.double() @ w.double().t())
        # float32 sums of K products and one addition
        assert err(mx.residual_linear(res, a, w, 0.5), want) < 2 ** -24 * K ** 0.5


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(257, 8, 8192), (300, 992, 8192),
                                   (300, 1000, 8192)])
def test_parts_of_few_results_stay_in_the_library(M, N, K, monkeypatch):
    a, w = rand(M, K, seed=1), rand(N, K, seed=2, scale=K ** -0.5)
    x, g = rand(M, N, seed=3).float(), rand(N, seed=4).float()
    want = x.double() + a.double() @ w.double().t()
    calls, parts = [], tiles.product_parts
    monkeypatch.setattr(tiles, "product_parts",
                        lambda *t: (calls.append(1), parts(*t))[1])
    # float32 sums of K products and one addition
    assert err(mx.residual_linear(x.clone(), a, w), want) < 2 ** -24 * K ** 0.5
    y, normed = mx.residual_norms(x, a, w, g, None, 1e-3, torch.bfloat16)
    assert err(y, want) < 2 ** -24 * K ** 0.5
    assert len(calls) == 2 * (N >= 1000) and (normed is None) == (N < 1000)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1301, 5704, 2048), (4001, 3072, 1984),
                                   (3777, 2568, 1088), (300, 512, 2048)])
def test_plain_products_of_many_rows(M, N, K):
    """Through the public op and inside a layer's input, rows with gaps too; the last
    is the library's."""
    x, w = rand(M, K, seed=1), rand(N, K, seed=2, scale=K ** -0.5)
    want = x.double() @ w.double().t()
    assert tiles.linear_ok(M, x, w) == (M > 300)
    # a result is rounded once, by 2^-9 at most
    assert err(ops.linear_decode(x.view(1, M, K), w)[0], want) < 2 ** -9
    for rows in (x, rand(M, K + 8, seed=1)[:, :K]):
        want = rows.double() @ w.double().t()
        assert err(mx.mix_in(rows, None, w, N, 0, rows), want) < 2 ** -9
    v = w.clone().requires_grad_()           # gradients are the library's
    assert not tiles.linear_ok(M, x, v)
    assert ops.linear_decode(x, v).requires_grad


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,pair", [
    (40, 8, 4096, True), (256, 1000, 4160, False), (257, 2048, 8192, True),
    (300, 4104, 8256, True), (300, 256, 4096, False)])
def test_residual_and_its_norms(M, N, K, pair):
    """What one kernel makes of a product in parts, some columns and more than its
    registers hold; the last is in the library, which leaves the norms to others."""
    a, w = rand(M, K, seed=1), rand(N, K, seed=2, scale=K ** -0.5)
    x, g = rand(M, N, seed=3).float(), rand(2, N, seed=4).float()
    want = x.double() + 0.5 * (a.double() @ w.double().t())
    y, normed = mx.residual_norms(x, a, w, g[0], g[1] if pair else None, 1e-3,
                                  torch.bfloat16, 0.5)
    # float32 sums of K products and one addition
    assert err(y, want) < 2 ** -24 * K ** 0.5
    assert (normed is None) == (K == 4096 and M > 256)
    if normed is None:
        return
    norm = want * (want.pow(2).mean(-1, keepdim=True) + 1e-3).rsqrt()
    # rounded once, by 2^-9 at most
    assert err(normed[0], norm * g[0].double()) < 2 ** -9
    assert err(normed[1], norm * g[1].double()) < 2 ** -9 if pair \
        else normed[1] is None


class Recorder(torch.overrides.TorchFunctionMode):
    def __init__(self):
        self.seen = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.seen.append(func)
        return func(*args, **(kwargs or {}))


class Tagged(torch.Tensor):
    """A class of its own, as users make them."""


def test_tensors_that_are_more_than_memory():
    """Tiles leave them to the library; no GPU is needed to say which they are."""
    x = rand(4, 8, dev="cpu")
    w = torch.nn.Parameter(x)
    assert tiles._memory(x, w)
    seen = []
    torch.func.vmap(lambda t: (seen.append(tiles._memory(t)), t)[1])(x[None])
    with torch.autograd.forward_ad.dual_level():
        seen.append(tiles._memory(x))
    with torch._subclasses.FakeTensorMode():
        seen.append(tiles._memory(x))
    torch.jit.trace(lambda t: (seen.append(tiles._memory(t)), t + 1)[1], x,
                    check_trace=False)
    with Recorder():
        seen.append(tiles._memory(x))
    seen.append(tiles._memory(x, x.as_subclass(Tagged)))
    for dtype in (torch.float16, torch.bfloat16):
        before = torch.get_autocast_dtype("cuda")
        torch.set_autocast_enabled("cuda", True)
        torch.set_autocast_dtype("cuda", dtype)
        try:             # bfloat16 stays as it is
            seen.append(tiles._memory(x) != (dtype is torch.bfloat16))
        finally:
            torch.set_autocast_enabled("cuda", False)
            torch.set_autocast_dtype("cuda", before)
    assert len(seen) >= 8 and not any(seen)
    with torch.device("cpu"):                # a default for new tensors
        assert tiles._memory(x)
    # rows with gaps, of which a copy goes to the kernel
    wide = rand(300, 256, dev="cpu").as_subclass(Tagged)[:, :128]
    ok, tiles.act_ok = tiles.act_ok, lambda M, a, b: tiles._memory(a, b)
    try:
        w = rand(64, 128, dev="cpu")
        assert ops._many_rows(300, torch.Tensor(wide.float())[:, :128], w)
        assert ops._many_rows(300, wide, w) is None
        x, room = rand(300, 128, dev="cpu"), rand(300 * 32 + 8, dev="cpu")
        for at in range(9):              # results on 16 bytes
            out = room[at:at + 300 * 32]
            assert bool(ops._many_rows(300, x, w, out)) == (at % 8 == 0)
    finally:
        tiles.act_ok = ok


@pytest.mark.gpu
def test_tensors_of_another_device_are_the_library_s(monkeypatch):
    M, N, K = 1301, 5704, 2048
    x, w = rand(M, K, seed=1), rand(N, K, seed=2, scale=K ** -0.5)
    assert tiles.linear_ok(M, x, w) and tiles.act_ok(M, x, w)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    assert not tiles.linear_ok(M, x, w) and not tiles.act_ok(M, x, w)
    long = rand(1024, 8192)
    assert not tiles.parts_ok(300, rand(300, 8192), long)


@pytest.mark.gpu
@pytest.mark.parametrize("I", [2048, 2052, 2056])
def test_swiglu_wants_a_multiple_of_8_columns(I):
    """Gates and ups are a multiple of 8 together before they are one each."""
    M, K = 2049, 512
    x, w = rand(M, K, seed=1), rand(2 * I, K, seed=2)
    assert tiles.act_ok(M, x, w)
    assert (ops._many_rows(M, x, w) == "tile") == (I % 8 == 0)
    act = torch.empty(M, 2056, device=DEV, dtype=torch.bfloat16)
    assert mx._act_tile(x, w, I, act) == (I % 8 == 0)
    assert not mx._act_tile(x, w, 2048, act[:, 4:])      # rows not on 16 bytes
    assert not mx._act_tile(x, w, 2048, act.float())


@pytest.mark.gpu
def test_many_rows_under_transforms():
    M, N, K = 1301, 5704, 2048
    x, w = rand(M, K, seed=1), rand(N, K, seed=2, scale=K ** -0.5)
    v = rand(M, K, seed=3)
    assert tiles.linear_ok(M, x, w)
    y, dy = torch.func.jvp(lambda t: ops.linear_decode(t, w), (x,), (v,))
    # results are rounded once, by 2^-9 at most
    assert err(y, x.double() @ w.double().t()) < 2 ** -9
    assert err(dy, v.double() @ w.double().t()) < 2 ** -9
    both = torch.func.vmap(lambda t: ops.linear_decode(t, w))(torch.stack([x, v]))
    assert err(both[1], v.double() @ w.double().t()) < 2 ** -9
    # what follows torch's operations sees one, and a cast is made
    with Recorder() as mode:
        ops.linear_decode(x, w)
    assert F.linear in mode.seen
    with torch.autocast("cuda", dtype=torch.float16):
        assert ops.linear_decode(x, w).dtype == torch.float16
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert torch.equal(ops.linear_decode(x, w), tiles.linear(x, w))
