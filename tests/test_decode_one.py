"""A decoding step of one row in one launch (csrc/decode_one.hip) against float64 with its
roundings and against the chain of launches, at the sizes where its blocks' shares are
uneven, empty ends or few."""

import one_launch_oracle as oracle
import pytest
import torch

from fei_amd import ops
from fei_amd.engine.config import ModelSpec
from fei_amd.models.llama import LlamaModel

gpu = pytest.mark.gpu
DEV = "cuda:0"

# two roundings of a residual and three of what is added to it a layer, 2^-9 each at
# most, on either side
TOL = 2 ** -6
# Against float64 that is rounded where the step is, sums alone differ. Most results are the
# same; where one falls on the other side of a middle, what follows is rounded otherwise:
# 2^-9 sqrt(2 / 3) = 1.6e-3 between two roundings of a value, five on the residual's way
# through a layer (norm, attention or activation, sum, twice, of which the inner ones are a
# part of it): 2^-8 a layer
TOL64 = 2 ** -8

SIZES = {
    # one pair of rows an item, a head of keys for each of queries
    "least": dict(C=512, I=512, Hq=8, Hkv=8, D=64, vocab=512),
    # steps' ends within rows, uneven items, one head of keys and 256 splits
    "uneven": dict(C=528, I=1040, Hq=16, Hkv=1, D=64, vocab=1030),
    # three heads of keys: blocks without any
    "three": dict(C=1536, I=2064, Hq=12, Hkv=3, D=128, vocab=514),
    "1b": dict(C=2048, I=8192, Hq=32, Hkv=8, D=64, vocab=4000),
    "8b": dict(C=4096, I=14336, Hq=32, Hkv=8, D=128, vocab=4000),
}


def model(size, layers, room, fp8, seed=1, dev=DEV):
    s = SIZES[size]
    spec = ModelSpec("one", s["vocab"], s["C"], layers, s["Hq"], s["Hkv"], s["D"],
                     s["I"])
    m = LlamaModel(spec, torch.device(dev), torch.bfloat16, seed=seed,
                   max_seq_len=room)
    g = torch.Generator(device=dev).manual_seed(seed)
    for lw in m.layers:
        for t in (lw.norm_attn, lw.norm_mlp):
            t.copy_(1 + 0.2 * torch.randn(t.shape, generator=g, device=dev))
    m.emb.mul_(50)
    if fp8:
        m.quantize_fp8()
    return m


def attentive(m):
    """Attention over thousands of unlike keys is small: the rest is made smaller, so
    that it is what the logits are."""
    m.emb.div_(50)
    for lw in m.layers:
        lw.wo.mul_(8)
        lw.wdown.mul_(0.02)
    return m


def caches(m, n, room, seed=2, dev=DEV):
    """Keys and values up to position n - 1; what lies past them is not to be read."""
    g = torch.Generator(device=dev).manual_seed(seed)
    shape = (m.spec.num_layers, 1, m.hkv_l, room, m.D)
    out = []
    for _ in range(2):
        t = torch.randn(shape, generator=g, device=dev).to(torch.bfloat16)
        t[..., n:, :] = float("nan")
        out.append(t)
    return out


def one(m, h, pos, k, v, fp8, **kw):
    return ops.llama_one(h, m.layers, list(k), list(v), m.hq_l, m.spec.norm_eps, pos,
                         m.rope, m.norm_f, m.lm_head, m.fp8 if fp8 else None,
                         m.fp8_lm_head if fp8 else None, **kw)


def rel(got, want):
    return ((got.double() - want.double()).norm() / want.double().norm()).item()


def near(got, want, tol=TOL):
    assert rel(got, want) < tol, f"rel err {rel(got, want)}"


def check(m, n, room, fp8, **kw):
    k, v = caches(m, n, room)
    k1, v1 = k.clone(), v.clone()
    tok = torch.tensor([7], dtype=torch.int32, device=DEV)
    pos = torch.tensor([n], dtype=torch.int32, device=DEV)
    with torch.no_grad():
        want = m.forward_decode(tok, pos, list(k), list(v), fused_norm=fp8)
        h = m._embed(tok)
        kept = h.clone()
        exact, *rows = oracle.step(m, h, n, k, v, fp8)
        got = one(m, h, pos, k1, v1, fp8, **kw)
    assert got is not None and torch.equal(h, kept)
    near(got, want)
    at, tol = min(n, room - 1), TOL64 * len(m.layers) ** 0.5
    near(got[0], exact, tol)
    for a, b in zip((k1, v1), rows):
        near(a[:, 0, :, at], b, tol)
    for a, b in ((k1, k), (v1, v)):
        near(a[..., at, :], b[..., at, :])
        a[..., at, :] = b[..., at, :] = 0
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@gpu
@pytest.mark.parametrize("size", list(SIZES))
@pytest.mark.parametrize("fp8", [False, True])
def test_sizes(size, fp8):
    check(model(size, 2, 320, fp8), 300, 320, fp8)


# a wave's 32 keys, the splits' 256 of a head (8 heads, 32 blocks each), two rounds
@pytest.mark.parametrize("n", [0, 1, 31, 32, 33, 1023, 1024, 8191, 8200])
@gpu
@pytest.mark.parametrize("size", ["1b", "three"])
def test_lengths(size, n):
    check(attentive(model(size, 1, n + 1, False)), n, n + 1, False)


@pytest.mark.parametrize("n", [33, 1024, 8200])
@pytest.mark.parametrize("size", ["1b", "three"])
def test_lengths_would_show_what_is_lost(size, n):
    """A wave's 32 keys, or what there is of them, left out or counted twice."""
    m = attentive(model(size, 1, n + 1, False, dev="cpu"))
    k, v = caches(m, n, n + 1, dev="cpu")
    with torch.no_grad():
        h = m._embed(torch.tensor([7]))
        want = oracle.step(m, h, n, k, v)[0]
        keys = torch.arange(n)
        for at in (0, n // 64 * 32, (n - 1) // 32 * 32):
            for seen in (torch.cat([keys[:at], keys[at + 32:]]),
                         torch.cat([keys, keys[at:at + 32]])):
                assert rel(oracle.step(m, h, n, k, v, keep=seen)[0], want) > 4 * TOL64


@gpu
def test_position_past_the_cache():
    check(model("least", 1, 64, False), 70, 64, False)


@gpu
@pytest.mark.parametrize("layers", [32, 33])
def test_launches_of_32_layers(layers):
    m = model("least", layers, 64, False)
    # the residual's error grows with the layers: held small against it
    for lw in m.layers:
        lw.wo.mul_(0.1)
        lw.wdown.mul_(0.1)
    check(m, 40, 64, False)


@gpu
@pytest.mark.parametrize("blocks", [1, 40, 255])
@pytest.mark.parametrize("size,fp8", [("uneven", False), ("three", True)])
def test_items_by_ticket(size, fp8, blocks):
    """Fewer blocks than items, as where something else holds CUs."""
    check(model(size, 2, 320, fp8), 300, 320, fp8, blocks=blocks)


@gpu
@pytest.mark.parametrize("change", ["odd vocabulary", "narrow", "gap", "type", "rope"])
def test_what_is_left_to_the_chain(change):
    m = model("least", 1, 64, False)
    k, v = caches(m, 3, 64)
    pos = torch.tensor([3], dtype=torch.int32, device=DEV)
    h = m._embed(torch.tensor([7], device=DEV))
    if change == "odd vocabulary":
        m.lm_head = m.lm_head[:511]
    elif change == "narrow":
        m.layers[0].wdown = m.layers[0].wdown[:, :256].contiguous()
        m.layers[0].wgu = m.layers[0].wgu[:512].contiguous()
    elif change == "gap":
        m.layers[0].wo = torch.cat([m.layers[0].wo] * 2, 1)[:, :512]
    elif change == "type":
        pos = pos.long()
    else:
        m.rope = m.rope[:32]
    with torch.no_grad():
        assert one(m, h, pos, k, v, False) is None


def captured(fn):
    fn()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = fn()
    return g, out


@gpu
@pytest.mark.parametrize("fp8", [False, True])
def test_captured_steps(fp8, monkeypatch):
    """Each replay reads tokens, positions and caches anew, also between others' work and
    beside a step on another stream."""
    calls = []
    real = ops.llama_one
    monkeypatch.setattr(ops, "llama_one", lambda *a, **k: calls.append(real(*a, **k))
                        or calls[-1])
    m = model("1b", 2, 256, fp8)
    steps = []
    with torch.no_grad():
        for i in range(2):
            k, v = caches(m, 100, 256, seed=5 + i)
            k.nan_to_num_()
            v.nan_to_num_()
            tok = torch.tensor([7 + i], dtype=torch.int32, device=DEV)
            pos = torch.tensor([90], dtype=torch.int32, device=DEV)
            g, out = captured(lambda: m.forward_decode(tok, pos, list(k), list(v),
                                                       fused_norm=fp8))
            steps.append((g, out, tok, pos, k, v))
        assert len(calls) == 2 and all(c is not None for c in calls)
        streams = [torch.cuda.Stream() for _ in steps]
        for n in (90, 95, 31, 200):
            want = []
            for g, out, tok, pos, k, v in steps:
                tok.fill_(n)
                pos.fill_(n)
                want.append(m.forward_decode(tok, pos, list(k.clone()),
                                             list(v.clone()), fused_norm=fp8))
            torch.cuda.synchronize()
            for (g, *_), s in zip(steps, streams):
                with torch.cuda.stream(s):
                    g.replay()
            torch.cuda.synchronize()
            for (g, out, *_), w in zip(steps, want):
                near(out, w)
