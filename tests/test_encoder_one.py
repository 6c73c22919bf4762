"""An encoder over up to 128 rows in one launch (csrc/encoder_one.hip) against float64 with
its roundings and against the chain of launches, at the edges of its tiles of rows and of the
blocks' and waves' shares."""

import dataclasses

import one_launch_oracle as oracle
import pytest
import torch

from fei_amd import ops
from fei_amd.engine.config import get_spec
from fei_amd.models.bge import BgeEncoder

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# 8 roundings a layer, 2^-9 / sqrt(3) each, that differ on either side: sqrt(2 * 96) of
# them make 0.016; twice that
TOL = 2 ** -5
# Against float64 that is rounded where the launch does: 2^-9 sqrt(2 / 3) = 1.6e-3 between two
# roundings of a value that fall otherwise, four on a row's way through a layer (two norms,
# attention, GELU), of three layers 5.5e-3 if all did
TOL64 = 2 ** -7

# (heads, width, inner): a wave with the only steps, lanes without columns, waves without
# steps, uneven shares, the widest
SIZES = [(1, 64, 64), (2, 192, 128), (5, 320, 704), (12, 768, 3072), (12, 704, 3008)]


def model(heads, C, inner, layers=3, seed=1):
    spec = dataclasses.replace(get_spec("bge-base"), num_layers=layers, num_heads=heads,
                               num_kv_heads=heads, hidden_size=C,
                               intermediate_size=inner)
    m = BgeEncoder(spec, device=torch.device(DEV), seed=seed)
    g = torch.Generator(device=DEV).manual_seed(seed)
    for lw in m.layers:
        for n in ("ln1_w", "ln2_w"):
            lw[n].copy_(1 + 0.2 * torch.randn(C, generator=g, device=DEV))
        for n in ("bqkv", "bo", "bi", "bo2", "ln1_b", "ln2_b"):
            lw[n].copy_(0.1 * torch.randn(lw[n].shape, generator=g, device=DEV))
    return m


def texts(B, S, seed=2):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randint(0, 1000, (B, S), generator=g, device=DEV)


def one(m, ids, lens, **kw):
    with torch.no_grad():
        from fei_amd.models.bge import NAMES
        return ops.encoder_one(ids, m.tok_emb, m.pos_emb, m.emb_ln_w, m.emb_ln_b,
                               [lw[n] for lw in m.layers for n in NAMES],
                               m.spec.num_heads, 64, m.spec.intermediate_size,
                               lens.int(), m.eps, **kw)


def chain(m, ids, lens):
    real, ops.encoder_one = ops.encoder_one, lambda *a: None
    try:
        return m.encode_ids(ids, lens)
    finally:
        ops.encoder_one = real


def near(got, want, tol=TOL):
    err = ((got - want).norm(dim=-1) / want.norm(dim=-1)).max()
    assert got.isfinite().all() and err < tol, f"rel err {err}"


def exact(m, ids, lens):
    h = ops.embed_layernorm(ids, m.tok_emb, m.pos_emb, m.emb_ln_w, m.emb_ln_b, m.eps,
                            torch.bfloat16)
    return oracle.encoder(m, h, lens)


@pytest.mark.parametrize("heads,C,inner", SIZES)
@pytest.mark.parametrize("B,S", [(1, 1), (1, 16), (1, 24), (2, 16), (1, 33), (7, 7),
                                 (1, 64), (64, 1), (3, 21),
                                 # each number of tiles of rows, and two an item
                                 (1, 65), (3, 32), (9, 11), (1, 112), (128, 1), (1, 128),
                                 (2, 61)])
def test_sizes(heads, C, inner, B, S):
    m, ids = model(heads, C, inner), texts(B, S)
    lens = torch.arange(B, device=DEV) * 5 % S + 1
    lens[0] = S
    got = one(m, ids, lens)
    assert got is not None and torch.equal(got, m.encode_ids(ids, lens))
    near(got, chain(m, ids, lens))
    near(got, exact(m, ids, lens), TOL64)


def test_all_layers_and_lengths():
    """Empty texts are 0, lengths beyond the text its length; no lengths are full ones."""
    m, ids = model(12, 768, 3072, layers=12), texts(4, 16)
    lens = torch.tensor([16, 0, 99, -3], device=DEV)
    got = m.encode_ids(ids, lens)
    assert not got[1].any() and not got[3].any()
    near(got[::2], chain(m, ids, lens.clamp(0, 16))[::2])
    # four times the layers, and means of 16 rows
    near(got[::2], exact(m, ids, lens)[::2], TOL64)
    near(m.encode_ids(ids), chain(m, ids, None))


def test_texts_and_padding_stay_apart():
    """What is not finite in one text, or behind another's end, does not reach a third."""
    m, ids = model(2, 192, 128), texts(3, 20)
    lens = torch.tensor([20, 13, 20], device=DEV)
    want = m.encode_ids(ids, lens)
    m.tok_emb[1001] = float("inf")
    m.tok_emb[1002] = float("nan")
    ids[0, 3], ids[1, 13], ids[1, 19] = 1001, 1002, 1001
    got = m.encode_ids(ids, lens)
    assert got[0].isnan().all() and torch.equal(got[1:], want[1:])


@pytest.mark.parametrize("blocks", [1, 50, 255])
@pytest.mark.parametrize("B,S", [(1, 24), (8, 8), (1, 85), (5, 25)])
@pytest.mark.parametrize("heads,C,inner", [(1, 64, 64), (12, 768, 3072)])
def test_items_by_ticket(heads, C, inner, B, S, blocks):
    """Fewer blocks than items, as where something else holds CUs: the same bits."""
    m, ids = model(heads, C, inner), texts(B, S)
    lens = torch.full((B,), S, device=DEV)
    assert torch.equal(one(m, ids, lens, blocks=blocks), one(m, ids, lens))


def test_streams_and_replays():
    m, lens = model(12, 768, 3072, layers=4), torch.tensor([24], device=DEV)
    runs = []
    for i in range(2):
        ids = texts(1, 24, seed=i)
        m.encode_ids(ids, lens)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            out = m.encode_ids(ids, lens)
        runs.append((g, ids, out, torch.cuda.Stream()))
    for k in range(4):
        want = []
        for i, (g, ids, out, s) in enumerate(runs):
            ids.copy_(texts(1, 24, seed=10 * k + i))
            want.append(m.encode_ids(ids, lens))
        torch.cuda.synchronize()
        for g, ids, out, s in runs:
            with torch.cuda.stream(s):
                g.replay()
        torch.cuda.synchronize()
        for (g, ids, out, s), w in zip(runs, want):
            assert torch.equal(out, w)


@pytest.mark.parametrize("change", ["rows", "wide", "inner", "gap", "lengths", "gradient"])
def test_what_is_left_to_the_chain(change):
    m, ids = model(*{"wide": (13, 832, 64), "inner": (1, 64, 3136)}
                   .get(change, (2, 192, 128))), texts(5, 25)
    lens = torch.full((5,), 25, device=DEV)
    if change == "rows":
        ids, lens = texts(5, 26), lens + 1
    elif change == "gap":
        m.layers[1]["wo"] = torch.cat([m.layers[1]["wo"]] * 2, 1)[:, :128]
    elif change == "lengths":
        lens = lens[:4]
    if change == "gradient":
        m.layers[0]["bo"].requires_grad_()
        with torch.enable_grad():
            from fei_amd.models.bge import NAMES
            assert ops.encoder_one(
                ids, m.tok_emb, m.pos_emb, m.emb_ln_w, m.emb_ln_b,
                [lw[n] for lw in m.layers for n in NAMES], 2, 64, 128, lens.int(),
                m.eps) is None
    else:
        assert one(m, ids, lens) is None
