"""When a decoding step or an encoder runs in one launch, and what it refuses: host code
alone where nothing says gpu."""

import ctypes

import pytest
import torch

from fei_amd import ops
from fei_amd.engine.config import ModelSpec
from fei_amd.models.llama import LlamaModel
from fei_amd.ops.layers import _EncoderShape, _OneShape


def room(kind, blocks):
    lib = ops.require_lib()
    if kind == "step":
        return lib.fei_decode_one_room(ctypes.byref(_OneShape(
            2, 2048, 8192, 32, 8, 64, 320, 4000, 0, blocks, 1e-5, 0.125)))
    return lib.fei_encoder_one_room(ctypes.byref(_EncoderShape(
        2, 1, 24, 12, 768, 3072, blocks, 1e-5, 0.125)))


@pytest.mark.parametrize("kind", ["step", "encoder"])
def test_blocks_of_a_launch(kind):
    """More than there are items would have items of their own past every end."""
    want = room(kind, 256)
    assert want > 0
    for blocks in (1, 2, 255):
        assert room(kind, blocks) == want
    for blocks in (-1, 0, 257, 512):
        assert room(kind, blocks) == 0


def weights(C, I, heads, kv_heads, dim):
    return C * dim * (2 * heads + 2 * kv_heads) + 3 * C * I


# sizes (a layer's and the head's), layers, and whether the one launch was measured to be
# faster: bfloat16, fp8
@pytest.mark.parametrize("sizes,vocab,layers,want", [
    ((512, 512, 8, 8, 64), 512, 24, (False, False)),
    ((1024, 1024, 16, 4, 64), 1024, 24, (False, False)),
    ((1024, 2048, 16, 4, 64), 4000, 16, (False, False)),
    ((1280, 3072, 20, 5, 64), 4000, 8, (True, False)),
    ((1536, 4096, 12, 4, 128), 1024, 4, (False, False)),
    ((1536, 6144, 12, 4, 128), 4000, 8, (True, True)),
    ((2048, 5632, 32, 4, 64), 32000, 1, (False, False)),
    ((2048, 5632, 32, 4, 64), 32000, 24, (True, True)),
    ((2048, 8192, 32, 8, 64), 128256, 4, (False, False)),
    ((2048, 8192, 32, 8, 64), 128256, 16, (True, True)),
    ((4096, 14336, 32, 8, 128), 128256, 32, (True, True))])
def test_steps_that_one_launch_is_faster_for(sizes, vocab, layers, want):
    w, head = weights(*sizes), vocab * sizes[0]
    assert tuple(ops.llama_one_pays(layers, w, head, f) for f in (False, True)) == want


def model(layers, C):
    spec = ModelSpec("route", 1024, C, layers, C // 64, C // 256, 64, 3 * C)
    return LlamaModel(spec, torch.device("cuda:0"), torch.bfloat16, seed=1, max_seq_len=64)


@pytest.mark.gpu
@pytest.mark.parametrize("layers,C,taken", [(2, 512, False), (12, 512, False),
                                            (8, 1280, True)])
@pytest.mark.parametrize("wanted", [True, False])
def test_route_of_a_captured_step(layers, C, taken, wanted, monkeypatch):
    """In one launch where that is faster and wanted; else with an eager step's bits."""
    taken = taken and wanted
    calls, real = [], ops.llama_one
    monkeypatch.setattr(ops, "llama_one",
                        lambda *a, **k: calls.append(real(*a, **k)) or calls[-1])
    m = model(layers, C)
    m.one_launch = wanted
    tok = torch.tensor([7], dtype=torch.int32, device="cuda:0")
    pos = torch.tensor([3], dtype=torch.int32, device="cuda:0")
    kc, vc = m.new_kv_cache(1, 64)
    with torch.no_grad():
        want = m.forward_decode(tok, pos, kc, vc)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            got = m.forward_decode(tok, pos, kc, vc)
    assert len(calls) == taken and all(c is not None for c in calls)
    for _ in range(3):
        got.zero_()
        g.replay()
        torch.cuda.synchronize()
        if taken:
            assert (got - want).float().norm() < 2 ** -6 * want.float().norm()
        else:
            assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("layers,C", [(2, 512), (8, 2048)])
@pytest.mark.parametrize("splits,room", [(32, 16), (16, 32), (65, 65)])
def test_what_a_captured_step_refuses(layers, C, splits, room, fp8):
    """Where it runs in one launch too, which has no use for a workspace."""
    m = model(layers, C)
    if fp8:
        m.quantize_fp8()
    tok = torch.tensor([7], dtype=torch.int32, device="cuda:0")
    pos = torch.tensor([3], dtype=torch.int32, device="cuda:0")
    kc, vc = m.new_kv_cache(1, 64)
    ws = [torch.zeros(1, C // 64, room, n, device="cuda:0") for n in (64, 2)]

    def step():
        with pytest.raises(AssertionError):
            m.forward_decode(tok, pos, kc, vc, attn_splits=splits, workspace=ws,
                             fused_norm=fp8)
        return tok + 1
    with torch.no_grad():
        step()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            out = step()
    g.replay()
    assert out.item() == 8


@pytest.mark.parametrize("layers,B,S,taken", [(1, 1, 32, True), (1, 3, 11, False),
                                              (2, 4, 16, True), (2, 5, 13, False),
                                              (3, 1, 128, True), (12, 128, 1, True)])
def test_encoders_that_one_launch_is_faster_for(layers, B, S, taken, monkeypatch):
    import dataclasses

    from fei_amd.engine.config import get_spec
    from fei_amd.models.bge import BgeEncoder
    spec = dataclasses.replace(get_spec("bge-base"), num_layers=layers, num_heads=1,
                               num_kv_heads=1, hidden_size=64, intermediate_size=64)
    m = BgeEncoder(spec, device=torch.device("cpu"), dtype=torch.float32)
    asked = []
    monkeypatch.setattr(ops, "encoder_one", lambda *a: asked.append(1))
    m.encode_ids(torch.ones(B, S, dtype=torch.int64))
    assert bool(asked) == taken
    m.one_launch = False
    m.encode_ids(torch.ones(B, S, dtype=torch.int64))
    assert len(asked) == taken


def test_models_that_were_kept_from_before():
    """What was pickled without the attribute runs."""
    from fei_amd.models.bge import BgeEncoder
    for cls in (LlamaModel, BgeEncoder):
        assert cls.__new__(cls).one_launch
