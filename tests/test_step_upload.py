"""What a step's batch is uploaded with (engine/step.py): one copy, from which the plans
of the model's mixers are views, the same as those made when they are asked for."""

import copy

import numpy as np
import pytest
import torch

from fei_amd.engine.config import get_spec
from fei_amd.engine.step import RaggedBatch, StepEntry, StepRunner, upload
from fei_amd.models import model_class

DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]


@pytest.mark.parametrize("device", DEVICES)
def test_upload(device):
    """Types, shapes, empty arrays, arrays with gaps; the copy is the stream's own."""
    g = np.random.default_rng(1)
    arrays = [g.integers(0, 99, n).astype(t).reshape(s) for n, t, s in (
        (5, np.int64, (5,)), (0, np.int64, (0,)), (7, np.int32, (7, 1)),
        (0, np.int32, (0, 3)), (1, np.int32, (1,)), (30, np.int32, (5, 6)))]
    arrays.append(arrays[-1][:, ::2])
    got = upload(arrays, torch.device(device))
    want = [a.copy() for a in arrays]
    for _ in range(4):                       # staging memory is not taken again too soon
        upload([a * 0 - 1 for a in arrays], torch.device(device))
    for a, t in zip(want, got):
        assert t.device.type == device and t.data_ptr() % 8 == 0
        assert t.dtype == torch.from_numpy(a).dtype
        assert np.array_equal(t.cpu().numpy(), a)
        if device == "cuda" and t.numel():
            assert t.data_ptr() % 16 == 0


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("model", ["tobarax-tiny", "bokenex-tiny"])
@pytest.mark.parametrize("lens", [[1, 1], [3], [1, 70, 1, 130, 2]])
def test_plans_of_a_batch(model, lens, device):
    spec = get_spec(model)
    runner = StepRunner(model_class(spec)(spec, torch.device(device)), 64, 8, 16)
    entries = [StepEntry(runner.admit(n), list(range(4, 4 + n)), [n - 1]) for n in lens]
    batch = runner.build(entries)
    later = RaggedBatch(batch.tokens, batch.pos, batch.row_seq, batch.table,
                        batch.slots, batch.n_dec, batch.portions)
    assert bool(batch._plans) == bool(batch.portions)
    for key in batch._plans:
        for a, b in zip(batch._plans[key], later._plan(key)):
            assert a.dtype == b.dtype and torch.equal(a, b)
    order = sorted(range(len(lens)), key=lambda i: lens[i] > 1)
    assert batch.tokens.tolist() == [t for i in order for t in entries[i].tokens]
    rows, at = {}, 0
    for i in order:
        rows[i], at = at + lens[i] - 1, at + lens[i]
    assert batch.want_rows.tolist() == [rows[i] for i in range(len(lens))]
    assert runner.build(entries, all_rows=True).want_rows is None


def test_upload_is_refused_under_capture(monkeypatch):
    """A graph would copy again from memory that is others' by then."""
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    with pytest.raises(RuntimeError, match="captured"):
        upload([np.zeros(3, np.int32)], torch.device("cuda"))


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["tobarax-tiny", "bokenex-tiny"])
def test_batch_of_another_stream(model):
    """Built on a stream that has much to do yet, run on another, as is and copied."""
    spec = get_spec(model)
    m = model_class(spec)(spec, torch.device("cuda"))
    results = []
    for busy in (None, lambda b: b, copy.copy):
        runner = StepRunner(m, 64, 8, 16)
        entries = [StepEntry(runner.admit(n), list(range(4, 4 + n)), [n - 1])
                   for n in (70, 1, 9)]
        torch.cuda.synchronize()
        side = torch.cuda.Stream()
        with torch.cuda.stream(side if busy else torch.cuda.current_stream()):
            if busy:
                torch.cuda._sleep(20_000_000)
            batch = runner.build(entries)
            waits = batch.stream["stream_id"]
        assert (waits == torch.cuda.current_stream().stream_id) == (busy is None)
        batch = busy(batch) if busy else batch
        with torch.no_grad():
            results.append(m.forward(batch, runner.cache).clone())
        torch.cuda.synchronize()
    assert all(torch.equal(r, results[0]) for r in results)
