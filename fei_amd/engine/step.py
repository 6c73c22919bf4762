"""One step of many sequences: the batch a model runs, and its runner.

A step takes, for each of several sequences, the next tokens of that
sequence: one token of a sequence that decodes, a portion of any length of
one that still reads its prompt. ``RaggedBatch`` packs them into flat rows,
decoding sequences first, so that every row-wise operation (projections,
norms, feed-forwards) runs once over all rows, and each mixer runs its decode
kernels over the first ``n_dec`` rows and its prompt kernels over the rest.

``StepRunner`` owns the cache and the bookkeeping of positions. Everything
that runs such a model goes through it: LocalEngine, the session scheduler
and the trace runner.
"""

from __future__ import annotations

from dataclasses import dataclass, field
from typing import Dict, List, Optional, Sequence, Tuple

import numpy as np
import torch

from fei_amd.engine.kv_cache import HybridCache

CHUNK = 64           # tokens per chunk of the linear-attention prompt kernels
Q_TILE = 128         # query rows per workgroup of the prompt attention kernel


def upload(arrays: Sequence[np.ndarray], device: torch.device
           ) -> List[torch.Tensor]:
    """The arrays on the device, 16-byte aligned views of one copy that the current
    stream makes and nobody waits for (who reads them on another stream has to): a copy
    from ordinary memory holds the host up until the GPU has done all that it was given. A
    step of prompts made ten of those, while the GPU had little to do: 1297 rows and 4
    tokens of tobarax-1b 4846 us, 4654 so; 1700 and 6 of bokenex-1b 4090, 3961."""
    arrays = [np.ascontiguousarray(a) for a in arrays]
    if device.type != "cuda":
        return [torch.from_numpy(a).to(device) for a in arrays]
    if torch.cuda.is_current_stream_capturing():
        # a replay would copy what lies there then
        raise RuntimeError("a step's batch cannot be built while a stream is captured")
    at, size = [], 0
    for a in arrays:
        at.append(size)
        size += -(-a.nbytes // 16) * 16
    host = torch.empty(size, dtype=torch.uint8, pin_memory=True)
    flat = host.numpy()
    for a, o in zip(arrays, at):
        flat[o:o + a.nbytes] = a.reshape(-1).view(np.uint8)
    dev = host.to(device, non_blocking=True)
    return [dev[o:o + a.nbytes].view(torch.from_numpy(a).dtype).view(a.shape)
            for a, o in zip(arrays, at)]


@dataclass
class RaggedBatch:
    """Device tensors of one step. Sequences are numbered 0 .. n_seq-1 in row
    order, the ``n_dec`` single-token ones first."""
    tokens: torch.Tensor               # [T] int64
    pos: torch.Tensor                  # [T] int32
    row_seq: torch.Tensor              # [T] int32, sequence of a row
    table: torch.Tensor                # [n_seq, W] int32, physical blocks
    slots: torch.Tensor                # [n_seq] int32
    n_dec: int
    # prompt portions, host side: (first row, rows, first position)
    portions: List[Tuple[int, int, int]] = field(default_factory=list)
    want_rows: Optional[torch.Tensor] = None     # [n] int64; None = all rows
    # device tensors that depend on the portions, by key (see below)
    _plans: Dict[object, object] = field(default_factory=dict)
    # the stream that uploads them all, by its numbers, as batches are copied; None = they
    # are there
    stream: Optional[Dict[str, int]] = None

    @property
    def n_rows(self) -> int:
        return self.tokens.shape[0]

    def settle(self) -> None:
        """What runs from now on in the current stream finds the tensors there. A capture
        begins behind them, and is not to wait for what is not captured."""
        if self.stream is not None:
            now = torch.cuda.current_stream(self.stream["device_index"])
            if (now.stream_id != self.stream["stream_id"]
                    and not torch.cuda.is_current_stream_capturing()):
                now.wait_stream(torch.cuda.Stream(**self.stream))
                self.table.record_stream(now)    # and all that was uploaded with it

    def plan_arrays(self, key) -> List[np.ndarray]:
        """Of one of the plans below: "spans", ("keys", window), "chunks"."""
        if key == "chunks":
            chunks, spans = [], []
            for p, (row, n, pos0) in enumerate(self.portions):
                first = len(chunks)
                chunks += [[p, row + c, min(CHUNK, n - c)]
                           for c in range(0, n, CHUNK)]
                spans.append([first, len(chunks) - first, pos0,
                              self.n_dec + p])
            out = [(chunks, 3), (spans, 4)]
        else:
            tiles = [[p, q] for p, (_, n, _) in enumerate(self.portions)
                     for q in range(0, n, Q_TILE)]
            out = [(self.portions, 3), (tiles, 2)]
        if key[0] == "keys":
            spans, owner, at = [], [], 0
            for p, (row, n, pos0) in enumerate(self.portions):
                k0 = 0 if key[1] is None else max(0, pos0 - key[1] + 1)
                spans.append([row, n, pos0, k0, at])
                owner.append(np.full(pos0 + n - k0, p, dtype=np.int32))
                at += pos0 + n - k0
            out = [(spans, 5), (tiles, 2), (np.concatenate(owner), 1)]
        return [np.asarray(a, dtype=np.int32).reshape(-1, w) for a, w in out]

    def _upload(self, rows: np.ndarray, width: int) -> torch.Tensor:
        # for whoever asks first, and there when the host goes on
        return torch.from_numpy(rows).view(-1, width).to(self.tokens.device)

    def _plan(self, key) -> List[torch.Tensor]:
        if key not in self._plans:
            self._plans[key] = [self._upload(a, a.shape[1])
                                for a in self.plan_arrays(key)]
        return self._plans[key]

    def span_plan(self):
        """The prompt portions [first row, rows, first position], and their
        query tiles [portion, first row in it]."""
        return tuple(self._plan("spans"))

    def key_plan(self, window: Optional[int]):
        """What the prompt portions read through a window: per portion
        [first row, rows, first position, first key position, first packed
        key], the number of packed keys, the query tiles [portion, first row
        in it], and the portion of every packed key."""
        spans, tiles, owner = self._plan(("keys", window))
        return spans, owner.shape[0], tiles, owner.view(-1)

    def chunk_plan(self):
        """Chunks of the prompt portions [portion, first row, rows], and per
        portion [first chunk, chunks, first position, state slot index]."""
        return tuple(self._plan("chunks"))


@dataclass
class StepEntry:
    seq: int                           # sequence id of the runner's cache
    tokens: Sequence[int]
    want: Sequence[int] = ()           # places in tokens whose logits to give


class StepRunner:
    def __init__(self, model, num_blocks: int, num_slots: int,
                 block_size: int = 64):
        self.model = model
        self.device = model.device
        self.cache: HybridCache = model.new_cache(num_blocks, num_slots,
                                                  block_size)
        self.length: Dict[int, int] = {}      # tokens run, by sequence
        # what its mixers read of a batch's prompt portions
        self.plans = list(dict.fromkeys(
            m.plan for m in model.mixers() if m.plan is not None))

    # -- sequences -----------------------------------------------------------

    def admit(self, reserve: int = 0) -> int:
        """A new sequence with blocks for ``reserve`` tokens; MemoryError if
        slots or blocks are short (nothing is kept then)."""
        sid = self.cache.new_sequence()
        try:
            self.cache.ensure_capacity(sid, reserve)
        except MemoryError:
            self.cache.release(sid)
            raise
        self.length[sid] = 0
        return sid

    def release(self, sid: int) -> None:
        self.cache.release(sid)
        self.length.pop(sid, None)

    def set_length(self, sid: int, n: int) -> None:
        """The sequence's next token is at position ``n``: 0 to start over,
        or what the caller ran on the device by itself."""
        self.length[sid] = n

    # -- steps ---------------------------------------------------------------

    def _tables(self, seqs: Sequence[int]) -> Tuple[np.ndarray, np.ndarray]:
        blocks = [self.cache.table(s).blocks for s in seqs]
        W = max(max((len(b) for b in blocks), default=1), 1)
        host = np.full((len(seqs), W), self.cache.scratch_block, np.int32)
        for i, b in enumerate(blocks):
            host[i, :len(b)] = b
        return host, np.array([self.cache.slot(s) for s in seqs], np.int32)

    def build(self, entries: Sequence[StepEntry],
              all_rows: bool = False) -> RaggedBatch:
        """Reserve cache room for the entries and pack them. Wanted rows are
        in the order of the entries (all rows in packed order if
        ``all_rows``)."""
        if not entries:
            raise ValueError("a step needs at least one entry")
        seqs = [e.seq for e in entries]
        if len(set(seqs)) != len(seqs):
            raise ValueError("a sequence may appear once in a step")
        V = self.model.spec.vocab_size
        limit = self.model.max_seq_len
        for e in entries:
            if not len(e.tokens):
                raise ValueError("an entry needs at least one token")
            t = np.asarray(e.tokens)
            if t.min() < 0 or t.max() >= V:
                raise ValueError(f"token outside the vocabulary of {V}")
            if any(w < 0 or w >= len(e.tokens) for w in e.want):
                raise ValueError("a wanted place is outside the entry")
            if self.length[e.seq] + len(e.tokens) > limit:
                raise ValueError(f"sequence longer than {limit} tokens")
        for e in entries:
            self.cache.ensure_capacity(e.seq,
                                       self.length[e.seq] + len(e.tokens))
        order = sorted(range(len(entries)),
                       key=lambda i: len(entries[i].tokens) > 1)
        # token, position and sequence of every row
        meta = np.empty((3, sum(len(e.tokens) for e in entries)), np.int32)
        portions: List[Tuple[int, int, int]] = []
        first_row: Dict[int, int] = {}
        n_dec = row = 0
        for s, i in enumerate(order):
            e = entries[i]
            p0, n = self.length[e.seq], len(e.tokens)
            first_row[i] = row
            if n == 1:
                n_dec += 1
            else:
                portions.append((row, n, p0))
            meta[0, row:row + n] = e.tokens
            meta[1, row:row + n] = np.arange(p0, p0 + n)
            meta[2, row:row + n] = s
            row += n
        table, slots = self._tables([entries[i].seq for i in order])
        want = [first_row[i] + w for i, e in enumerate(entries)
                for w in e.want]
        batch = RaggedBatch(None, None, None, None, None, n_dec, portions)
        arrays = [meta[0].astype(np.int64), meta[1], meta[2], table, slots,
                  np.array(want, np.int64)]
        plans = [batch.plan_arrays(key) for key in self.plans if portions]
        dev = upload(arrays + sum(plans, []), self.device)
        if self.device.type == "cuda":
            now = torch.cuda.current_stream(self.device)
            batch.stream = {n: getattr(now, n) for n in (
                "stream_id", "device_index", "device_type")}
        (batch.tokens, batch.pos, batch.row_seq, batch.table, batch.slots,
         batch.want_rows) = dev[:6]
        if all_rows:
            batch.want_rows = None
        at = 6
        for key, plan in zip(self.plans, plans):
            batch._plans[key] = dev[at:at + len(plan)]
            at += len(plan)
        return batch

    @torch.no_grad()
    def step(self, entries: Sequence[StepEntry],
             all_rows: bool = False) -> torch.Tensor:
        """Run one batch; float32 logits [wanted, vocab]."""
        batch = self.build(entries, all_rows)
        logits = self.model.forward(batch, self.cache)
        for e in entries:
            self.length[e.seq] += len(e.tokens)
        return logits

    def decode_batch(self, seqs: Sequence[int], room: int,
                     tokens: Optional[Sequence[int]] = None) -> RaggedBatch:
        """A batch of one token per sequence whose ``tokens`` and ``pos`` the
        caller advances in place; blocks for ``room`` more tokens are
        reserved. The caller reports what it ran with ``set_length``."""
        for s in seqs:
            if self.length[s] + room > self.model.max_seq_len:
                raise ValueError("sequence longer than "
                                 f"{self.model.max_seq_len} tokens")
            self.cache.ensure_capacity(s, self.length[s] + room)
        dev = self.device
        table, slots = (torch.from_numpy(a).to(dev)
                        for a in self._tables(seqs))
        return RaggedBatch(
            tokens=torch.tensor(list(tokens) if tokens is not None
                                else [0] * len(seqs),
                                dtype=torch.int64, device=dev),
            pos=torch.tensor([self.length[s] for s in seqs],
                             dtype=torch.int32, device=dev),
            row_seq=torch.arange(len(seqs), dtype=torch.int32, device=dev),
            table=table, slots=slots, n_dec=len(seqs))
