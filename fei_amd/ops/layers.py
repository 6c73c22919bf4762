"""Layers of a Llama-style decoder over few rows, each launched from one call
(csrc/layers.hip), and in one launch a whole decoding step of one row
(csrc/decode_one.hip) and a whole encoder of few (csrc/encoder_one.hip). bfloat16 GPU
tensors only, and of the step fp8 weights."""

from __future__ import annotations

import ctypes
import math
from typing import Optional, Sequence, Tuple

import torch

import fei_amd.ops as _ops     # half made yet: it imports this
from fei_amd.ops import tiles as _tiles
from fei_amd.ops.mixers import SKINNY_ROWS

_vp, _i, _f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
_BF16 = torch.bfloat16


class _FewRows(ctypes.Structure):
    """FewRows of csrc/layers.hip."""
    _fields_ = ([(n, _i) for n in ("B", "S", "C", "I", "Hq", "Hkv", "D", "room",
                                   "bs_log", "W", "splits")] +
                [("eps", _f), ("scale", _f)] +
                [(n, _vp) for n in ("pos", "table", "cos_sin", "po", "pml")])


class _OneShape(ctypes.Structure):
    """OneShape of csrc/decode_one.hip."""
    _fields_ = ([(n, _i) for n in ("layers", "C", "I", "Hq", "Hkv", "D", "room",
                                   "vocab", "fp8", "blocks")] +
                [("eps", _f), ("scale", _f)])


class _EncoderShape(ctypes.Structure):
    """EncoderShape of csrc/encoder_one.hip."""
    _fields_ = ([(n, _i) for n in ("layers", "B", "S", "H", "C", "I", "blocks")] +
                [("eps", _f), ("scale", _f)])


ONE_BLOCKS = 256               # of decode_one.hip and encoder_one.hip, one a CU


def declare(lib: ctypes.CDLL) -> None:
    lib.fei_llama_few.argtypes = [_vp, _i] + [_vp] * 8
    lib.fei_decode_one_room.argtypes = [_vp]
    lib.fei_decode_one_room.restype = ctypes.c_long
    lib.fei_decode_one.argtypes = [_vp] * 8
    lib.fei_encoder_one_room.argtypes = [_vp]
    lib.fei_encoder_one_room.restype = ctypes.c_long
    lib.fei_encoder_one.argtypes = [_vp] * 7


def _pointers(tensors, shapes, device: int, grad: bool):
    """Where kernels find the tensors, 16 bytes at a time, or None if one is not what
    lies there."""
    out = []
    for t, shape in zip(tensors, shapes):
        p = t.data_ptr()
        if not (t.dtype is _BF16 and t.shape == shape and t.is_contiguous()
                and t.get_device() == device and not p % 16
                and _tiles.types_ok(t) and not (grad and t.requires_grad)):
            return None
        out.append(p)
    return out


def llama_few(h: torch.Tensor, layers: Sequence, k_caches: Sequence[torch.Tensor],
              v_caches: Sequence[torch.Tensor], heads: int, eps: float,
              pos: torch.Tensor, rope: torch.Tensor, splits: int = 0,
              workspace=None, table: Optional[torch.Tensor] = None, S: int = 0,
              attn_out: Optional[torch.Tensor] = None
              ) -> Tuple[int, Optional[torch.Tensor]]:
    """``layers`` over the rows h [M, C], in place: a decoding step's, or (``S``) those
    of prompts of S tokens. Caches [B, Hkv, room, D], or with a ``table`` pools
    [blocks, Hkv, size, D]; at pos[b] and on the rows' keys and values are written.
    ``workspace``: see attn_decode; ``attn_out``: room for M rows of its results, if the
    caller has some. Returns how many layers are done, up to the first that
    the kernels for few rows do not take, and what a norm's product behind them takes as
    ``sums``. The launches, and their order, are those of the operations one by one, but of
    one decoded row: there the output product sums few splits of the keys itself, in
    another order than the launch that is left out, and nothing is left in ``attn_out``. A
    layer a call: the GPU has the first one's while the others are looked at (all 16 looked
    at first, a step of 20 sessions took 1130 us, 1068 one by one)."""
    M, C = h.shape
    lw, grad = layers[0], torch.is_grad_enabled()
    if not (h.is_cuda and 0 < M <= SKINNY_ROWS and 0 < C <= 16384
            and k_caches[0].dim() == 4 and (not S or M % S == 0)):
        return 0, None
    Hkv, room, D = k_caches[0].shape[1:]
    HD, width, I = heads * D, (heads + 2 * Hkv) * D, lw.wdown.shape[-1]
    B, dev, bs_log, W = M // (S or 1), h.get_device(), 0, 0
    cache = k_caches[0].shape if table is not None else (B, Hkv, room, D)
    if not (dev == torch.cuda.current_device() and D in (64, 128) and I > 0 < Hkv
            and heads % Hkv == 0 and heads // Hkv <= 16
            and not any(n % (64 if M > 1 else 8) for n in (C, HD, I))
            and _pointers((h,), ((M, C),), dev, grad)
            and rope.dtype is torch.float32 and pos.dtype is torch.int32
            and pos.is_contiguous() and rope.is_contiguous()
            and pos.get_device() == rope.get_device() == dev and pos.numel() == B
            and not rope.data_ptr() % 16 and _tiles._memory(pos, rope)):
        return 0, None
    if table is not None:
        if not (table.dtype is torch.int32 and table.is_contiguous()
                and table.shape[0] == B and table.get_device() == dev
                and not room & (room - 1) and not S):
            return 0, None
        bs_log, W = room.bit_length() - 1, table.shape[1]
        room = W << bs_log
    if S:
        splits = _ops._prefill_splits(B, Hkv, S * (heads // Hkv), room, D)
        n = M * heads * splits if splits > 1 else 0
        ws = torch.empty(n * (D + 2), dtype=torch.float32, device=h.device)
        po, pml = ws.data_ptr(), ws.data_ptr() + n * D * 4
    else:
        if not 0 < splits <= 64:
            return 0, None
        if workspace is None:
            workspace = [torch.empty(B, heads, splits, n, dtype=torch.float32,
                                     device=h.device) for n in (D, 2)]
        po, pml = (t.data_ptr() for t in workspace[:2])
        assert all(t.shape[2] == splits for t in workspace[:2])

    def rows(n):
        return torch.empty(M, n, dtype=h.dtype, device=h.device)
    att = attn_out if attn_out is not None else rows(HD)
    if not (_pointers((att,), (att.shape,), dev, False) and att.numel() == M * HD):
        return 0, None
    room_for = [rows(width), att, rows(I), rows(C)]
    sums = torch.empty(M, -(-C // (8 if C <= 2048 else 16)), dtype=torch.float32,
                       device=h.device)
    p = _FewRows(B, S, C, I, heads, Hkv, D, room, bs_log, W, splits, eps,
                 1.0 / math.sqrt(D), pos.data_ptr(),
                 None if table is None else table.data_ptr(), rope.data_ptr(), po,
                 pml)
    args = (h.data_ptr(), *(t.data_ptr() for t in room_for), sums.data_ptr(),
            ctypes.byref(p), _ops._stream())
    launch = _ops.require_lib().fei_llama_few
    shapes = ((C,), (width, C), (C, HD), (C,), (2 * I, C), (C, I), cache, cache)
    done = 0
    for lw, kc, vc in zip(layers, k_caches, v_caches):
        at = _pointers((lw.norm_attn, lw.wqkv, lw.wo, lw.norm_mlp, lw.wgu, lw.wdown,
                        kc, vc), shapes, dev, grad)
        if at is None:
            break
        launch((_vp * 8)(*at), done, *args)
        done += 1
    return done, sums if done and M > 1 else None


def llama_one_pays(layers: int, weights: int, head: int, fp8: bool) -> bool:
    """Whether a captured step of one row is faster in one launch than as a chain, by the
    numbers of weights of a layer and of the head. The launch costs 10 us more, and gains a
    layer what the chain's five launches cost beyond their bytes: of few weights nothing, as
    its seams are no shorter; fp8's are as long for half the bytes. Steps of 30 keys by a
    graph, us, the chain's first. Layers of 1.8 million weights: 2 of them 46, 58; 24 434,
    463. Of 6: 12 245, 245, 24 482, 469; of 8.9: 8 171, 174; of 12.8 and 15.9: 8 191, 178
    and 200, 186; of 44: 24 763, 670; of 61, two and three 83, 85 and 119, 115. fp8: of 12.8
    24 522, 530; of 25 8 203, 199 (1000 keys 210, 214); of 34.6 8 228, 209; of 44 24 666,
    597; of 61, two and three 71, 74 and 100, 99. The head's product is no faster: of 262
    million weights behind layers of 61 takes 4 of them as long, 223, and 8 370, 354."""
    return (weights >= (32 if fp8 else 10) * 10 ** 6
            and layers * weights >= max(120 * 10 ** 6, head))


def llama_one(h: torch.Tensor, layers: Sequence, k_caches: Sequence[torch.Tensor],
              v_caches: Sequence[torch.Tensor], heads: int, eps: float,
              pos: torch.Tensor, rope: torch.Tensor, norm: torch.Tensor,
              head: torch.Tensor, fp8: Optional[Sequence] = None,
              fp8_head: Optional[Tuple[torch.Tensor, torch.Tensor]] = None,
              blocks: int = ONE_BLOCKS) -> Optional[torch.Tensor]:
    """A decoding step of one row h [1, C], which is left as it is, in one launch of
    csrc/decode_one.hip: logits [1, vocab], or None where it does not take the step. Caches
    [1, Hkv, room, D]; keys and values are written at pos[0]. ``fp8``: of each layer the
    products' names -> (w, scales). ``blocks``: up to 256; fewer have items taken by ticket."""
    M, C = h.shape
    lw, grad = layers[0], torch.is_grad_enabled()
    if not (h.is_cuda and M == 1 and k_caches[0].dim() == 4 and len(layers) > 0):
        return None
    Hkv, room, D = k_caches[0].shape[1:]
    I, vocab, dev = lw.wdown.shape[-1], head.shape[0], h.get_device()
    HD, width, cache = heads * D, (heads + 2 * Hkv) * D, (1, Hkv, room, D)
    shape = _OneShape(len(layers), C, I, heads, Hkv, D, room, vocab, fp8 is not None,
                      blocks, eps, 1.0 / math.sqrt(D))
    lib = _ops.require_lib()
    if not (Hkv > 0 and dev == torch.cuda.current_device()
            and torch.cuda.get_device_properties(dev).multi_processor_count >= ONE_BLOCKS
            and rope.dtype is torch.float32 and pos.dtype is torch.int32
            and pos.is_contiguous() and rope.is_contiguous() and pos.numel() == 1
            and pos.get_device() == rope.get_device() == dev
            and rope.shape == (rope.shape[0], D // 2, 2) and rope.shape[0] >= room
            and not rope.data_ptr() % 16 and _tiles._memory(pos, rope)):
        return None
    size = lib.fei_decode_one_room(ctypes.byref(shape))
    shapes = ((width, C), (C, HD), (2 * I, C), (C, I))
    ends = _pointers((h, norm), ((1, C), (C,)), dev, grad)
    if not size or ends is None:
        return None

    def weights(names, tensors, pairs):
        """Where w and its rows' scales lie."""
        if pairs is None:
            at = _pointers(tensors, names, dev, grad)
            return at and (at, [None] * len(at))
        at = ([], [])
        for (w, scale), (N, K) in zip(pairs, names):
            if not (w.dtype is torch.uint8 and w.shape == (N, K) and w.is_contiguous()
                    and scale.dtype is torch.float32 and scale.numel() == N
                    and scale.is_contiguous() and not w.data_ptr() % 16
                    and w.get_device() == scale.get_device() == dev
                    and _tiles.types_ok(w, scale)):
                return None
            at[0].append(w.data_ptr())
            at[1].append(scale.data_ptr())
        return at

    table = []
    for i, (lw, kc, vc) in enumerate(zip(layers, k_caches, v_caches)):
        q = fp8 and [fp8[i][n] for n in ("wqkv", "wo", "wgu", "wdown")]
        at = weights(shapes, (lw.wqkv, lw.wo, lw.wgu, lw.wdown), q)
        rest = _pointers((lw.norm_attn, lw.norm_mlp, kc, vc),
                         ((C,), (C,), cache, cache), dev, grad)
        if at is None or rest is None:
            return None
        table += [*at[0], *at[1], *rest]
    at = weights(((vocab, C),), (head,), fp8 and [fp8_head])
    if at is None or len(table) != 12 * len(layers):
        return None
    table += [at[0][0], at[1][0], ends[1]]
    room_for = torch.empty(size, dtype=torch.uint8, device=h.device)
    out = torch.empty(1, vocab, dtype=h.dtype, device=h.device)
    lib.fei_decode_one((_vp * len(table))(*table), ctypes.byref(shape), ends[0],
                       out.data_ptr(), room_for.data_ptr(), pos.data_ptr(),
                       rope.data_ptr(), _ops._stream())
    return out


def encoder_one(ids: torch.Tensor, tok: torch.Tensor, pos: torch.Tensor,
                gain: torch.Tensor, shift: torch.Tensor, weights, heads: int,
                dim: int, inner: int, lens: torch.Tensor, eps: float,
                blocks: int = ONE_BLOCKS) -> Optional[torch.Tensor]:
    """An encoder over up to 128 rows in one launch of csrc/encoder_one.hip, behind that
    of the embeddings: arguments and result are encoder_packed's; None where it does not
    take them. ``blocks``: up to 256; fewer have items taken by ticket."""
    if not (tok.is_cuda and ids.dim() == 2 and 0 < ids.numel() <= 128 and dim == 64
            and _ops._embedding_ok(ids, tok, pos, gain, shift)):
        return None
    (B, S), C, dev = ids.shape, tok.shape[1], ids.get_device()
    shape = _EncoderShape(len(weights) // 12, B, S, heads, C, inner, blocks, eps,
                          1.0 / math.sqrt(dim))
    lib = _ops.require_lib()
    size = lib.fei_encoder_one_room(ctypes.byref(shape))
    if not (size and torch.cuda.get_device_properties(dev).multi_processor_count
            >= ONE_BLOCKS
            and all(t.get_device() == dev for t in weights)
            and not (torch.is_grad_enabled() and any(t.requires_grad for t in weights))
            and lens.device == ids.device and lens.dtype is torch.int32
            and lens.shape == (B,) and lens.is_contiguous()
            and _tiles.types_ok(lens, *weights)):
        return None
    at = _ops._encoder_weights(weights, C, heads * dim, inner)
    if at is None:
        return None
    h = _ops.embed_layernorm(ids, tok, pos, gain, shift, eps, tok.dtype)
    room = torch.empty(size, dtype=torch.uint8, device=ids.device)
    out = torch.empty(B, C, dtype=torch.float32, device=ids.device)
    lib.fei_encoder_one((_vp * len(at))(*at), ctypes.byref(shape), h.data_ptr(),
                        out.data_ptr(), room.data_ptr(), lens.data_ptr(),
                        _ops._stream())
    return out
