"""Ops of decoders made of unlike layers (models/tobarax.py, models/bokenex.py,
models/mixers.py).

Same dispatch rule as the rest of ``fei_amd.ops``: GPU tensors go to the HIP
kernels (csrc/hybrid.hip, latent_attn.hip, gla.hip), in bfloat16 or float32 by
the dtype of the rows; CPU tensors to the reference implementations.
"""

from __future__ import annotations

import ctypes
from typing import Optional, Tuple

import torch

import fei_amd.ops as _ops     # half made yet: it imports this
from fei_amd.ops import reference as ref
from fei_amd.ops import rows as _rows
from fei_amd.ops import tiles as _tiles
from fei_amd.ops.rows import SKINNY_ROWS

_c = ctypes
_vp, _i, _f, _l = _c.c_void_p, _c.c_int, _c.c_float, _c.c_long

MAX_SPLITS = 64          # splits of a decode row's keys
TARGET_BLOCKS = 256      # workgroups of a decode attention launch


def declare(lib: ctypes.CDLL) -> None:
    lib.fei_norm_pair.argtypes = [_vp] * 5 + [_i, _i, _f, _i, _vp]
    lib.fei_cat_cast.argtypes = [_vp, _vp, _vp, _i, _i, _i, _vp]
    lib.fei_swiglu_rows.argtypes = [_vp, _l, _vp, _l, _i, _i, _i, _vp]
    lib.fei_softcap.argtypes = [_vp, _l, _f, _f, _vp]
    lib.fei_gemv_mix_in.argtypes = [_vp] * 5 + [_l] + [_i] * 4 + [_i, _vp]
    lib.fei_gemv_f32.argtypes = [_vp] * 4 + [_i] * 3 + [_i, _f, _f, _i, _vp]
    lib.fei_embed_pos.argtypes = [_vp] * 5 + [_i] * 3 + [_vp]
    lib.fei_relu2_rows.argtypes = [_vp, _l, _vp, _l, _i, _i, _i, _vp]
    lib.fei_gemv_gain.argtypes = [_vp] * 4 + [_f] + [_i] * 3 + [_vp]
    lib.fei_gemv_parallel_in.argtypes = (
        [_vp] * 5 + [_f] + [_vp, _l] + [_i] * 5 + [_vp])
    lib.fei_latent_decode.argtypes = (
        [_vp, _l, _vp, _l] + [_vp] * 10 + [_i] * 8 +
        [_f, _i, _f, _i, _i, _i, _vp, _i] + [_vp] * 4 + [_i, _vp])
    lib.fei_latent_decode.restype = _i
    lib.fei_latent_append.argtypes = (
        [_vp, _l] + [_vp] * 6 + [_i] * 8 + [_f, _i, _vp])
    lib.fei_latent_gather.argtypes = [_vp] * 6 + [_i] * 7 + [_vp]
    lib.fei_window_prefill.argtypes = (
        [_vp, _l, _vp, _l] + [_vp] * 4 + [_i] * 6 + [_f, _i, _i, _vp])
    lib.fei_gla_decode.argtypes = (
        [_vp, _l, _vp, _vp, _vp, _l] + [_vp] * 5 + [_i] * 5 + [_f, _f, _i, _vp])
    lib.fei_gla_prefill.argtypes = (
        [_vp, _l, _vp, _l] + [_vp] * 5 + [_i, _vp, _i] + [_vp] * 4 +
        [_i, _vp, _vp] + [_i] * 4 + [_f, _f, _i, _vp])


def _lib() -> ctypes.CDLL:
    return _ops.require_lib()


def _stream() -> int:
    return _ops._stream()


def _p(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def _f32(t: torch.Tensor) -> int:
    """Element switch of the kernels: 0 = bfloat16, 1 = float32."""
    if t.dtype == torch.float32:
        return 1
    if t.dtype != torch.bfloat16:
        raise TypeError(f"rows must be bfloat16 or float32, not {t.dtype}")
    return 0


# -- row-wise ops ----------------------------------------------------------------

def norm_pair(x: torch.Tensor, w1: torch.Tensor, w2: Optional[torch.Tensor],
              eps: float, dtype: torch.dtype
              ) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """x [T, C] float32 -> (norm(x) * w1, norm(x) * w2) in ``dtype``; the
    second is None without w2."""
    if not x.is_cuda:
        return ref.norm_pair(x, w1, w2, eps, dtype)
    x = x.contiguous()
    T, C = x.shape
    o1 = torch.empty(T, C, dtype=dtype, device=x.device)
    o2 = None if w2 is None else torch.empty_like(o1)
    if T:
        _lib().fei_norm_pair(_p(o1), _p(o2), _p(x), _p(w1), _p(w2), T, C, eps,
                             _f32(o1), _stream())
    return o1, o2


def cat_cast(x: torch.Tensor, y: torch.Tensor,
             dtype: torch.dtype) -> torch.Tensor:
    """[x; y] along columns, float32 -> ``dtype``."""
    if not x.is_cuda:
        return torch.cat([x, y], dim=-1).to(dtype)
    T, C = x.shape
    out = torch.empty(T, 2 * C, dtype=dtype, device=x.device)
    _lib().fei_cat_cast(_p(out), _p(x.contiguous()), _p(y.contiguous()), T, C,
                        _f32(out), _stream())
    return out


def embed_pos(tokens: torch.Tensor, pos: torch.Tensor, emb: torch.Tensor,
              pos_emb: torch.Tensor) -> torch.Tensor:
    """emb[tokens] + pos_emb[pos], float32 [T, C]."""
    if not emb.is_cuda:
        return emb[tokens.long()].float() + pos_emb[pos.long()].float()
    T, C = tokens.shape[0], emb.shape[1]
    out = torch.empty(T, C, dtype=torch.float32, device=emb.device)
    if tokens.dtype not in (torch.int32, torch.int64):
        raise TypeError(f"token ids are {tokens.dtype}")
    if T:
        _lib().fei_embed_pos(
            _p(out), _p(tokens.contiguous()), _p(pos), _p(emb), _p(pos_emb),
            T, C, _f32(emb) | (2 if tokens.dtype == torch.int64 else 0),
            _stream())
    return out


class GainNorm:
    """RMS norm with one gain for all columns."""

    def __init__(self, gain: torch.Tensor, width: int, eps: float):
        self.gain, self.eps = gain, eps
        # as a weight per column, for the norm of rows
        self.cols = gain.expand(width).contiguous()


class GainNormed:
    """Rows x (float32) under a GainNorm. The gain and the root mean square
    commute with a product, so a product of a row or two takes x as it is
    and makes the norm inside; the others take the normed ``rows``."""

    def __init__(self, x: torch.Tensor, norm: GainNorm, dtype: torch.dtype,
                 rows: Optional[torch.Tensor] = None):
        self.x, self.norm, self.dtype = x, norm, dtype
        self._rows = rows

    @property
    def rows(self) -> torch.Tensor:
        if self._rows is None:
            self._rows, _ = norm_pair(self.x, self.norm.cols, None,
                                      self.norm.eps, self.dtype)
        return self._rows

    @property
    def inside(self) -> bool:
        """Whether products make the norm inside."""
        return (self.x.is_cuda and self.dtype == torch.bfloat16
                and self.x.shape[0] <= 2 and self.x.shape[1] % 8 == 0
                and self.x.shape[0] > 0)


_BF16 = torch.bfloat16


def match(x: torch.Tensor, w: torch.Tensor, K: int) -> bool:
    """Whether pointers stand for x [.., K], or a copy without gaps, and w
    [N, K] in a kernel: bfloat16, w without gaps, sizes that fit, on one device;
    and nobody asks for a gradient, which the library's products have."""
    # 1 us, once or twice a launch: get_device, which is -1 of the CPU, is a
    # third of what comparing devices takes
    size = w.shape
    return (x.dtype is _BF16 and w.dtype is _BF16 and len(size) == 2
            and size[1] == K and w.is_contiguous()
            and x.get_device() == w.get_device()
            and not ((x.requires_grad or w.requires_grad)
                     and torch.is_grad_enabled()))


def plain(x: torch.Tensor, w: torch.Tensor) -> bool:
    """The same for x as it lies."""
    return x.is_contiguous() and match(x, w, x.shape[-1])


def dense(t: torch.Tensor, dtype: torch.dtype, like: torch.Tensor,
           *shape: int) -> bool:
    """Whether a pointer stands for t of this type and shape."""
    return (t.dtype == dtype and t.shape == shape and t.is_contiguous()
            and t.device == like.device)


def gemv_sizes(T: int, K: int) -> bool:
    return T in (1, 2, 4, 8) and K % 8 == 0


def _gemv_rows(T: int, K: int, x: torch.Tensor, w: torch.Tensor) -> bool:
    return gemv_sizes(T, K) and plain(x, w)


# What becomes of a skinny product's sums (csrc/fei_epilogue.h).
(EPI_BF16, EPI_F32, EPI_RES, EPI_PARALLEL, EPI_RES_BF16, EPI_SWIGLU,
 EPI_GELU) = range(7)


def skinny_sizes(T: int, K: int, x: torch.Tensor, w: torch.Tensor,
                 least: int = 3) -> bool:
    """Rows and sizes that the matrix-core tile for few rows takes: its loads
    are of 16 bytes, 128 a row. From 3 rows on it beats the vector units (whole
    decoding steps, 3 rows: 3.24 ms for 4.75 on 8B, 0.79 for 1.12 on 1B), from 2
    (``least``) where it also makes the norm or adds to the residual (3.01 for
    3.54, 0.84 for 0.88); beyond 32 its repeated reads of x cost more than the
    library's."""
    return (least <= T <= SKINNY_ROWS and K > 0 and K % 64 == 0
            and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0)


def skinny_ok(T: int, K: int, x: torch.Tensor, w: torch.Tensor,
              least: int = 3) -> bool:
    return skinny_sizes(T, K, x, w, least) and plain(x, w)


def skinny(out, x, w, n: int, epi: int, bias=None, scale: float = 1.0,
           cap: float = 0.0, n_mix: int = 0, router=None, act=None,
           stride: int = 0, bias16=None, norm=None, sums_out=None) -> None:
    """x [T, K] with the rows of ``w``: ``n`` results a row. ``norm``: (gains,
    sums of squares, eps) of an RMS norm that x is under."""
    T, K = x.shape
    gain, sums, eps = norm or (None, None, 0.0)
    of = sums if sums is not None else sums_out
    tiles = 0 if of is None else of.shape[1]
    _lib().fei_skinny(_p(out), _p(x), _p(w), T, n, K, epi, _p(bias), scale,
                      cap, n_mix, 0 if router is None else router.shape[1],
                      _p(router), _p(act), stride, _p(bias16), _p(gain),
                      _p(sums), tiles, eps, _p(sums_out), _stream())


def _linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x [T, K] @ w^T of more rows than the kernels for few take."""
    if (x.shape[0] > 256 and x.stride(-1) == 1
            and _tiles.linear_ok(x.shape[0], x, w)):
        return _tiles.linear(x, w)
    return torch.nn.functional.linear(x, w)


def _act_tile(x: torch.Tensor, w: torch.Tensor, ff: int,
              act: torch.Tensor) -> bool:
    """Whether the product of many rows writes its activations, ``ff`` a row, to
    ``act`` itself."""
    return (x.shape[0] > 128 and ff % 8 == 0 and plain(x, w)
            and _tiles.act_ok(x.shape[0], x, w)
            and act.dtype is _BF16 and act.stride(1) == 1
            and act.stride(0) % 8 == 0 and act.data_ptr() % 16 == 0)


def mix_in(n1: torch.Tensor, n2: Optional[torch.Tensor], w_in: torch.Tensor,
           n_mix: int, ff: int, act: torch.Tensor) -> torch.Tensor:
    """All products of a layer's input: returns n1 @ w_in[:n_mix]^T and writes
    silu(gate) * up of n2, gate and up being the next ``ff`` rows each, into
    ``act`` (a column range of a wider buffer)."""
    T, K = n1.shape
    own = n1.is_cuda and (not ff or (
        n2.shape == n1.shape and plain(n2, w_in) and n2.data_ptr() % 16 == 0))
    if own and skinny_ok(T, K, n1, w_in):
        proj = torch.empty(T, n_mix, dtype=n1.dtype, device=n1.device)
        if n_mix:
            skinny(proj, n1, w_in, n_mix, EPI_BF16)
        if ff:
            skinny(None, n2, w_in[n_mix:], ff, EPI_SWIGLU, act=act,
                   stride=act.stride(0))
        return proj
    if own and _gemv_rows(T, K, n1, w_in):
        proj = torch.empty(T, n_mix, dtype=n1.dtype, device=n1.device)
        _lib().fei_gemv_mix_in(_p(proj), _p(act), _p(n1), _p(n2), _p(w_in),
                               act.stride(0), T, n_mix, ff, K, 1, _stream())
        return proj
    proj = _linear(n1, w_in[:n_mix])
    if ff and own and _act_tile(n2, w_in[n_mix:], ff, act):
        _tiles.product(n2, w_in[n_mix:], act, ff, _tiles.TILE_SWIGLU)
    elif ff:
        gu = torch.nn.functional.linear(n2, w_in[n_mix:])
        if n1.is_cuda:
            if T:
                _lib().fei_swiglu_rows(_p(act), act.stride(0), _p(gu),
                                       gu.stride(0), T, ff, _f32(gu),
                                       _stream())
        else:
            act.copy_(ref.swiglu(gu))
    return proj


def parallel_in(h: GainNormed, w_in: torch.Tensor, n_mix: int, ff: int,
                n_router: int, act: torch.Tensor
                ) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """All products of a parallel layer's input. The rows of ``w_in`` are
    n_mix of the mixer, whose products are returned, then either ``ff`` of a
    feed-forward, relu(.)^2 of which goes into ``act`` (a column range of a
    wider buffer), or ``n_router`` of a router, whose float32 logits are
    returned second (None without)."""
    x, norm = h.x, h.norm
    T, K = x.shape
    n = n_mix + ff + n_router
    gpu = x.is_cuda and h.dtype == torch.bfloat16
    if h.inside or (gpu and skinny_ok(T, K, h.rows, w_in)):
        proj = torch.empty(T, n_mix, dtype=h.dtype, device=x.device)
        router = torch.empty(T, n_router, dtype=torch.float32,
                             device=x.device) if n_router else None
        if h.inside:
            _lib().fei_gemv_parallel_in(
                _p(proj), _p(router), _p(x), _p(w_in), _p(norm.gain), norm.eps,
                _p(act), act.stride(0), T, n_mix, n_router, n, K, _stream())
        else:
            skinny(proj, h.rows, w_in, n, EPI_PARALLEL, n_mix=n_mix,
                   router=router, act=act, stride=act.stride(0))
        return proj, router
    rows = h.rows
    proj = _linear(rows, w_in[:n_mix])
    if ff and gpu and _act_tile(rows, w_in[n_mix:], ff, act):
        _tiles.product(rows, w_in[n_mix:], act, ff, _tiles.TILE_RELU2)
    elif ff:
        up = torch.nn.functional.linear(rows, w_in[n_mix:])
        if not x.is_cuda:
            act.copy_(ref.square_relu(up))
        elif T:
            _lib().fei_relu2_rows(_p(act), act.stride(0), _p(up),
                                  up.stride(0), T, ff, _f32(up), _stream())
    router = _mm_f32(rows, w_in[n_mix:], None) if n_router else None
    return proj, router


def gain_logits(h: GainNormed, w: torch.Tensor) -> torch.Tensor:
    """normed rows @ w^T, float32."""
    if not h.inside:
        return logits_head(h.rows, w, 1.0, None)
    T, K = h.x.shape
    out = torch.empty(T, w.shape[0], dtype=torch.float32, device=w.device)
    _lib().fei_gemv_gain(_p(out), _p(h.x.contiguous()), _p(w),
                         _p(h.norm.gain), h.norm.eps, T, w.shape[0], K,
                         _stream())
    return out


def _mm_f32(a: torch.Tensor, w: torch.Tensor,
            add: Optional[torch.Tensor]) -> torch.Tensor:
    """a @ w^T (+ add) with a float32 result; a 2-d ``add`` may be
    overwritten with it."""
    if not a.is_cuda or a.dtype == torch.float32:
        y = torch.nn.functional.linear(a.float(), w.float())
        return y if add is None else add + y
    if add is None:
        return torch.mm(a, w.t(), out_dtype=torch.float32)
    if add.dim() == 1:
        return torch.addmm(add.expand(a.shape[0], -1), a, w.t(),
                           out_dtype=torch.float32)
    return torch.addmm(add, a, w.t(), out_dtype=torch.float32, out=add)


def residual_linear(x: torch.Tensor, a: torch.Tensor, w: torch.Tensor,
                    mult: float = 1.0) -> torch.Tensor:
    """x + mult * (a @ w^T), float32; x may be overwritten with it."""
    T, K = a.shape
    own = a.is_cuda and dense(x, torch.float32, a, T, w.shape[0])
    if own and skinny_ok(T, K, a, w):
        skinny(x, a, w, w.shape[0], EPI_RES, scale=mult)
        return x
    if own and _gemv_rows(T, K, a, w):
        _lib().fei_gemv_f32(_p(x), _p(a), _p(w), None, T, w.shape[0], K, 1,
                            mult, 0.0, 1, _stream())
        return x
    if not a.is_cuda or a.dtype == torch.float32:
        return x + mult * _mm_f32(a, w, None)
    if own and _rows.add_ok(x, a, w):
        _rows.add_product(x, a, w, mult)
        return x
    if own and _tiles.parts_pay(T, w) and _tiles.add_ok(x, a, w):
        _rows.add_parts(x, _tiles.product_parts(a, w), mult)
        return x
    return torch.addmm(x, a, w.t(), out_dtype=torch.float32, alpha=mult,
                       out=x)


def _gain(g: torch.Tensor, C: int, like: torch.Tensor) -> bool:
    """Whether a pointer stands for C float32 gains, four at a time."""
    return (g.dtype is torch.float32 and g.shape[0] == C and C % 4 == 0
            and g.dim() == 1 and g.is_contiguous() and g.data_ptr() % 16 == 0
            and g.get_device() == like.get_device()
            and not (g.requires_grad and torch.is_grad_enabled()))


def residual_norms(x: torch.Tensor, a: torch.Tensor, w: torch.Tensor,
                   w1: torch.Tensor, w2: Optional[torch.Tensor], eps: float,
                   dtype: torch.dtype, mult: float = 1.0
                   ) -> Tuple[torch.Tensor, Optional[Tuple]]:
    """residual_linear, and the norm_pair of its result where one kernel makes
    both: that of many rows, whose product comes in parts. Else None, and who
    needs the norms asks for them."""
    T, C = x.shape
    if T <= SKINNY_ROWS:
        return residual_linear(x, a, w, mult), None
    if (dtype is _BF16 and a.is_cuda and a.shape[0] == T and w.shape[0] == C
            and _gain(w1, C, a) and (w2 is None or _gain(w2, C, a))
            and dense(x, torch.float32, a, T, C)):
        parts = (_rows.product_parts(a, w) if _rows.add_ok(x, a, w)
                 else _tiles.product_parts(a, w)
                 if _tiles.parts_pay(T, w) and _tiles.add_ok(x, a, w) else None)
        if parts is not None:
            return x, _rows.add_parts_norms(x, parts, mult, w1, w2, eps)
    return residual_linear(x, a, w, mult), None


def linear_f32(a: torch.Tensor, w: torch.Tensor,
               bias: torch.Tensor) -> torch.Tensor:
    """a @ w^T + bias, float32."""
    T, K = a.shape
    own = a.is_cuda and dense(bias, torch.float32, a, w.shape[0])
    if own and skinny_ok(T, K, a, w):
        out = torch.empty(T, w.shape[0], dtype=torch.float32, device=a.device)
        skinny(out, a, w, w.shape[0], EPI_F32, bias=bias)
        return out
    if own and _gemv_rows(T, K, a, w):
        out = torch.empty(T, w.shape[0], dtype=torch.float32, device=a.device)
        _lib().fei_gemv_f32(_p(out), _p(a), _p(w), _p(bias), T, w.shape[0], K,
                            0, 1.0, 0.0, 1, _stream())
        return out
    return _mm_f32(a, w, bias)


def logits_head(y: torch.Tensor, w: torch.Tensor, scale: float,
                cap: Optional[float]) -> torch.Tensor:
    """(y @ w^T) * scale, then cap * tanh(. / cap); float32."""
    T, K = y.shape
    if not y.is_cuda:
        return ref.softcap_logits(_mm_f32(y, w, None), scale, cap)
    c = float(cap or 0.0)
    if skinny_ok(T, K, y, w):
        out = torch.empty(T, w.shape[0], dtype=torch.float32, device=y.device)
        skinny(out, y, w, w.shape[0], EPI_F32, scale=scale, cap=c)
        return out
    if _gemv_rows(T, K, y, w):
        out = torch.empty(T, w.shape[0], dtype=torch.float32, device=y.device)
        _lib().fei_gemv_f32(_p(out), _p(y), _p(w), None, T, w.shape[0], K, 0,
                            scale, c, 1, _stream())
        return out
    out = _mm_f32(y, w, None)
    if T:
        _lib().fei_softcap(_p(out), out.numel(), scale, c, _stream())
    return out


# -- latent attention --------------------------------------------------------------

def check_latent_geometry(m) -> None:
    """Largest sizes the kernels are built for."""
    if m.dim + m.rot_dim > 256 or m.vdim > 256 or m.kv_rank > 1024 \
            or m.row_width > 1088:
        raise ValueError(f"latent attention sizes out of range: {m}")


def _dst(batch, lo: int, hi: Optional[int], block_size: int) -> torch.Tensor:
    """Physical cache row of batch rows lo .. hi-1."""
    pos = batch.pos[lo:hi].long()
    blk = batch.table[batch.row_seq[lo:hi].long(), pos // block_size]
    return blk.long() * block_size + pos % block_size


def _keys(batch, seq: int, lo: int, hi: int, rows, block_size: int):
    """Cached rows of positions lo .. hi-1 of a sequence."""
    p = torch.arange(lo, hi)
    blk = batch.table[seq].long()[p // block_size]
    return rows[blk * block_size + p % block_size]


def _latent_out(o, proj, m, out) -> None:
    g = proj[:, m.in_rows - m.heads * m.vdim:].float()
    out.copy_((o.flatten(1) * torch.sigmoid(g)).to(out.dtype))


def latent_attn_decode(proj, out, m, w, rot, batch, rows,
                       block_size: int) -> None:
    """One new token per sequence: cache its row, attend, gate. proj
    [B, m.in_rows] (q | latent and rotated key | gate), out [B, H*vdim]."""
    if not proj.is_cuda:
        n = batch.n_dec
        q = ref.latent_append(proj, m, w.norm, rot, w.eps, batch.pos[:n],
                              _dst(batch, 0, n, block_size), rows)
        o = torch.empty(n, m.heads, m.vdim)
        for b in range(n):
            p = int(batch.pos[b])
            k0 = 0 if m.window is None else max(0, p - m.window + 1)
            o[b] = ref.latent_attend(
                q[b:b + 1], batch.pos[b:b + 1],
                _keys(batch, b, k0, p + 1, rows, block_size), k0, m, w.uk,
                w.uv, m.scale)[0]
        _latent_out(o, proj, m, out)
        return
    _latent_decode(proj, out, m, w, rot, batch, rows, block_size, proj.shape[0],
                   (0, None, 0, None, None, None, None))


def _latent_decode(proj, out, m, w, rot, batch, rows, block_size: int, B: int,
                   beside: tuple) -> None:
    dev = proj.device
    W = batch.table.shape[1]
    n_max = W * block_size
    if m.window is not None:
        n_max = min(n_max, m.window)
    groups = B * -(-m.heads // 32)
    splits = max(1, min(MAX_SPLITS, -(-n_max // 32),
                        -(-TARGET_BLOCKS // groups)))
    per_split = -(-n_max // splits)
    tile = 32 if per_split <= 48 else 64
    qa = torch.empty(B, m.heads, m.row_width, dtype=proj.dtype, device=dev)
    part_o = torch.empty(B, m.heads, splits, m.kv_rank, dtype=torch.float32,
                         device=dev)
    part_ml = torch.empty(B, m.heads, splits, 2, dtype=torch.float32,
                          device=dev)
    rc = _lib().fei_latent_decode(
        _p(out), out.stride(0), _p(proj), proj.stride(0), _p(w.uk), _p(w.uv),
        _p(w.norm), _p(rot), _p(rows), _p(batch.pos), _p(batch.table), _p(qa),
        _p(part_o), _p(part_ml), B, W, block_size.bit_length() - 1, m.heads,
        m.dim, m.rot_dim, m.vdim, m.kv_rank, m.scale, m.window or 0, w.eps,
        splits, tile, *beside, _f32(proj), _stream())
    if rc:
        raise ValueError(f"no decode tile for {m}")


def latent_attn_prefill(proj, out, m, w, rot, batch, rows,
                        block_size: int) -> None:
    """Prompt portions: rows n_dec .. of proj and out."""
    n = batch.n_dec
    if not proj.is_cuda:
        p_, o_ = proj[n:], out[n:]
        q = ref.latent_append(p_, m, w.norm, rot, w.eps, batch.pos[n:],
                              _dst(batch, n, None, block_size), rows)
        o = torch.empty(p_.shape[0], m.heads, m.vdim)
        for i, (row, cnt, pos0) in enumerate(batch.portions):
            k0 = 0 if m.window is None else max(0, pos0 - m.window + 1)
            at = slice(row - n, row - n + cnt)
            o[at] = ref.latent_attend(
                q[at], batch.pos[row:row + cnt],
                _keys(batch, n + i, k0, pos0 + cnt, rows, block_size), k0, m,
                w.uk, w.uv, m.scale)
        _latent_out(o, p_, m, o_)
        return
    lib, st = _lib(), _stream()
    W, bs_log = batch.table.shape[1], block_size.bit_length() - 1
    f32, T = _f32(proj), proj.shape[0] - n
    pr = proj[n:]
    lib.fei_latent_append(
        _p(pr), proj.stride(0), _p(rows), _p(w.norm), _p(rot),
        _p(batch.pos[n:]), _p(batch.row_seq[n:]), _p(batch.table), T, W,
        bs_log, m.heads, m.dim, m.rot_dim, m.vdim, m.kv_rank, w.eps, f32, st)
    spans, n_keys, tiles, owner, c, kr = _key_room(proj, m, batch)
    lib.fei_latent_gather(_p(c), _p(kr), _p(rows), _p(owner), _p(spans),
                          _p(batch.table), n_keys, W, bs_log, n, m.kv_rank,
                          m.rot_dim, f32, st)
    _window_prefill(proj, out, m, w, spans, tiles, c, kr)


def _key_room(proj, m, batch):
    """batch.key_plan, and room for the keys: latents and rotated parts."""
    spans, n_keys, tiles, owner = batch.key_plan(m.window)
    c, kr = (torch.empty(n_keys, k, dtype=proj.dtype, device=proj.device)
             for k in (m.kv_rank, m.rot_dim))
    return spans, n_keys, tiles, owner, c, kr


def _window_prefill(proj, out, m, w, spans, tiles, c, kr) -> None:
    kv = torch.nn.functional.linear(c, w.ukv)
    _lib().fei_window_prefill(
        _p(out), out.stride(0), _p(proj), proj.stride(0), _p(kv), _p(kr),
        _p(spans), _p(tiles), tiles.shape[0], m.heads, m.dim, m.rot_dim,
        m.vdim, m.kv_rank, m.scale, m.window or 0, _f32(proj), _stream())


def _keys_beside(m, tokens: int, rows: int, n_keys: int, size: int) -> bool:
    """Whether the launches of so many tokens prepare the portions' rows and keys, of
    values of ``size`` bytes. Their blocks gather 4 keys each, 8 where there are more
    than 16 heads, and few of them fit a CU beside the attention's LDS: by themselves
    keys take 5 us, here as many as the tokens leave time for. Both launches, beside
    and in launches of their own, us, rows of 1152 bytes: 16 heads, 2 tokens of 600 keys,
    8000 gathered 34, 42, 16000 46, 47; 4 of 1500, 8000 34, 42, 16000 51, 48, 64000 115,
    67; 8 of 600, 4000 37, 39, 6000 41, 41, 12000 50, 43; 64 of 300, 4000 74, 76, 8000 80,
    78. 32 heads, 4 of 1500, 16000 43 to 48, 48, 64000 84, 68; 8 of 600, 8000 45, 47, 16000
    51, 50. Rows of 320 to 2176 bytes part at as many bytes or more."""
    room = 14 if tokens <= 4 else 5
    return (0 < tokens < 1024 and rows < 1 << 16 and n_keys < 1 << 17   # of a grid
            and n_keys * m.row_width * size <= room << (21 if m.heads > 16 else 20))


def latent_attn_mixed(proj, out, m, w, rot, batch, rows, block_size: int) -> None:
    """latent_attn_decode of the first n_dec rows and latent_attn_prefill of the others,
    whose rows and keys the former's launches prepare where there are both and that
    pays."""
    n = batch.n_dec
    args = (m, w, rot, batch, rows, block_size)
    if (proj.is_cuda and n and batch.portions
            and _keys_beside(m, n, proj.shape[0], batch.key_plan(m.window)[1],
                             proj.element_size())):
        spans, n_keys, tiles, owner, c, kr = _key_room(proj, m, batch)
        _latent_decode(proj, out, *args, n, (
            proj.shape[0] - n, _p(batch.row_seq[n:]), n_keys, _p(c), _p(kr), _p(owner),
            _p(spans)))
        _window_prefill(proj, out, m, w, spans, tiles, c, kr)
        return
    if n:
        latent_attn_decode(proj[:n], out[:n], *args)
    if batch.portions:
        latent_attn_prefill(proj, out, *args)


# -- gated linear attention ----------------------------------------------------------

def check_gla_geometry(m) -> None:
    if m.dim > 256 or m.vdim > 512 or m.gate_rank > 128:
        raise ValueError(f"gated linear attention sizes out of range: {m}")


def _gla_split(proj, m, w):
    """q (scaled), k, v as [T, H, .] float32, gate columns, log decay."""
    T, a, b = proj.shape[0], m.heads * m.dim, m.heads * m.vdim
    q, k, v, g, a1 = proj.split([a, a, b, b, m.gate_rank], dim=-1)
    ld = ref.gla_log_decay(a1, w.a2, w.bias, m.tau)
    return (q.float().view(T, m.heads, m.dim) * m.dim ** -0.5,
            k.float().view(T, m.heads, m.dim),
            v.float().view(T, m.heads, m.vdim), g,
            ld.view(T, m.heads, m.dim))


def _gla_cpu(proj, out, m, w, state, fresh: bool) -> None:
    q, k, v, g, ld = _gla_split(proj, m, w)
    o, S = ref.gla_scan(q, k, v, ld, torch.zeros_like(state) if fresh
                        else state)
    state.copy_(S)
    out.copy_(ref.gla_gate_out(o, g, w.norm, w.eps).to(out.dtype))


def gla_decode(proj, out, m, w, batch, states) -> None:
    """One new token per sequence. proj [B, m.in_rows] (q | k | v | gate |
    low-rank decay input), out [B, H*vdim], states [slots+1, H, vdim, dim]."""
    if not proj.is_cuda:
        for b in range(batch.n_dec):
            _gla_cpu(proj[b:b + 1], out[b:b + 1], m, w,
                     states[int(batch.slots[b])], int(batch.pos[b]) == 0)
        return
    B = proj.shape[0]
    o = torch.empty(B, m.heads * m.vdim, dtype=torch.float32,
                    device=proj.device)
    _lib().fei_gla_decode(
        _p(out), out.stride(0), _p(o), _p(states), _p(proj), proj.stride(0),
        _p(w.a2), _p(w.bias), _p(w.norm), _p(batch.pos), _p(batch.slots), B,
        m.heads, m.dim, m.vdim, m.gate_rank, m.tau, w.eps, _f32(proj),
        _stream())


def gla_prefill(proj, out, m, w, batch, states) -> None:
    """Prompt portions: rows n_dec .. of proj and out."""
    if not proj.is_cuda:
        for i, (row, n, pos0) in enumerate(batch.portions):
            _gla_cpu(proj[row:row + n], out[row:row + n], m, w,
                     states[int(batch.slots[batch.n_dec + i])], pos0 == 0)
        return
    _gla_prefill(proj, out, m, w, batch, states, 0)


def gla_mixed(proj, out, m, w, batch, states) -> None:
    """gla_decode of the first n_dec rows and gla_prefill of the others, in the launches
    of the latter where there are both."""
    if proj.is_cuda and batch.n_dec and batch.portions:
        _gla_prefill(proj, out, m, w, batch, states, batch.n_dec)
        return
    if batch.n_dec:
        gla_decode(proj[:batch.n_dec], out[:batch.n_dec], m, w, batch, states)
    if batch.portions:
        gla_prefill(proj, out, m, w, batch, states)


def _gla_prefill(proj, out, m, w, batch, states, tokens: int) -> None:
    dev = proj.device
    chunks, spans = batch.chunk_plan()
    n = chunks.shape[0]
    f = dict(dtype=torch.float32, device=dev)
    G = torch.empty(proj.shape[0], m.heads * m.dim, **f)
    U = torch.empty(n, m.heads, m.vdim, m.dim, **f)
    A = torch.empty(n, m.heads, 64, 64, **f)
    o = torch.empty(tokens, m.heads * m.vdim, **f)
    _lib().fei_gla_prefill(
        _p(out), out.stride(0), _p(proj), proj.stride(0), _p(w.a2),
        _p(w.bias), _p(w.norm), _p(states), _p(chunks), n, _p(spans),
        spans.shape[0], _p(batch.slots), _p(G), _p(U), _p(A), tokens,
        _p(o), _p(batch.pos) if tokens else None, m.heads, m.dim, m.vdim,
        m.gate_rank, m.tau, w.eps, _f32(proj), _stream())
