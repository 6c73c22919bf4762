"""Products of tens of rows (csrc/rows.hip): cut along K into parts that the
kernel after them sums, or with the SwiGLU inside. bfloat16 GPU tensors only."""

from __future__ import annotations

import ctypes
from typing import Optional, Tuple

import torch

import fei_amd.ops as _ops     # half made yet: it imports this

_vp, _i, _f, _l = (ctypes.c_void_p, ctypes.c_int, ctypes.c_float,
                   ctypes.c_long)

SKINNY_ROWS = 32     # most rows of the matrix-core tile for few rows


def declare(lib: ctypes.CDLL) -> None:
    lib.fei_rows.argtypes = [_vp, _vp, _l, _vp] + [_i] * 7 + [_vp]
    lib.fei_rows_bias.argtypes = [_vp] * 4 + [_i] * 4 + [_vp]
    lib.fei_parts_layernorm.argtypes = ([_vp, _vp, _i] + [_vp] * 4 +
                                        [_i, _i, _f, _vp])
    lib.fei_parts_norm.argtypes = [_vp, _vp, _vp, _i, _vp, _i, _i, _f, _vp]
    lib.fei_rope_kv_parts.argtypes = [_vp, _vp, _i] + [_vp] * 4 + [_i] * 6 + [_vp]
    lib.fei_parts_add.argtypes = [_vp, _vp, _i, _l, _f, _vp]
    lib.fei_parts_add_norms.argtypes = (
        [_vp] * 4 + [_i] + [_vp] * 2 + [_i, _i, _f, _f, _vp])


def _lib() -> ctypes.CDLL:
    return _ops.require_lib()


def _stream() -> int:
    return _ops._stream()


def _p(t: torch.Tensor) -> int:
    return t.data_ptr()


def rows_ok(M: int, w: torch.Tensor) -> bool:
    """Whether tens of rows of w's type times w may run in parts
    (product_parts). At 256 rows the parts are still the faster way (2048 to
    6144 results of 2048 to 14336: 1.04 to 1.5 times a library product), and
    beyond that the library fills the chip by itself."""
    return (SKINNY_ROWS < M <= 256 and w.is_cuda and w.dim() == 2
            and w.dtype == torch.bfloat16 and w.is_contiguous()
            and w.shape[1] > 0 and w.shape[1] % 64 == 0
            and w.shape[0] > 0 and w.shape[0] % 8 == 0
            and w.data_ptr() % 16 == 0)


def _tile(M: int) -> Tuple[int, int]:
    """Tiles of rows, and 32 rows in each: 2 to 4."""
    nm = -(-M // 128)
    return nm, max(2, -(-M // (32 * nm)))


def _launch(out, x, w, N, swiglu, xj, wide, parts) -> None:
    _lib().fei_rows(_p(out), _p(x), x.stride(0), _p(w), x.shape[0], N,
                    w.shape[1], swiglu, xj, wide, parts, _stream())


def product_parts(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x [M, K] @ w^T as float32 parts [p, M, N] that are to be summed, for
    rows_ok.

    K is cut so that there is about a tile a CU, into parts of 1024 steps at
    least (512 of a short K): 75 rows, 4096 x 14336 in 8 parts 27 us, in 4 36,
    the library 50; 4096 x 4096 in 4 11.4, in 8 11.7, 16.2. Tiles of 128 rows of
    w repeat x least, of 64 make more of them where 128 leave CUs without."""
    M, K = x.shape
    N = w.shape[0]
    if x.stride(1) != 1 or x.stride(0) % 8 or x.data_ptr() % 16:
        x = x.clone(memory_format=torch.contiguous_format)
    nm, xj = _tile(M)
    most = max(1, min(8, K // (1024 if K >= 4096 else 512)))

    def cut(tiles):
        p = max(1, min(most, 256 // tiles))
        return p, p * tiles
    p, blocks = cut(nm * -(-N // 128))
    wide = blocks >= 192
    if not wide:
        p, _ = cut(nm * -(-N // 64))
    out = torch.empty(p, M, N, dtype=torch.float32, device=x.device)
    _launch(out, x, w, N, 0, xj, int(wide), p)
    return out


def add_norm_parts(parts: torch.Tensor, residual: torch.Tensor,
                   weight: torch.Tensor, eps: float) -> torch.Tensor:
    """residual += the sum of the parts (in place); rmsnorm(residual)."""
    p, M, N = parts.shape
    out = torch.empty_like(residual)
    _lib().fei_parts_norm(_p(out), _p(residual), _p(parts), p, _p(weight), M,
                          N, eps, _stream())
    return out


def rope_kv_parts(parts, S: int, Hq: int, k_cache, v_cache, pos0,
                  table) -> torch.Tensor:
    """The projections of q, k and v in parts [p, B * S, (Hq + 2 Hkv) D] ->
    roped q [B, S, Hq, D]; roped k and v go to the caches at pos0[b] + s."""
    p, T, _ = parts.shape
    Hkv, D = k_cache.shape[1], k_cache.shape[3]
    q = torch.empty(T // S, S, Hq, D, dtype=k_cache.dtype,
                    device=parts.device)
    _lib().fei_rope_kv_parts(
        _p(q), _p(parts), p, _p(k_cache), _p(v_cache), _p(table),
        _p(pos0), T // S, S, Hq, Hkv, D, k_cache.shape[2], _stream())
    return q


def swiglu_ok(M: int, x: torch.Tensor, wgu: torch.Tensor) -> bool:
    """Whether tens of rows take the SwiGLU product whole: one tile of rows, or
    two where all tiles are on the chip at once. Against the library and a
    SwiGLU pass, 2 x 14336 x 4096: 75 rows 48 us, 57.6; 128: 53, 58; 192: 77, 71.
    2 x 8192 x 2048: 75 rows 21, 24; 256: 27, 34."""
    return (rows_ok(M, wgu) and wgu.shape[0] % 16 == 0
            and x.dtype == wgu.dtype and
            (M <= 128 or _tile(M)[0] * -(-wgu.shape[0] // 128) <= 256))


def swiglu_product(x: torch.Tensor, wgu: torch.Tensor,
                   out: torch.Tensor) -> None:
    """silu(g) * u of the gates and ups x @ wgu^T, for swiglu_ok."""
    if x.data_ptr() % 16:
        x = x.clone()
    nm, xj = _tile(x.shape[0])
    # 64 rows of w a tile where 128 leave CUs without one
    wide = nm * -(-wgu.shape[0] // 128) >= 192
    _launch(out, x, wgu, wgu.shape[0] // 2, 1, xj, int(wide), 1)


def add_ok(x: torch.Tensor, a: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether x += a @ w^T runs in parts: of a short K the second launch costs
    what they gain (200 rows, 2048 x 2048: 11 us in the library)."""
    return (rows_ok(a.shape[0], w) and w.shape[1] >= 4096
            and a.dtype == w.dtype and a.shape[1] == w.shape[1]
            and a.device == w.device == x.device and x.dtype == torch.float32
            and x.shape == (a.shape[0], w.shape[0])
            and x.is_contiguous() and x.data_ptr() % 16 == 0)


def add_product(x: torch.Tensor, a: torch.Tensor, w: torch.Tensor,
                mult: float) -> None:
    """x += mult * (a @ w^T), for add_ok."""
    add_parts(x, product_parts(a, w), mult)


def add_parts(x: torch.Tensor, parts: torch.Tensor, mult: float) -> None:
    """x += mult * the sum of the parts, float32 on 16 bytes, a multiple of 4
    values."""
    _lib().fei_parts_add(_p(x), _p(parts), parts.shape[0], x.numel(), mult,
                         _stream())


def add_parts_norms(x: torch.Tensor, parts: torch.Tensor, mult: float,
                    w1: torch.Tensor, w2: Optional[torch.Tensor], eps: float
                    ) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """add_parts to x [M, C], and its norms with the float32 gains in bfloat16."""
    M, C = x.shape
    o1 = torch.empty(M, C, dtype=torch.bfloat16, device=x.device)
    o2 = None if w2 is None else torch.empty_like(o1)
    _lib().fei_parts_add_norms(
        _p(o1), None if o2 is None else _p(o2), _p(x), _p(parts),
        parts.shape[0], _p(w1), None if w2 is None else _p(w2), M, C, mult,
        eps, _stream())
    return o1, o2
