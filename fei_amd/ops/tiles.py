"""Products of hundreds of rows and more (csrc/tile.hip) with what follows them
inside, or cut along K for the kernel after them. bfloat16 GPU tensors only."""

from __future__ import annotations

import ctypes
from functools import lru_cache
from typing import Optional, Tuple

import torch
from torch.utils._device import DeviceContext

import fei_amd.ops as _ops     # half made yet: it imports this

_vp, _i, _l = ctypes.c_void_p, ctypes.c_int, ctypes.c_long

# csrc/tile.hip
TILE_BF16, TILE_SWIGLU, TILE_GELU, TILE_RELU2, TILE_PARTS, TILE_BIAS = range(6)

CUS = 256
FAR = 1 << 24        # rows this far apart: what 128 of them span takes more than 32 bits
# Rows of x and w a tile, and us of a step of 64 of K: with one tile on the chip, and
# what comes on top with one on every CU, when the card lowers its clock. k_tile_counted of
# csrc/tile.hip has its own copy of those that it chooses from, which a test compares.
TILES = ((256, 256, 1.0, 0.46), (256, 192, 0.875, 0.36), (192, 256, 0.82, 0.34),
         (256, 128, 0.73, 0.13), (128, 256, 0.73, 0.13))


def declare(lib: ctypes.CDLL) -> None:
    lib.fei_tile.argtypes = [_vp, _l, _vp, _l, _vp, _vp] + [_i] * 7 + [_vp]
    lib.fei_tile_counted.argtypes = ([_vp, _l, _vp, _l, _vp, _vp] + [_i] * 5 +
                                     [_vp, _vp])


def _p(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def types_ok(*tensors: torch.Tensor) -> bool:
    """Whether the tensors are of no class that does more than torch's own."""
    return all(type(t) in (torch.Tensor, torch.nn.Parameter) for t in tensors)


def _memory(*tensors: torch.Tensor) -> bool:
    """Whether the tensors are what lies at their pointers, and nothing follows what
    is done to them: tracing, transforms, tangents, modes and casts to another type are
    for the library's operations."""
    c = torch._C                 # 2.5 us
    return (types_ok(*tensors)
            and c._functorch.peek_interpreter_stack() is None
            and torch.autograd.forward_ad._current_level < 0
            and not c._len_torch_dispatch_stack()
            # that of a default device changes nothing here
            and all(type(c._get_function_stack_at(i)) is DeviceContext
                    for i in range(c._len_torch_function_stack()))
            and (not torch.is_autocast_enabled("cuda")
                 or torch.get_autocast_dtype("cuda") is torch.bfloat16)
            and c._get_tracing_state() is None
            and not torch.compiler.is_compiling())


def _near(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether 16 bytes at a time and 32-bit offsets from a tile's first row reach
    the rows of both."""
    return (x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
            and x.stride(-1) == 1 and x.stride(-2) % 8 == 0
            and x.stride(-2) < FAR and w.shape[-1] < FAR)


def tile_ok(M: int, x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether M rows x times w run here; x's rows may lie apart."""
    K = w.shape[-1]
    return (M > 128 and w.is_cuda and w.dim() == 2 and K > 0 and K % 64 == 0
            and w.shape[0] > 0 and w.shape[0] % 8 == 0 and _memory(x, w)
            # a launch goes to the current device, the library's to the tensors'
            and w.get_device() == torch.cuda.current_device() and _near(x, w))


def _time(M: int, cols: int, K: int, parts: int, rows: int, width: int,
          alone: float, full: float) -> float:
    """About how many us a product takes: rounds of tiles over the CUs. A last round that
    runs in halves counts as a whole one; what it spares is 1 to 5 us of 35 to 360."""
    tiles = -(-M // rows) * -(-cols // width) * parts
    rounds = -(-tiles // CUS)
    return rounds * (-(-K // 64 // parts) * (alone + full * tiles /
                                             (CUS * rounds)) + 3.0)


@lru_cache(maxsize=1024)
def size_for(M: int, cols: int, K: int) -> Tuple[int, int]:
    """Rows of x and of w a tile for a product with ``cols`` of them.
    6006 x 3072, K = 2048, in tiles of 192 rows takes two rounds, three quarters full, 69
    us; in 256 x 256 two, a little over half full, 86; 16384 x 3072, K = 768, three rounds
    of 256, 70, four of 192, 89."""
    return min(TILES, key=lambda t: _time(M, cols, K, 1, *t))[:2]


@lru_cache(maxsize=1024)
def _rate(M: int, cols: int, K: int) -> float:
    """About how many PFLOP/s the tiles of a product reach: few where there are few, or
    where a last round has few."""
    return 2e-9 * M * cols * K / min(_time(M, cols, K, 1, *t) for t in TILES)


@lru_cache(maxsize=1024)
def _plain_pays(M: int, N: int, K: int) -> bool:
    """Whether a product with nothing behind it is faster in tiles than in the library,
    which whole rounds of 256 x 256 suit best, and three quarters of one of whole tiles:
    3 to 14 % faster there (8192 x 2048, 4096 rows 98 us, 103 here; 6144 x 1024, 2048
    rows 29, 31). Else from 0.88 PFLOP/s on (1.02 of more than a round where
    K < 2048: 6144 x 1536, 3000 rows 64 us, 60 in the library). Of 657 sizes, M of 300 to
    16384 and N of 768 to 16384, it takes 341, 222 of which gain 3 to 32 % (5000 x 1024,
    2600 rows 30 us for 43; 8192 x 2048, 2600 rows 76 for 97; 3072 x 2048, 6006 rows 76 for
    82), and at worst loses 6 (2560 x 1280, 6006 rows 37 for 35)."""
    tiles = -(-M // 256) * -(-N // 256)
    rounds = -(-tiles // CUS)
    if N % 256 == 0 and (tiles == rounds * CUS or
                         M % 256 == 0 and 4 * tiles >= 3 * rounds * CUS):
        return False
    return _rate(M, N, K) > (1.02 if K < 2048 and rounds > 1 else 0.88)


def linear_ok(M: int, x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether x [M, K] @ w^T is faster here than in the library: of K 1024 to 2048
    (of 4096 x 4096 and 6144 x 4096 neither is better by more than 5 % up to 6006
    rows)."""
    N, K = w.shape
    return (M > 256 and 1024 <= K <= 2048 and tile_ok(M, x, w)
            and _ops._mixers.match(x, w, x.shape[-1]) and _plain_pays(M, N, K))


def act_ok(M: int, x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether the product of all of w's rows with an activation inside is faster here
    than in the library with a pass for it. Over 43 sizes of 8 to 28672 results and K of
    64 to 14336, 129 to 8192 rows, nowhere by more than 6 % slower from 0.7 PFLOP/s on, and
    past K = 8192, which the library cuts, from 0.86. Without a rule, us: GELU of 256 x
    4096, 300 rows 56 (14), 1024 x 1024, 1000 rows 23 (15); SwiGLU of 2 x 1024 x 2048, 1000
    rows 29 (21); relu^2 of 6144 x 4096, 512 rows 55 (42). What the rule leaves out that
    would gain most: SwiGLU of 2 x 2048 x 512, 1301 rows 13 (22)."""
    N, K = w.shape
    return (tile_ok(M, x, w)
            and _rate(M, N, K) > (0.7 if K <= 8192 else 0.86))


def product(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor, N: int,
            epi: int, bias: Optional[torch.Tensor] = None) -> None:
    """x [M, K] with the rows of ``w``: N results a row, for tile_ok; rows of
    ``out`` on 16 bytes."""
    K = x.shape[1]
    size = size_for(x.shape[0], w.shape[0], K)
    _launch(out, x, w, N, epi, size, bias)


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x [M, K] @ w^T, for linear_ok."""
    out = torch.empty(x.shape[0], w.shape[0], dtype=x.dtype, device=x.device)
    product(x, w, out, w.shape[0], TILE_BF16)
    return out


def _launch(out, x, w, N, epi, size, bias=None, parts=1) -> None:
    M, K = x.shape
    _ops.require_lib().fei_tile(
        _p(out), out.stride(-2), _p(x), x.stride(0), _p(w), _p(bias), M, N, K,
        epi, *size, parts, _ops._stream())


def parts_ok(M: int, x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether x @ w^T may run in parts of K that the norm after it sums: a long
    K, and results for less than half of the CUs' tiles, so that it is faster if there
    are not too few (parts_pay). With the norm, against the
    library's product and a norm: 4096 x 14336 of 512 rows 66 us (95), 1000 106
    (138), 2048 187 (212); 2048 x 8192 of 512 32 (35), 2048 72 (79), 4000 117 (121);
    of 6006 172 (166). 4096 x 4096 is a draw."""
    N, K = w.shape
    return (K >= 8192 and M > 256 and tile_ok(M, x, w)
            and _ops._mixers.match(x, w, x.shape[-1])
            and 2 * -(-M // 256) * -(-N // 256) <= CUS)


def parts_pay(M: int, w: torch.Tensor) -> bool:
    """Whether products with w that parts_ok takes have the tiles for it: of few results
    a row eight parts leave most CUs without, and the library cuts K further; and of
    just half of the CUs' tiles, up to K = 10240, it is as good. With float32 results
    added, K = 8192, 257 rows, us: 8 results 19 (12), 256 23 (16), 512 25 (23), 768 26
    (23), 1000 26 (29), 1024 25 (27); 1024 of 8192 rows 126 (115)."""
    N, K = w.shape
    return N >= 1000 and (K >= 10240
                          or 2 * -(-M // 256) * -(-N // 256) < CUS)


def add_ok(x: torch.Tensor, a: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether x += a @ w^T, x [M, N] float32 without gaps, is faster in parts of K
    and a pass that adds them. Against the library's product with float32 results,
    us: 2048 x 10240 of 300 rows 31 (48), 1301 62 (78), 1900 80 (95), 4096 141
    (150); 2048 x 14336 of 1706 97 (124); 4096 x 10240 of 1900 143 (147); 4096 x
    25600 of 1030 207 (319). 2048 x 4096 of 1301 40 (32): there the pass costs more
    than the parts gain."""
    return (parts_ok(a.shape[0], a, w) and types_ok(x)
            and x.data_ptr() % 16 == 0
            and not (x.requires_grad and torch.is_grad_enabled()))


@lru_cache(maxsize=1024)
def parts_for(M: int, N: int, K: int) -> Tuple[Tuple[int, int], int]:
    """Rows of x and of w a tile, and parts of K. A part's sums are written and
    read once, 8 bytes at about 4.5 TB/s."""
    tile, p = min(((t, p) for t in TILES for p in range(1, 9)),
                  key=lambda c: _time(M, N, K, c[1], *c[0]) +
                  c[1] * M * N * 1.8e-6)
    return tile[:2], p


@lru_cache(maxsize=1024)
def parts_up_to(M: int, N: int, K: int) -> int:
    """Parts of K where only the device knows how many of M rows there are, half of them
    or more, which chooses its tiles, and something reads the results of a product in one
    part too."""
    def us(m, p):
        return (min(_time(m, N, K, p, *t) for t in TILES if t[1] > 128) +
                m * N * (1.8e-6 * p if p > 1 else 0.9e-6))
    most = max(1, min(8, K // 256))
    times = [[us(M * f // 8, p) for p in range(1, most + 1)] for f in range(4, 9)]
    loss = [sum(row[i] / min(row) for row in times) for i in range(len(times[0]))]
    return loss.index(min(loss)) + 1


def product_parts(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x [M, K] @ w^T as float32 parts [p, M, N] that are to be summed, for
    parts_ok."""
    M, K = x.shape
    N = w.shape[0]
    size, p = parts_for(M, N, K)
    out = torch.empty(p, M, N, dtype=torch.float32, device=x.device)
    _launch(out, x, w, N, TILE_PARTS, size, None, p)
    return out
