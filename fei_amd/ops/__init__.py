"""fei_amd.ops — engine ops with a single dispatch rule:

  - CUDA (= ROCm/HIP) tensors -> the in-tree gfx950 kernel library,
    loaded via ctypes. If the library is missing on a GPU machine, ops
    FAIL LOUDLY — there is no silent eager fallback on GPU.
  - CPU tensors -> the fp32-accurate torch reference implementations
    (fei_amd/ops/reference.py), used by CPU tests and tiny models.

All kernels launch on torch's current CUDA stream, so the decode step can
be captured into a hipGraph (torch.cuda.CUDAGraph) — see engine/engine.py.
"""

from __future__ import annotations

import ctypes
import math
import os
from typing import Optional, Tuple

import torch

from fei_amd.ops import layers as _layers
from fei_amd.ops import mixers as _mixers
from fei_amd.ops import moe as _moe
from fei_amd.ops import reference as ref
from fei_amd.ops import rows as _rows
from fei_amd.ops import sigmoid_attn as _sigmoid_attn
from fei_amd.ops import tiles as _tiles
from fei_amd.ops.layers import (  # noqa: F401
    encoder_one, llama_few, llama_one, llama_one_pays)
from fei_amd.ops.mixers import (  # noqa: F401
    GainNorm, GainNormed, cat_cast, check_gla_geometry,
    check_latent_geometry, embed_pos, gain_logits, gla_decode, gla_mixed, gla_prefill,
    latent_attn_decode, latent_attn_mixed, latent_attn_prefill, linear_f32,
    logits_head, mix_in, norm_pair, parallel_in, residual_linear, residual_norms)
from fei_amd.ops.moe import (  # noqa: F401
    check_moe_geometry, residual_moe, route)
from fei_amd.ops.rows import (  # noqa: F401
    add_norm_parts, product_parts, rope_kv_parts, rows_ok)
from fei_amd.ops.sigmoid_attn import (  # noqa: F401
    check_sigmoid_geometry, sigmoid_attn_decode, sigmoid_attn_mixed,
    sigmoid_attn_prefill)
from fei_amd.ops.tiles import (  # noqa: F401
    parts_ok as tile_parts_ok, parts_pay as tile_parts_pay,
    product_parts as tile_parts)

_LIB: Optional[ctypes.CDLL] = None
_LIB_ERR: Optional[str] = None
_LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)),
                         "libfei_kernels.so")

_c = ctypes
_vp, _i, _f, _u64, _l = _c.c_void_p, _c.c_int, _c.c_float, _c.c_ulonglong, _c.c_long


def _try_load() -> None:
    global _LIB, _LIB_ERR
    if _LIB is not None or _LIB_ERR is not None:
        return
    try:
        lib = ctypes.CDLL(_LIB_PATH)
    except OSError as e:
        _LIB_ERR = str(e)
        return
    lib.fei_rmsnorm.argtypes = [_vp, _vp, _vp, _i, _i, _f, _vp]
    lib.fei_add_rmsnorm.argtypes = [_vp, _vp, _vp, _vp, _i, _i, _f, _vp]
    lib.fei_rope_kv_decode.argtypes = [_vp, _vp, _vp, _vp, _vp, _vp, _vp,
                                       _i, _i, _i, _i, _i, _l, _l, _vp]
    lib.fei_rope_kv_prefill.argtypes = [_vp, _vp, _vp, _vp, _vp, _vp, _vp,
                                        _i, _i, _i, _i, _i, _i, _l, _l, _vp]
    lib.fei_attn_decode.argtypes = ([_vp] * 8 + [_i] * 8 + [_f, _l] +
                                    [_vp] * 3 + [_l, _vp])
    lib.fei_attn_decode_product.argtypes = ([_vp] * 8 + [_i] * 7 + [_f, _l] +
                                            [_vp] * 3 + [_l] + [_vp] * 3 +
                                            [_i, _vp])
    lib.fei_swiglu.argtypes = [_vp, _vp, _l, _i, _vp]
    lib.fei_sample.argtypes = [_vp, _vp, _vp, _vp, _vp, _i, _i, _i, _f, _u64,
                               _i, _i, _vp]
    lib.fei_advance.argtypes = [_vp, _vp, _i, _i, _vp]
    lib.fei_attn_prefill.argtypes = [_vp, _vp, _vp, _vp, _vp, _vp,
                                     _i, _i, _i, _i, _i, _i, _f, _i, _l, _i,
                                     _vp, _vp, _l, _l, _l, _vp]
    lib.fei_mfma_probe.argtypes = [_vp, _vp, _vp, _vp]
    lib.fei_gemv.argtypes = [_vp, _vp, _vp, _vp, _vp, _i, _i, _i, _f, _i,
                             _vp, _vp]
    lib.fei_skinny.argtypes = ([_vp] * 3 + [_i] * 4 + [_vp, _f, _f, _i, _i] +
                               [_vp, _vp, _l] + [_vp] * 3 + [_i, _f, _vp, _vp])
    lib.fei_pool_unit.argtypes = [_vp] * 3 + [_i] * 3 + [_vp]
    lib.fei_argmax.argtypes = [_vp] * 3 + [_i] * 4 + [_vp]
    lib.fei_encoder_layers.argtypes = ([_vp, _i] + [_vp] * 8 + [_i] * 6 +
                                       [_f, _f, _i] + [_vp] * 3 + [_i, _i, _vp])
    lib.fei_embed_layernorm.argtypes = ([_vp] * 6 + [_i] * 4 + [_f] + [_vp] * 2)
    lib.fei_encoder_packed.argtypes = ([_vp, _i] + [_vp] * 4 + [_i] +
                                       [_vp] * 10 + [_i] * 6 +
                                       [_f, _f, _i, _vp, _i, _i, _vp])
    lib.fei_attn_decode_fused.argtypes = [_vp, _vp, _vp, _vp, _vp, _vp, _vp,
                                          _vp, _i, _i, _i, _i, _i, _f,
                                          _l, _l, _vp]
    lib.fei_sample_onepass.argtypes = [_vp, _vp, _vp, _vp, _i, _i, _f, _u64,
                                       _i, _i, _vp]
    lib.fei_sample_shard.argtypes = [_vp, _vp, _vp, _i, _i, _i, _f, _u64, _vp]
    lib.fei_stream_layer_check.argtypes = [_i, _i, _i, _i, _i]
    lib.fei_stream_layer_check.restype = _i
    lib.fei_stream_layer.argtypes = [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp,
                                     _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp,
                                     _vp, _vp, _vp, _i, _i, _i, _i, _i,
                                     _i, _i, _f, _f, _vp]
    lib.fei_add_layernorm.argtypes = [_vp, _vp, _vp, _vp, _vp, _i, _i, _f,
                                      _i, _vp]
    lib.fei_gelu.argtypes = [_vp, _vp, _l, _vp]
    lib.fei_quant_fp8_rows.argtypes = [_vp, _vp, _vp, _i, _i, _vp]
    lib.fei_prefetch.argtypes = [_vp, _l, _vp, _i, _vp]
    _mixers.declare(lib)
    _rows.declare(lib)
    _tiles.declare(lib)
    _layers.declare(lib)
    _moe.declare(lib)
    _sigmoid_attn.declare(lib)
    _LIB = lib


def kernels_available() -> bool:
    _try_load()
    return _LIB is not None


def require_lib() -> ctypes.CDLL:
    _try_load()
    if _LIB is None:
        raise RuntimeError(
            "fei_amd HIP kernel library not found at "
            f"{_LIB_PATH} ({_LIB_ERR}). Build it with "
            "`python -m fei_amd.ops.build` — GPU execution refuses to fall "
            "back to eager PyTorch.")
    return _LIB


def build_if_missing() -> None:
    """Compile the kernel library if this checkout has none (or an older
    one); needs hipcc, takes about a minute."""
    global _LIB_ERR
    from fei_amd.ops import build as _build
    if _build.needs_build():
        _build.build(verbose=False)
        _LIB_ERR = None


def _stream() -> int:
    # the raw handle: a Stream object per launch costs more than the launch
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device())


def _ptr(t: torch.Tensor) -> int:
    return t.data_ptr()


# ---------------------------------------------------------------------------


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float = 1e-5,
            out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """RMSNorm over the last dim. x: [..., C] bf16 (GPU) / any float (CPU)."""
    if not x.is_cuda:
        return ref.rmsnorm(x, weight, eps)
    lib = require_lib()
    x2 = x.contiguous()
    if out is None:
        out = torch.empty_like(x2)
    rows = x2.numel() // x2.shape[-1]
    lib.fei_rmsnorm(_ptr(out), _ptr(x2), _ptr(weight), rows, x2.shape[-1],
                    eps, _stream())
    return out


def fused_add_rmsnorm(x: torch.Tensor, residual: torch.Tensor,
                      weight: torch.Tensor, eps: float = 1e-5,
                      out: Optional[torch.Tensor] = None
                      ) -> Tuple[torch.Tensor, torch.Tensor]:
    """residual += x (in place on GPU); out = rmsnorm(residual)."""
    if not x.is_cuda:
        o, res = ref.fused_add_rmsnorm(x, residual, weight, eps)
        residual.copy_(res)
        return o, residual
    lib = require_lib()
    x2 = x.contiguous()
    if out is None:
        out = torch.empty_like(x2)
    rows = x2.numel() // x2.shape[-1]
    lib.fei_add_rmsnorm(_ptr(out), _ptr(residual), _ptr(x2), _ptr(weight),
                        rows, x2.shape[-1], eps, _stream())
    return out, residual


def rope_kv_decode(q, k, v, k_cache, v_cache, pos, table) -> torch.Tensor:
    """In-place RoPE on q; k roped + v appended into caches at pos[b].
    q [B,Hq,D], k/v [B,Hkv,D], caches [B,Hkv,max_seq,D], pos [B] int32."""
    if not q.is_cuda:
        q_out = ref.rope_kv_decode(q, k, v, k_cache, v_cache, pos, table)
        q.copy_(q_out)
        return q
    lib = require_lib()
    B, Hq, D = q.shape
    Hkv = k.shape[1]
    assert q.stride(2) == 1 and q.stride(1) == D, "head rows must be contiguous"
    assert k.stride(1) == D and v.stride(1) == D
    assert k.stride(0) == v.stride(0)
    lib.fei_rope_kv_decode(_ptr(q), _ptr(k), _ptr(v), _ptr(k_cache),
                           _ptr(v_cache), _ptr(table), _ptr(pos),
                           B, Hq, Hkv, D, k_cache.shape[2],
                           q.stride(0), k.stride(0), _stream())
    return q


def rope_kv_prefill(q, k, v, k_cache, v_cache, pos0, table) -> torch.Tensor:
    """In-place RoPE on q [B,S,Hq,D]; k roped + v appended at pos0[b]+s."""
    if not q.is_cuda:
        q_out = ref.rope_kv_prefill(q, k, v, k_cache, v_cache, pos0, table)
        q.copy_(q_out)
        return q
    lib = require_lib()
    B, S, Hq, D = q.shape
    Hkv = k.shape[2]
    assert q.stride(3) == 1 and q.stride(2) == D
    assert q.stride(0) == S * q.stride(1), "token rows must be uniform"
    assert k.stride(2) == D and k.stride(0) == S * k.stride(1)
    assert k.stride(1) == v.stride(1)
    lib.fei_rope_kv_prefill(_ptr(q), _ptr(k), _ptr(v), _ptr(k_cache),
                            _ptr(v_cache), _ptr(table), _ptr(pos0),
                            B, S, Hq, Hkv, D, k_cache.shape[2],
                            q.stride(1), k.stride(1), _stream())
    return q


def attn_decode(q, k_cache, v_cache, pos, splits: int = 32,
                scale: Optional[float] = None,
                workspace: Optional[Tuple[torch.Tensor, torch.Tensor]] = None,
                out: Optional[torch.Tensor] = None,
                k: Optional[torch.Tensor] = None,
                v: Optional[torch.Tensor] = None,
                table: Optional[torch.Tensor] = None,
                layer: int = 0) -> torch.Tensor:
    """Single-token GQA attention over n = pos[b]+1 cache entries.
    q [B,Hq,D] -> out [B,Hq,D]. The length is read on DEVICE (hipGraph).
    When (k, v, table) are given, the kernel also fuses the step's RoPE +
    KV-append: q is the RAW qkv view and cache[pos] is written in-kernel.
    ``workspace``: float32 [B,Hq,splits,D] and [B,Hq,splits,2]; more entries,
    and ``layer``, are taken and not used."""
    B, Hq, D = q.shape
    scale = scale if scale is not None else 1.0 / math.sqrt(D)
    if not q.is_cuda:
        if table is not None:
            rope_kv_decode(q, k, v, k_cache, v_cache, pos, table)
        seqlen = pos + 1
        return ref.attn_decode(q, k_cache, v_cache, seqlen, scale)
    return _launch_attn_decode(q, k_cache, v_cache, None, k_cache.shape[2], 0,
                               k_cache.shape[1], pos, splits, scale,
                               workspace, out, k, v, table)


def _launch_attn_decode(q, kc, vc, blocks, max_seq: int, bs_log: int,
                        Hkv: int, pos, splits: int, scale: float, workspace,
                        out, k, v, rope, product=None) -> torch.Tensor:
    """Contiguous caches (``blocks`` None) or paged pools. ``product``: (w, its scales or
    None, res) of an output product that is added to res, of one sequence."""
    B, Hq, D = q.shape
    if workspace is None:
        part_o = torch.empty(B, Hq, splits, D, dtype=torch.float32, device=q.device)
        part_ml = torch.empty(B, Hq, splits, 2, dtype=torch.float32, device=q.device)
    else:
        part_o, part_ml = workspace[0], workspace[1]
        assert part_o.shape[2] == splits and part_ml.shape[2] == splits, \
            f"workspace sized for {part_o.shape[2]} splits, kernel asked {splits}"
    if out is None:
        out = torch.empty(B, Hq, D, dtype=q.dtype, device=q.device)
    assert q.stride(2) == 1 and q.stride(1) == D
    # a lane's share of a row: D/16 columns
    assert D in (64, 128), f"decode attention supports D in (64,128), got {D}"
    assert splits <= 64, "the combine kernel takes at most 64 splits"
    assert Hq // Hkv <= 16, "at most 16 query heads per kv head"
    if rope is not None:
        assert k is not None and v is not None
        assert k.stride(1) == D and k.stride(0) == v.stride(0)
        kin, vin, cs, kv_bs = _ptr(k), _ptr(v), _ptr(rope), k.stride(0)
    else:
        kin = vin = cs = None
        kv_bs = 0
    if not B:
        return out
    args = (_ptr(q), _ptr(kc), _ptr(vc), None if blocks is None else _ptr(blocks),
            _ptr(part_o), _ptr(part_ml), _ptr(out), _ptr(pos))
    sizes = (Hq, Hkv, D, max_seq, bs_log, 0 if blocks is None else blocks.shape[1],
             splits, scale, q.stride(0), kin, vin, cs, kv_bs)
    if product is None:
        require_lib().fei_attn_decode(*args, B, *sizes, _stream())
    else:
        w, wscale, res = product
        require_lib().fei_attn_decode_product(
            *args, *sizes, _ptr(res), _ptr(w),
            None if wscale is None else _ptr(wscale), w.shape[0], _stream())
    return out


def attn_decode_fused(q, k, v, k_cache, v_cache, pos, table,
                      scale: Optional[float] = None,
                      out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Fused decode attention: RoPE(q,k) + KV-append + GQA attention in one
    kernel (grid Hkv x B, no split partials). For agent-length sequences;
    long-context uses rope_kv_decode + attn_decode (split-K)."""
    B, Hq, D = q.shape
    Hkv = k.shape[1]
    scale = scale if scale is not None else 1.0 / math.sqrt(D)
    if not q.is_cuda:
        rope_kv_decode(q, k, v, k_cache, v_cache, pos, table)
        return ref.attn_decode(q, k_cache, v_cache, pos + 1, scale)
    lib = require_lib()
    assert q.stride(2) == 1 and q.stride(1) == D
    assert k.stride(1) == D and k.stride(0) == v.stride(0)
    if out is None:
        out = torch.empty(B, Hq, D, dtype=torch.bfloat16, device=q.device)
    lib.fei_attn_decode_fused(_ptr(q), _ptr(k), _ptr(v), _ptr(k_cache),
                              _ptr(v_cache), _ptr(out), _ptr(table), _ptr(pos),
                              B, Hq, Hkv, D, k_cache.shape[2], scale,
                              q.stride(0), k.stride(0), _stream())
    return out


def attn_prefill(q, k_cache, v_cache, pos0, scale: Optional[float] = None,
                 causal: bool = True, kv_len: Optional[torch.Tensor] = None,
                 out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Causal (or bidirectional) GQA attention of q [B,S,Hq,D] over the
    caches. q token s attends [0, pos0[b]+s] when causal, else [0, kv_len[b])."""
    B, S, Hq, D = q.shape
    scale = scale if scale is not None else 1.0 / math.sqrt(D)
    if not q.is_cuda:
        if causal:
            return ref.attn_prefill(q, k_cache, v_cache, pos0, scale)
        # bidirectional reference: softmax over [0, kv_len)
        return _ref_bidir(q, k_cache, v_cache, kv_len, scale)
    lib = require_lib()
    if out is None:
        out = torch.empty_like(q)
    if kv_len is None:
        kv_len = pos0  # unused when causal
    Hkv = k_cache.shape[1]
    assert q.stride(3) == 1 and q.stride(2) == D
    assert q.stride(0) == S * q.stride(1)
    assert out.is_contiguous()
    if not q.numel():
        return out
    k_cache, v_cache = _cache_rows(k_cache, v_cache)
    splits = _prefill_splits(B, Hkv, S * (Hq // Hkv), k_cache.shape[2], D)
    po = pml = None
    if splits > 1:
        ws = torch.empty(B * S * Hq * splits * (D + 2), dtype=torch.float32,
                         device=q.device)
        po, pml = _ptr(ws), _ptr(ws) + B * S * Hq * splits * D * 4
    lib.fei_attn_prefill(_ptr(q), _ptr(k_cache), _ptr(v_cache), _ptr(out),
                         _ptr(pos0), _ptr(kv_len), B, S, Hq, Hkv, D,
                         k_cache.shape[2], scale, 1 if causal else 0,
                         q.stride(1), splits, po, pml, k_cache.stride(0),
                         k_cache.stride(1), k_cache.stride(2), _stream())
    return out


def _cache_rows(k: torch.Tensor, v: torch.Tensor):
    """Caches as the prompt attention's loads of 16 bytes take them: contiguous
    rows, all 16-byte aligned, both laid out alike; copies where they are not
    (what it reads is not written to)."""
    def fits(t):
        return (t.stride(3) == 1 and t.data_ptr() % 16 == 0
                and all(s % 8 == 0 for s in t.stride()[:3]))
    if k.stride() == v.stride() and fits(k) and fits(v):
        return k, v
    return (t.clone(memory_format=torch.contiguous_format) for t in (k, v))


def _prefill_splits(B: int, Hkv: int, rows: int, max_seq: int,
                    dim: int = 64) -> int:
    """Shares of the keys that the prompt attention's blocks of 128 rows are
    cut into, so that few rows over many keys fill the chip's 512 places (two
    blocks per CU), or of heads of 128 a CU each, if that leaves them three shares and
    more. One block too many is a round more, and each share's sums are written and read
    once. 32 layers of 4096 in all, us, by 512 places and one block too many / 512 / 256:
    65 tokens over 2500 keys 4262 / 4262 / 4200, over 7500 4550 / 4550 / 4478; 75 4348 /
    4348 / 4282, 4623 / 4623 / 4539; 96 4540 / 4540 / 4410, 4832 / 4832 / 4703; 128 5090 /
    5090 / 4925, 5463 / 5463 / 5308; 192 6400 / 6192 / 6037, 6990 / 6708 / 6587; 320 8033 /
    7743 / 7711, 8979 / 8512 / 8678; four prompts of 40 over 3000 6303 / 6303 / 5975. Heads
    of 64 gain up to 2 % from whole rounds, and lose with 256 places: 16 layers of 2048, 600
    over 4000, 2730 / 2711 / 2987.

    How many keys there are is known on the device only; the kernel uses fewer
    shares where one would have under three tiles of 64, and one where there are
    few keys in all. Of ``max_seq`` that is asked here, for half of the ``B`` and
    one more as if they were long; a launch without shares saves 3 us and more."""
    blocks = B * Hkv * -(-rows // 128)
    if blocks > 192 or max_seq <= 64 * 6 + Hkv * rows * (B + 1) // 20:
        return 1
    places = 256 if dim > 64 and 3 * blocks <= 256 else 512
    return max(1, min(16, places // blocks, max_seq // 192))


def _ref_bidir(q, k_cache, v_cache, kv_len, scale):
    B, S, Hq, D = q.shape
    Hkv = k_cache.shape[1]
    G = Hq // Hkv
    out = torch.empty_like(q)
    for b in range(B):
        n = int(kv_len[b])
        k = k_cache[b, :, :n, :].float()
        v = v_cache[b, :, :n, :].float()
        qb = q[b].float().view(S, Hkv, G, D)
        s = torch.einsum("shgd,hnd->hgsn", qb, k) * scale
        p = torch.softmax(s, dim=-1)
        o = torch.einsum("hgsn,hnd->shgd", p, v)
        out[b] = o.reshape(S, Hq, D).to(q.dtype)
    return out


def swiglu(gate_up: torch.Tensor,
           out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """gate_up [..., 2*inter] -> [..., inter]: silu(gate) * up."""
    if not gate_up.is_cuda:
        return ref.swiglu(gate_up)
    lib = require_lib()
    gu = gate_up.contiguous()
    inter = gu.shape[-1] // 2
    rows = gu.numel() // gu.shape[-1]
    if out is None:
        out = torch.empty(*gu.shape[:-1], inter, dtype=gu.dtype, device=gu.device)
    lib.fei_swiglu(_ptr(out), _ptr(gu), rows, inter, _stream())
    return out


def argmax(x: torch.Tensor) -> torch.Tensor:
    """x.argmax(-1) of rows [B, V]: the first of the largest values."""
    if not (x.is_cuda and x.dim() == 2 and x.is_contiguous() and x.numel()
            and x.shape[0] <= 65535 and x.shape[1] < 1 << 30
            and x.dtype in (torch.bfloat16, torch.float32)):
        return x.argmax(dim=-1)
    B, V = x.shape               # rows are the second dimension of a grid
    chunks = max(1, min(64, 512 // B, -(-V // 2048)))
    out = torch.empty(B, dtype=torch.int64, device=x.device)
    part = torch.empty(B, chunks, dtype=torch.int64, device=x.device)
    require_lib().fei_argmax(_ptr(out), _ptr(part), _ptr(x), B, V, chunks,
                             1 if x.dtype == torch.float32 else 0, _stream())
    return out


def sample(logits: torch.Tensor, token: torch.Tensor,
           step: torch.Tensor, workspace: torch.Tensor,
           out_tokens: Optional[torch.Tensor] = None,
           temperature: float = 0.0, seed: int = 0,
           nchunks: int = 64) -> torch.Tensor:
    """Greedy (T<=0) or Gumbel-max categorical (T>0) sampling.
    logits [B,V] bf16 or float32 -> token [B] int32 (written in place; also appended to
    out_tokens[b, step] when given). All state on device (hipGraph-safe)."""
    B, V = logits.shape
    if not logits.is_cuda:
        if temperature <= 0:
            t = ref.argmax_sample(logits)
        else:
            # deterministic by (seed, step) like the GPU kernel's splitmix
            # hash (not bit-identical, but the same reproducibility
            # contract on both paths)
            g = torch.Generator().manual_seed(
                (int(seed) * 1000003 + int(step)) & 0x7FFFFFFF)
            t = ref.gumbel_sample(logits, temperature, g)
        token.copy_(t)
        if out_tokens is not None:
            st = int(step)
            for b in range(B):
                if st < out_tokens.shape[1]:
                    out_tokens[b, st] = t[b]
        return token
    lib = require_lib()
    f32 = 1 if logits.dtype == torch.float32 else 0
    max_new = out_tokens.shape[1] if out_tokens is not None else 0
    out_ptr = _ptr(out_tokens) if out_tokens is not None else None
    if B <= 8:
        lib.fei_sample_onepass(_ptr(logits), _ptr(token), out_ptr, _ptr(step),
                               B, V, temperature, seed, max_new, f32,
                               _stream())
    else:
        lib.fei_sample(_ptr(logits), _ptr(token), out_ptr, _ptr(step),
                       _ptr(workspace), B, V, nchunks, temperature, seed,
                       max_new, f32, _stream())
    return token


def sample_shard(logits: torch.Tensor, step: torch.Tensor,
                 v_offset: int, out: torch.Tensor,
                 temperature: float = 0.0, seed: int = 0) -> torch.Tensor:
    """Tensor-parallel shard sampler: reduce THIS rank's logits shard
    [B, V_local] (bf16 on GPU) to (best value, best GLOBAL index) per
    sequence, written into ``out`` [B, 2] f32 (index stored as int bits).
    The ranks then all-gather 8 bytes/seq instead of the vocab row.
    Gumbel noise is keyed by the global index (same splitmix hash as the
    full sampler), so shard+combine is bit-identical to sampling the
    gathered logits. CPU path mirrors the hash exactly."""
    B, Vl = logits.shape
    if not logits.is_cuda:
        vals = logits.float()
        if temperature > 0:
            vals = vals / temperature + ref.hash_gumbel(
                B, Vl, v_offset, int(seed), int(step))
        best = vals.max(dim=-1)
        out[:, 0] = best.values
        out[:, 1].view(torch.int32).copy_(
            (best.indices + v_offset).to(torch.int32))
        return out
    lib = require_lib()
    lib.fei_sample_shard(_ptr(logits), _ptr(out), _ptr(step), B, Vl,
                         int(v_offset), float(temperature), int(seed),
                         _stream())
    return out


# -- persistent weight-streaming decode layer (csrc/stream_layer.hip) -------

STREAM_NSPLIT = 32


def stream_layer_check(C: int, Hq: int, Hkv: int, D: int, I: int) -> int:
    """Residency + shape guard for the persistent layer engine. 0 = OK;
    negative = unsupported (caller uses the launch path). GPU only."""
    lib = require_lib()
    return int(lib.fei_stream_layer_check(C, Hq, Hkv, D, I))


def stream_workspace(spec, device) -> dict:
    """Granule buffers (u64 {tag, payload}) + fail word for the stream
    engine. ~1.3 MB for llama3-8b; zeroed by the engine whenever pos can
    move backwards (prefill) — tags are pos-keyed otherwise."""
    C, D = spec.hidden_size, spec.head_dim
    Hq, Hkv, I = spec.num_heads, spec.num_kv_heads, spec.intermediate_size
    mk = lambda n: torch.zeros(n, dtype=torch.int64, device=device)
    return {
        "g_qkv": mk((Hq + 2 * Hkv) * D),
        "g_att": mk(Hq * D // 2),
        "g_h2": mk(C // 2),
        "g_act": mk(I),
        "g_done": mk(6 * 256),        # [stage, NWG] producer-done granules
        "fail": torch.zeros(1, dtype=torch.int32, device=device),
    }


def stream_layer(x_in: torch.Tensor, h_out: torch.Tensor, lw, spec,
                 k_cache: torch.Tensor, v_cache: torch.Tensor,
                 cos_sin: torch.Tensor, pos: torch.Tensor, ws: dict,
                 layer: int, scale: float) -> None:
    """ONE persistent launch = one decode layer at batch 1 (S1 qkv GEMV ->
    attention -> combine -> O GEMV -> SwiGLU GEMV -> down GEMV with the
    LDS-DMA loader streaming weights ahead across every stage edge).
    Replaces six launch-path kernels; see csrc/stream_layer.hip."""
    lib = require_lib()
    lib.fei_stream_layer(
        _ptr(x_in), _ptr(h_out), _ptr(lw.wqkv), _ptr(lw.wo), _ptr(lw.wgu),
        _ptr(lw.wdown), _ptr(lw.norm_attn), _ptr(lw.norm_mlp),
        _ptr(k_cache), _ptr(v_cache), _ptr(cos_sin), _ptr(pos),
        _ptr(ws["g_qkv"]), _ptr(ws["g_att"]),
        _ptr(ws["g_h2"]), _ptr(ws["g_act"]), _ptr(ws["g_done"]),
        _ptr(ws["dbg"]) if "dbg" in ws else None,
        _ptr(ws["fail"]),
        spec.hidden_size, spec.num_heads, spec.num_kv_heads, spec.head_dim,
        spec.intermediate_size, k_cache.shape[-2], layer, spec.norm_eps,
        scale, _stream())


def advance(pos: torch.Tensor, step: torch.Tensor,
            max_pos: int = 1 << 30) -> None:
    """pos[b] = min(pos[b]+1, max_pos); step += 1 (device-side,
    graph-capturable). max_pos guards the RoPE table / KV cache against
    out-of-bounds indexing when a caller decodes at capacity."""
    if not pos.is_cuda:
        pos.clamp_(max=max_pos - 1)
        pos += 1
        step += 1
        return
    lib = require_lib()
    lib.fei_advance(_ptr(pos), _ptr(step), pos.shape[0], max_pos, _stream())


def mfma_probe(A: torch.Tensor, B: torch.Tensor) -> torch.Tensor:
    """GPU-only: 16x32 @ 32x16 through one MFMA with the kernels' fragment
    maps; falsifies layout assumptions (tests/test_ops_gpu.py)."""
    lib = require_lib()
    C = torch.empty(16, 16, dtype=torch.float32, device=A.device)
    lib.fei_mfma_probe(_ptr(A.contiguous()), _ptr(B.contiguous()), _ptr(C),
                       _stream())
    return C


# -- decode GEMV dispatch ----------------------------------------------------

# What becomes of a GEMV's sums (csrc/gemv.hip).
_BF16, _RES, _SWIGLU = 0, 1, 2


def _launch_gemv(out, x2, gain, w, wscale, N: int, eps: float, epi: int,
                 ssq=None) -> None:
    M, K = x2.shape
    if M not in _GEMV_ROWS:
        raise ValueError(f"the GEMV takes {_GEMV_ROWS} rows, got {M}")
    opt = lambda t: None if t is None else _ptr(t)
    require_lib().fei_gemv(_ptr(out), _ptr(x2), opt(gain), _ptr(w),
                           opt(wscale), M, N, K, eps, epi, opt(ssq),
                           _stream())


_GEMV_ROWS = (1, 2, 3, 4, 8)


def _gemv_ok(M: int, K: int) -> bool:
    return M in _GEMV_ROWS and K % 8 == 0


def _norm_inside(how: str, M: int, K: int, sums, wnorm) -> bool:
    """Whether a product takes rows under a norm: the GEMV keeps them in LDS;
    the tile for few rows needs their sums of squares, and keeps the gains,
    which go to LDS by loads that have to be aligned."""
    if how == "skinny":
        return (sums is not None and K <= 16384
                and wnorm.data_ptr() % 16 == 0)
    return M * K * 2 <= 128 * 1024


def _product(x: torch.Tensor, w: torch.Tensor, M: int, K: int, rows_out: int,
             out: Optional[torch.Tensor] = None) -> Optional[str]:
    """Which kernel takes the M rows x @ w^T: "skinny" (matrix units), "gemv",
    or None (the library; CPU). ``out``: where the caller wants the results."""
    if not (x.is_cuda and M and rows_out and (
            out is None or _fits(out, x, M * rows_out))):
        return None
    return _kernel_for(x, w, M, K)


def _fits(out: Optional[torch.Tensor], x: torch.Tensor, n: int) -> bool:
    """Whether a kernel can write its n results, of x's type, to out."""
    return out is None or (out.dtype is x.dtype and out.numel() == n
                           and out.is_contiguous()
                           and out.get_device() == x.get_device())


def _kernel_for(x: torch.Tensor, w: torch.Tensor, M: int,
                K: int) -> Optional[str]:
    if not _mixers.match(x, w, K):
        return None
    # the callers copy rows with gaps; a copy is aligned
    if _mixers.skinny_sizes(M, K, x if x.is_contiguous() else w, w, 2):
        return "skinny"
    return "gemv" if _gemv_ok(M, K) else None


def own_product(M: int, w: torch.Tensor) -> bool:
    """Whether M rows of w's type (a tensor of their own) times w run in this
    library's kernels, which add to a residual and make a SwiGLU without a
    launch of its own."""
    N, K = w.shape
    return w.is_cuda and N > 0 and _kernel_for(w, w, M, K) is not None


def linear_decode(x: torch.Tensor, w: torch.Tensor,
                  out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """F.linear for skinny M: streaming GEMV or matrix-core tile on GPU. Falls
    back to torch for unsupported shapes, types and layouts, and on the CPU."""
    K, N = x.shape[-1], w.shape[0]
    M = x.numel() // K
    how = _product(x, w, M, K, N, out)
    if how is None:
        # M > 256 for one: nothing is asked of few rows that they have not been
        if (M > 256 and out is None and x.is_cuda and w.dim() == 2
                and x.is_contiguous() and _tiles.linear_ok(M, x, w)):
            return _tiles.linear(x.view(M, K), w).view(*x.shape[:-1], N)
        return torch.nn.functional.linear(x, w)
    x2 = x.contiguous().view(M, K)
    if out is None:
        out = torch.empty(*x.shape[:-1], N, dtype=x.dtype, device=x.device)
    if how == "skinny":
        _mixers.skinny(out, x2, w, N, _mixers.EPI_BF16)
    else:
        _launch_gemv(out, x2, None, w, None, N, 0.0, _BF16)
    return out


def _many_rows(M: int, x: torch.Tensor, wgu: torch.Tensor,
               out: Optional[torch.Tensor] = None) -> Optional[str]:
    """The kernel of more than a few rows that makes a SwiGLU, if one does. Tiles
    write 16 bytes at a time."""
    if _rows.swiglu_ok(M, x, wgu):
        return "rows"
    # a copy of rows with gaps is aligned
    if (wgu.shape[0] % 16 == 0 and _tiles.types_ok(x)
            and (out is None or out.data_ptr() % 16 == 0)
            and _tiles.act_ok(M, x if x.is_contiguous() else wgu, wgu)):
        return "tile"
    return None


def gemv_swiglu(x: torch.Tensor, wgu: torch.Tensor,
                out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Fused gate/up product + SwiGLU: x [M,K] @ [2I,K]^T -> silu(g)*u [M,I]."""
    K, I = x.shape[-1], wgu.shape[0] // 2
    M = x.numel() // K
    how = _product(x, wgu, M, K, I, out)
    if (how is None and M and x.is_cuda and _mixers.match(x, wgu, K)
            and _fits(out, x, M * I)):
        how = _many_rows(M, x, wgu, out)
    if how is None:
        return swiglu(torch.nn.functional.linear(x, wgu))
    x2 = x.contiguous().view(M, K)
    if out is None:
        out = torch.empty(*x.shape[:-1], I, dtype=x.dtype, device=x.device)
    if how == "rows":
        _rows.swiglu_product(x2, wgu, out)
        return out
    if how == "tile":
        _tiles.product(x2, wgu, out.view(M, I), I, _tiles.TILE_SWIGLU)
        return out
    if how == "skinny":
        _mixers.skinny(out, x2, wgu, I, _mixers.EPI_SWIGLU, act=out, stride=I)
    else:
        _launch_gemv(out, x2, None, wgu, None, I, 0.0, _SWIGLU)
    return out


def gemv_res(x: torch.Tensor, w: torch.Tensor, res: torch.Tensor,
             ssq_out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """res += x @ w^T (epilogue residual add; in place on res [M,N]).

    ``ssq_out`` [M] f32, pre-zeroed: the kernel also accumulates the
    sum-of-squares of the updated residual rows, which a following
    gemv_norm/gemv_swiglu_norm takes as ``ssq``. Ignored on the CPU fallback —
    consumers recompute exactly there."""
    K, N = x.shape[-1], w.shape[0]
    M = x.numel() // K
    how = _product(x, w, M, K, N, res)
    if ssq_out is not None and how == "skinny" and _gemv_ok(M, K):
        how = "gemv"
    if how is None:
        lin = torch.nn.functional.linear(x, w)
        res.copy_((res.float() + lin.float().view_as(res)).to(res.dtype))
        if ssq_out is not None and x.is_cuda:
            ssq_out += res.float().reshape(M, N).pow(2).sum(-1)
    elif how == "skinny":
        _mixers.skinny(res, x.contiguous().view(M, K), w, N,
                       _mixers.EPI_RES_BF16)
    else:
        _launch_gemv(res, x.contiguous().view(M, K), None, w, None, N, 0.0,
                     _RES, ssq_out)
    return res


def add_product(x: torch.Tensor, w: torch.Tensor, res: torch.Tensor,
                any_tiles: bool = False) -> Optional[torch.Tensor]:
    """gemv_res, for a chain: returns the sums of squares of the new rows by
    tiles of 16 columns, for the ``sums`` of the products that read them under a
    norm, or None where those do not need them. ``any_tiles``: of any number of
    columns, which leaves the kernel its choice of blocks."""
    K, N = x.shape[-1], w.shape[0]
    M = x.numel() // K
    if _product(x, w, M, K, N, res) != "skinny":
        gemv_res(x, w, res)
        return None
    # blocks have 8 columns where with 16 CUs would be left without
    sums = torch.empty(M, -(-N // (8 if any_tiles and N <= 2048 else 16)),
                       dtype=torch.float32, device=x.device)
    _mixers.skinny(res, x.contiguous().view(M, K), w, N, _mixers.EPI_RES_BF16,
                   sums_out=sums)
    return sums


def gemv_norm(res: torch.Tensor, wnorm: torch.Tensor, w: torch.Tensor,
              eps: float = 1e-5,
              out: Optional[torch.Tensor] = None,
              ssq: Optional[torch.Tensor] = None,
              sums: Optional[torch.Tensor] = None) -> torch.Tensor:
    """out = rmsnorm(res)*wnorm @ w^T, the norm inside the product.

    ``ssq`` [M] f32: the sums of squares of res rows, if the caller has them
    (from a prior gemv_res ``ssq_out``). ``sums``: what add_product returned
    for these rows."""
    K, N = res.shape[-1], w.shape[0]
    M = res.numel() // K
    how = _product(res, w, M, K, N, out)
    if how is None:
        return torch.nn.functional.linear(rmsnorm(res, wnorm, eps), w)
    if not _norm_inside(how, M, K, sums, wnorm):
        return linear_decode(rmsnorm(res, wnorm, eps), w, out)
    if out is None:
        out = torch.empty(*res.shape[:-1], N, dtype=res.dtype, device=res.device)
    if how == "skinny":
        _mixers.skinny(out, res.contiguous().view(M, K), w, N,
                       _mixers.EPI_BF16, norm=(wnorm, sums, eps))
        return out
    _launch_gemv(out, res.contiguous().view(M, K), wnorm, w, None, N, eps,
                 _BF16, ssq)
    return out


def gemv_swiglu_norm(res: torch.Tensor, wnorm: torch.Tensor,
                     wgu: torch.Tensor, eps: float = 1e-5,
                     out: Optional[torch.Tensor] = None,
                     ssq: Optional[torch.Tensor] = None,
                     sums: Optional[torch.Tensor] = None) -> torch.Tensor:
    """out = silu(g)*u where [g;u] = rmsnorm(res)*wnorm @ wgu^T.
    ``ssq``, ``sums``: see gemv_norm."""
    K, I = res.shape[-1], wgu.shape[0] // 2
    M = res.numel() // K
    how = _product(res, wgu, M, K, I, out)
    if how is None:
        return swiglu(torch.nn.functional.linear(rmsnorm(res, wnorm, eps), wgu))
    if not _norm_inside(how, M, K, sums, wnorm):
        return gemv_swiglu(rmsnorm(res, wnorm, eps), wgu, out)
    if out is None:
        out = torch.empty(*res.shape[:-1], I, dtype=res.dtype, device=res.device)
    if how == "skinny":
        _mixers.skinny(None, res.contiguous().view(M, K), wgu, I,
                       _mixers.EPI_SWIGLU, act=out, stride=I,
                       norm=(wnorm, sums, eps))
        return out
    _launch_gemv(out, res.contiguous().view(M, K), wnorm, wgu, None, I, eps,
                 _SWIGLU, ssq)
    return out


def prefetch(w: torch.Tensor, max_bytes: int, sink: torch.Tensor,
             n_blocks: int = 512, stream=None) -> None:
    """Stream the first ``max_bytes`` of ``w`` through cache-filling loads
    (L2/L3 prefill for a later kernel's reads). GPU-only no-op helper for
    the decode prefetch experiment; launched on a side stream."""
    if not w.is_cuda:
        return
    lib = require_lib()
    bytes_ = min(max_bytes, w.numel() * w.element_size())
    sp = stream if stream is not None else _stream()
    lib.fei_prefetch(_ptr(w), bytes_, _ptr(sink), n_blocks, sp)


def attn_decode_paged(q, k_pool, v_pool, block_table, pos, splits: int = 32,
                      scale: Optional[float] = None,
                      workspace: Optional[Tuple[torch.Tensor, torch.Tensor]] = None,
                      out: Optional[torch.Tensor] = None,
                      k: Optional[torch.Tensor] = None,
                      v: Optional[torch.Tensor] = None,
                      table: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Decode attention over a PAGED KV pool (engine/kv_cache.PagedKVPool):
    pools [num_blocks, Hkv, BS, D], block_table [B, max_blocks] int32 maps
    logical key blocks to physical pool blocks. n = pos[b]+1 keys.
    When (k, v, table) are given the kernel also fuses the step's RoPE +
    paged KV-append: q is the RAW qkv view and the pool row for position
    pos[b] is written in-kernel (mirrors attn_decode's fused form)."""
    B, Hq, D = q.shape
    n_blocks, Hkv, BS, _ = k_pool.shape
    assert BS & (BS - 1) == 0, "block size must be a power of two"
    bs_log = BS.bit_length() - 1
    scale = scale if scale is not None else 1.0 / math.sqrt(D)
    if not q.is_cuda:
        if table is not None:
            # reference path: rope q/k and append into the POOL rows
            q = ref.apply_rope(q, pos.long(), table).to(q.dtype)
            k_r = ref.apply_rope(k, pos.long(), table).to(k.dtype)
            for b in range(B):
                p = int(pos[b])
                blk = int(block_table[b, p >> bs_log])
                k_pool[blk, :, p & (BS - 1), :] = k_r[b]
                v_pool[blk, :, p & (BS - 1), :] = v[b]
        # gather logical order into a contiguous cache, then reference
        max_len = block_table.shape[1] * BS
        kc = torch.zeros(B, Hkv, max_len, D, dtype=k_pool.dtype)
        vc = torch.zeros_like(kc)
        for b in range(B):
            for j, blk in enumerate(block_table[b].tolist()):
                if blk < 0:
                    continue
                kc[b, :, j * BS:(j + 1) * BS] = k_pool[blk]
                vc[b, :, j * BS:(j + 1) * BS] = v_pool[blk]
        return ref.attn_decode(q, kc, vc, pos + 1, scale)
    return _launch_attn_decode(
        q, k_pool, v_pool, block_table, block_table.shape[1] << bs_log,
        bs_log, Hkv, pos, splits, scale, workspace, out, k, v, table)


def layernorm(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor,
              eps: float = 1e-5, residual: Optional[torch.Tensor] = None,
              out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """LayerNorm of (x [+ residual]) over the last dim (encoder blocks)."""
    if not x.is_cuda:
        return ref.layernorm(x, weight, bias, eps, residual)
    lib = require_lib()
    x2 = x.contiguous()
    rows = x2.numel() // x2.shape[-1]
    if out is None:
        out = torch.empty_like(x2)
    res_ptr = _ptr(residual.contiguous()) if residual is not None else _ptr(x2)
    lib.fei_add_layernorm(_ptr(out), _ptr(x2), res_ptr, _ptr(weight),
                          _ptr(bias), rows, x2.shape[-1], eps,
                          1 if residual is not None else 0, _stream())
    return out


def linear_bias(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor,
                act_gelu: bool = False) -> torch.Tensor:
    """x @ w^T + bias, and its GELU if asked for (encoder blocks)."""
    M = x.numel() // max(x.shape[-1], 1)
    if (x.is_cuda and _mixers.skinny_ok(M, x.shape[-1], x, w)
            and _mixers.dense(bias, torch.bfloat16, x, w.shape[0])):
        out = torch.empty(*x.shape[:-1], w.shape[0], dtype=x.dtype,
                          device=x.device)
        _mixers.skinny(out, x.view(M, -1), w, w.shape[0],
                       _mixers.EPI_GELU if act_gelu else _mixers.EPI_BF16,
                       bias16=bias)
        return out
    if (act_gelu and x.is_cuda and _mixers.plain(x, w)
            and _tiles.act_ok(M, x, w)
            and _tiles.types_ok(bias)
            and _mixers.dense(bias, torch.bfloat16, x, w.shape[0])
            and bias.data_ptr() % 16 == 0):
        out = torch.empty(*x.shape[:-1], w.shape[0], dtype=x.dtype,
                          device=x.device)
        _tiles.product(x.view(M, -1), w, out.view(M, -1), w.shape[0],
                       _tiles.TILE_GELU, bias)
        return out
    y = torch.nn.functional.linear(x, w, bias)
    return gelu(y) if act_gelu else y


# Rows up to which all layers are launched from one call; one by one, with the
# library's products, they take 1.6 ms and more from Python (12 layers of 768), of
# which the GPU works a part: 100 rows 667 us, 512 848, 1000 979. Beyond, the
# library's products are the faster ones and the GPU is never idle.
ENCODER_ROWS = 1024


def _encoder_weights(weights, C: int, HD: int, inner: int):
    """Where kernels find an encoder's weights, 12 a layer (see encoder_layers), 16 bytes
    at a time, or None if one is not of the sizes that they read."""
    shapes = ((3 * HD, C), (3 * HD,), (C, HD), (C,), (C,), (C,),
              (inner, C), (inner,), (C, inner), (C,), (C,), (C,))
    layers, rest = divmod(len(weights), len(shapes))
    at, low = [], rest
    for t, shape in zip(weights, shapes * layers):
        if (t.dtype is not torch.bfloat16 or t.shape != shape
                or not t.is_contiguous()):
            return None
        p = t.data_ptr()
        at.append(p)
        low |= p % 16
    return None if low else at


def encoder_layers(h: torch.Tensor, weights, heads: int, dim: int, inner: int,
                   pos0: torch.Tensor, kv_len: torch.Tensor,
                   eps: float) -> Optional[torch.Tensor]:
    """All layers of an encoder over h [B, S, C], which is overwritten, launched
    from one call, or None where its few-row kernels do not take them. ``weights``: 12 a layer, a
    product's followed by its bias: q, k and v; output; LayerNorm; inner;
    outer; LayerNorm. 24 rows, 12 layers of 768: 392 us, 942 launched one by one."""
    B, S, C = h.shape
    M, HD = B * S, heads * dim
    if not (h.is_cuda and h.is_contiguous() and dim in (64, 128)
            and h.dtype == torch.bfloat16 and 2 < M <= ENCODER_ROWS
            and C % 64 == HD % 64 == inner % 64 == 0
            and h.data_ptr() % 16 == 0):
        return None
    ptrs = _encoder_weights(weights, C, HD, inner)
    if ptrs is None:
        return None

    def rows(n):
        return torch.empty(M, n, dtype=h.dtype, device=h.device)
    h1, tmp = rows(C), rows(C)
    qkv, att, mid = rows(3 * HD), rows(HD), rows(inner)
    splits = _prefill_splits(B, heads, S, S, dim)
    po = pml = None
    if splits > 1:
        ws = torch.empty(M * heads * splits * (dim + 2), dtype=torch.float32,
                         device=h.device)
        po, pml = _ptr(ws), _ptr(ws) + M * heads * splits * dim * 4
    # parts of K for about a tile of 64 x 64 a CU, of 256 steps at least
    tiles = -(-M // 64) * -(-C // 64)
    p1, p2 = (min(256 // tiles, 8, k // 256) if M > 64 and C <= 2048 else 0
              for k in (HD, inner))
    p1, p2 = (p if p > 1 else 0 for p in (p1, p2))
    parts = torch.empty(max(p1, p2, 1) * M * C, dtype=torch.float32,
                        device=h.device)
    require_lib().fei_encoder_layers(
        (_vp * len(ptrs))(*ptrs), len(ptrs) // 12, _ptr(h), _ptr(h1),
        _ptr(tmp), _ptr(qkv), _ptr(att), _ptr(mid), _ptr(pos0), _ptr(kv_len),
        B, S, heads, dim, C, inner, 1.0 / math.sqrt(dim), eps, splits, po, pml,
        _ptr(parts), p1, p2, _stream())
    return h


# Rows, padding among them, from which those that texts have are packed, and up to which
# their products run in tiles of 64 x 64, beyond in k_tile's. Us of 12 layers of 768,
# texts of a quarter to all of the length, with padding, in tiles of 64, in k_tile's: 660
# rows 712, 645, 1053; 1500 1475, 782, 1088; 2560 1310, 1015, 1145; 3200 1396, 1077, 1202;
# 3600 1360, 1185, 1249; 4500 1594, 1441, 1396; 6400 1944, -, 1507; 16384 3779, -, 2575.
# Of as little as a fifth padding 3072 part at: 1336, 1216, 1255, and 3600 1362, 1434, 1361.
ENCODER_PACKED_FROM = 640
ENCODER_PACKED_ROWS = 3072


def encoder_packing_pays(M: int, texts: int, inner: int) -> bool:
    """Whether an encoder that could leave out padding is faster so, where the host knows
    that of the M rows the texts have ``texts``. All rows have fewer launches up to
    ENCODER_ROWS, the library's tiles beyond, which suit some sizes better. Us, all rows,
    packed; no padding, a tenth, a fifth: 1024 rows 738, 760; 737, 759; 736, 729. 2560 1314,
    1211; 1316, 1182; 1306, 1094. 3600 1406, 1506; 1366, 1399; 1362, 1361. 6144 1973, 2071;
    2000, 2041; 1989, 1771. 9000 2695, 2545. 12800 3507, 3337. Rows whose widest product is
    whole rounds of the library's tiles: 16384 3791, 3890, of 3 % padding 3801, 3625; 32768
    7488, 7576, of 3 % 7468, 7345."""
    if M <= ENCODER_ROWS or 2700 < M <= 8192:
        return texts <= 0.85 * M
    if M <= 2700:
        return True
    tiles = -(-M // 256) * -(-inner // 256)
    return texts <= 0.98 * M or tiles % _tiles.CUS != 0


def _embedding_ok(ids, tok, pos, gain, shift) -> bool:
    """Whether a kernel can look up the rows of ids [B, S] and norm them: all on the
    current device, 16 bytes at a time."""
    C = tok.shape[-1]
    tensors = (tok, pos, gain, shift)
    return (tok.is_cuda and ids.dtype is torch.int64 and ids.is_contiguous()
            and ids.dim() == 2 and ids.numel() > 0 and ids.numel() * C < 1 << 31
            and tok.dim() == pos.dim() == 2 and ids.shape[1] <= pos.shape[0]
            and C % 8 == 0 and 0 < C <= 2048 and pos.shape[1] == C
            and gain.shape == shift.shape == (C,)
            and all(t.dtype is torch.bfloat16 and t.is_contiguous()
                    and t.data_ptr() % 16 == 0 for t in tensors)
            and all(t.get_device() == torch.cuda.current_device()
                    for t in (ids, *tensors))
            and _tiles._memory(ids, *tensors)
            and not (torch.is_grad_enabled()
                     and any(t.requires_grad for t in tensors)))


def embed_layernorm(ids: torch.Tensor, tok: torch.Tensor, pos: torch.Tensor,
                    gain: torch.Tensor, shift: torch.Tensor, eps: float,
                    dtype: torch.dtype) -> torch.Tensor:
    """LayerNorm of tok[ids] + pos[:S], ids [B, S] -> [B, S, C]."""
    B, S = ids.shape
    if not (dtype is torch.bfloat16 and _embedding_ok(ids, tok, pos, gain, shift)):
        h = torch.nn.functional.embedding(ids, tok) + pos[:S].unsqueeze(0)
        return layernorm(h.to(dtype), gain, shift, eps)
    out = torch.empty(B, S, tok.shape[1], dtype=dtype, device=ids.device)
    require_lib().fei_embed_layernorm(
        _ptr(out), _ptr(ids), _ptr(tok), _ptr(pos), _ptr(gain), _ptr(shift), B, S,
        tok.shape[1], tok.shape[0], eps, None, _stream())
    return out


def encoder_packed(ids: torch.Tensor, tok: torch.Tensor, pos: torch.Tensor,
                   gain: torch.Tensor, shift: torch.Tensor, weights, heads: int,
                   dim: int, inner: int, lens: torch.Tensor, eps: float
                   ) -> Optional[torch.Tensor]:
    """An encoder over texts of unlike lengths: ids [B, S], of which text b has lens[b],
    and what embed_layernorm takes -> embeddings [B, C] float32, or None where its
    kernels do not take them. Rows that no text has are left out, without the host's
    knowing how many those are. ``weights``: see encoder_layers."""
    B, S = ids.shape
    C, HD = tok.shape[1], heads * dim
    M = B * S
    if not (tok.is_cuda and dim in (64, 128) and M > ENCODER_PACKED_FROM
            and M * max(3 * HD, inner, C) < 1 << 31
            and C % 64 == HD % 64 == inner % 64 == 0
            and _embedding_ok(ids, tok, pos, gain, shift)
            and all(t.get_device() == ids.get_device() for t in weights)
            and lens.device == ids.device and lens.dtype is torch.int32
            and lens.shape == (B,) and lens.is_contiguous()
            and _tiles.types_ok(lens, *weights)
            and _prefill_splits(B, heads, S, S, dim) == 1):
        return None
    ptrs = _encoder_weights(weights, C, HD, inner)
    if ptrs is None:
        return None

    def rows(n):
        return torch.empty(M, n, dtype=tok.dtype, device=ids.device)
    room = [rows(n) for n in (C, C, C, 3 * HD, HD, inner)]
    starts = torch.empty(B + 1, dtype=torch.int32, device=ids.device)
    out = torch.empty(B, C, dtype=torch.float32, device=ids.device)
    parts, many = None, M > ENCODER_PACKED_ROWS
    if many:
        p1, p2 = (_tiles.parts_up_to(M, C, k) for k in (HD, inner))
    else:
        # as in encoder_layers, for two thirds of the rows
        tiles = -(-M * 2 // 3 // 64) * -(-C // 64)
        p1, p2 = (min(256 // tiles, 8, k // 256) for k in (HD, inner))
    p1, p2 = (p if p > 1 else 0 for p in (p1, p2))
    if p1 or p2:
        parts = torch.empty(max(p1, p2) * M * C, dtype=torch.float32,
                            device=ids.device)
    require_lib().fei_encoder_packed(
        (_vp * len(ptrs))(*ptrs), len(ptrs) // 12, _ptr(out), _ptr(ids), _ptr(tok),
        _ptr(pos), tok.shape[0], _ptr(gain), _ptr(shift),
        *(_ptr(t) for t in room), _ptr(lens), _ptr(starts), B, S, heads, dim, C,
        inner, 1.0 / math.sqrt(dim), eps, many,
        None if parts is None else _ptr(parts), p1, p2, _stream())
    return out


def pool_unit(h: torch.Tensor, lens: torch.Tensor) -> torch.Tensor:
    """Mean of the first lens[b] rows of h [B, S, C], scaled to length 1 ->
    [B, C] float32."""
    B, S, C = h.shape
    if not (h.is_cuda and h.dtype == torch.bfloat16 and h.is_contiguous()
            and h.numel() and C % 8 == 0 and C <= 2048
            and h.data_ptr() % 16 == 0 and lens.device == h.device
            and lens.dtype == torch.int32
            and lens.is_contiguous()):
        mask = (torch.arange(S, device=h.device).unsqueeze(0)
                < lens.unsqueeze(1)).float().unsqueeze(-1)
        mean = (h.float() * mask).sum(1) / mask.sum(1).clamp_min(1.0)
        return torch.nn.functional.normalize(mean, dim=-1)
    out = torch.empty(B, C, dtype=torch.float32, device=h.device)
    require_lib().fei_pool_unit(_ptr(out), _ptr(h), _ptr(lens), B, S, C,
                                _stream())
    return out


def gelu(x: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    if not x.is_cuda:
        return ref.gelu(x)
    lib = require_lib()
    x2 = x.contiguous()
    if out is None:
        out = torch.empty_like(x2)
    lib.fei_gelu(_ptr(out), _ptr(x2), x2.numel(), _stream())
    return out


# -- fp8 weight-quantized decode path (OCP e4m3fn; serving mode) -------------

def quant_fp8(w: torch.Tensor):
    """Quantize a weight matrix [N,K] to e4m3fn + per-row fp32 scales."""
    if not w.is_cuda:
        return ref.quant_fp8(w)
    lib = require_lib()
    N, K = w.shape
    w8 = torch.empty(N, K, dtype=torch.uint8, device=w.device)
    scales = torch.empty(N, dtype=torch.float32, device=w.device)
    lib.fei_quant_fp8_rows(_ptr(w8), _ptr(scales), _ptr(w.contiguous()),
                           N, K, _stream())
    return w8, scales


def gemv_norm_fp8(res, wnorm, w8, wscale, eps: float = 1e-5,
                  out: Optional[torch.Tensor] = None) -> torch.Tensor:
    M = res.numel() // res.shape[-1]
    K = res.shape[-1]
    N = w8.shape[0]
    if not res.is_cuda:
        w = ref.dequant_fp8(w8, wscale).to(res.dtype)
        return torch.nn.functional.linear(rmsnorm(res, wnorm, eps), w)
    assert M * K * 2 <= 64 * 1024, \
        "fp8 norm-GEMV stages M*K bf16 activations in LDS (<=64 KB)"
    if out is None:
        out = torch.empty(*res.shape[:-1], N, dtype=res.dtype, device=res.device)
    _launch_gemv(out, res.contiguous().view(M, K), wnorm, w8, wscale, N, eps,
                 _BF16)
    return out


def gemv_res_fp8(x, w8, wscale, res) -> torch.Tensor:
    M = x.numel() // x.shape[-1]
    K = x.shape[-1]
    N = w8.shape[0]
    if not x.is_cuda:
        w = ref.dequant_fp8(w8, wscale).to(x.dtype)
        lin = torch.nn.functional.linear(x, w)
        res.copy_((res.float() + lin.float().view_as(res)).to(res.dtype))
        return res
    _launch_gemv(res, x.contiguous().view(M, K), None, w8, wscale, N, 0.0,
                 _RES)
    return res


def attn_decode_product_fp8(q, k_cache, v_cache, pos, w8, wscale, res,
                            splits: int = 32, scale: Optional[float] = None,
                            workspace=None, out=None, k=None, v=None,
                            table=None) -> torch.Tensor:
    """attn_decode of one sequence, and gemv_res_fp8 of its result, which may be left to
    the product to sum: ``out`` need not have it afterwards."""
    B, Hq, D = q.shape
    if not (q.is_cuda and B == 1 and Hq * D % 16 == 0 and res.is_contiguous()
            and res.dtype == torch.bfloat16 and res.numel() == w8.shape[0]):
        att = attn_decode(q, k_cache, v_cache, pos, splits, scale, workspace, out, k,
                          v, table)
        return gemv_res_fp8(att.reshape(B, -1), w8, wscale, res)
    _launch_attn_decode(q, k_cache, v_cache, None, k_cache.shape[2], 0,
                        k_cache.shape[1], pos, splits,
                        scale if scale is not None else 1.0 / math.sqrt(D),
                        workspace, out, k, v, table, (w8, wscale, res))
    return res


def gemv_swiglu_norm_fp8(res, wnorm, w8, wscale, eps: float = 1e-5,
                         out: Optional[torch.Tensor] = None) -> torch.Tensor:
    M = res.numel() // res.shape[-1]
    K = res.shape[-1]
    I = w8.shape[0] // 2
    if not res.is_cuda:
        w = ref.dequant_fp8(w8, wscale).to(res.dtype)
        return swiglu(torch.nn.functional.linear(rmsnorm(res, wnorm, eps), w))
    assert M * K * 2 <= 64 * 1024
    if out is None:
        out = torch.empty(*res.shape[:-1], I, dtype=res.dtype, device=res.device)
    _launch_gemv(out, res.contiguous().view(M, K), wnorm, w8, wscale, I, eps,
                 _SWIGLU)
    return out
