"""HIP kernels at the sizes where their tiles, splits and dispatch rules
meet, against float64 on the same bfloat16 inputs."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def lib():
    from fei_amd import ops
    ops.require_lib()
    return ops


def randbf(*shape, seed=0, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * scale).bfloat16()


def row_err(got, want):
    """Largest error of a row, relative to the row."""
    d = (got.double() - want).norm(dim=-1)
    return float((d / want.norm(dim=-1).clamp_min(1e-30)).max())


# -- prompt attention ----------------------------------------------------------

def attend64(q, k, v, pos0, scale, kv_len=None):
    S, T = q.shape[1], k.shape[2]
    G = q.shape[2] // k.shape[1]
    k, v = (t.double().repeat_interleave(G, 1) for t in (k, v))
    s = torch.matmul(q.transpose(1, 2).double(),
                     k.transpose(2, 3).contiguous()) * scale
    key = torch.arange(T, device=DEV).view(1, 1, 1, T)
    last = (pos0.view(-1, 1, 1, 1) + torch.arange(S, device=DEV).view(1, 1, S, 1)
            if kv_len is None else kv_len.view(-1, 1, 1, 1) - 1)
    p = torch.softmax(s.masked_fill(key > last, float("-inf")), -1)
    return torch.matmul(p.nan_to_num(0.0), v).transpose(1, 2)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S,Hq,Hkv,T,pos0,kv_len,scale", [
    (1, 8, 2, 64, [0], None, None),             # one key
    (33, 4, 1, 128, [31, 0], None, None),       # 132 rows: a block and a bit
    (63, 5, 1, 700, [637], None, None),         # groups of 5, splits
    (32, 12, 3, 1400, [1368, 2], None, None),   # one split used, or all
    (257, 3, 3, 257, [0], None, -0.2),          # groups of 1; scale < 0
    (40, 4, 2, 64, [10], None, 0.0),            # all keys alike
    (65, 3, 3, 65, [0, 0, 0], [65, 1, 0], None),   # no key at all
    (70, 2, 2, 4000, [0, 0], [4000, 129], None),
])
def test_attn_prefill_geometries(lib, D, S, Hq, Hkv, T, pos0, kv_len, scale):
    B, W = len(pos0), (Hq + 2 * Hkv) * D
    qkv = randbf(B, S, W, seed=S)
    q = qkv.as_strided((B, S, Hq, D), (S * W, W, D, 1))
    k, v = randbf(B, Hkv, T, D, seed=1), randbf(B, Hkv, T, D, seed=2)
    # what lies past the keys is never used
    ends = kv_len or [p + S for p in pos0]
    kn, vn = k.clone(), v.clone()
    for b, n in enumerate(ends):
        kn[b, :, n:] = vn[b, :, n:] = float("nan")
    p0 = torch.tensor(pos0, dtype=torch.int32, device=DEV)
    kl = None if kv_len is None else torch.tensor(kv_len, dtype=torch.int32,
                                                  device=DEV)
    got = lib.attn_prefill(q, kn, vn, p0, scale=scale, causal=kv_len is None,
                           kv_len=kl)
    want = attend64(q, k, v, p0, D ** -0.5 if scale is None else scale, kl)
    # weights and results are each rounded to bfloat16 once: 2^-9 of each
    # weight times its value, and 2^-9 of the result
    assert row_err(got, want) < 2 ** -7
