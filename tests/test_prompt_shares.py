"""How prompt attention's keys are cut into shares, at the numbers of blocks where the
rule changes."""

import math

import pytest
import torch

from fei_amd import ops

DEV = "cuda:0"


@pytest.mark.parametrize("dim", [64, 128])
def test_shares_fill_whole_rounds(dim):
    for B in (1, 2, 7):
        for Hkv in (1, 8, 12):
            for rows in (1, 128, 129, 1360, 1361, 3000):
                for max_seq in (64, 500, 2000, 9000):
                    n = ops._prefill_splits(B, Hkv, rows, max_seq, dim)
                    blocks = B * Hkv * -(-rows // 128)
                    assert 1 <= n <= 16
                    assert n == 1 or (n * blocks <= 512 and n * 192 <= max_seq)
                    places = 256 if dim == 128 and blocks <= 85 else 512
                    if n > 1:
                        assert n * blocks <= places
                        # and no more do, of 16 and of three tiles of 64 keys each
                        assert (n == min(16, max_seq // 192)
                                or (n + 1) * blocks > places)


# on both sides of the blocks at which the rule changes
@pytest.mark.parametrize("blocks,wide,narrow", [
    (1, 16, 16), (16, 16, 16), (24, 10, 16), (32, 8, 16), (64, 4, 8), (85, 3, 6),
    (86, 5, 5), (128, 4, 4), (170, 3, 3), (171, 2, 2), (192, 2, 2), (193, 1, 1)])
def test_shares_of_blocks(blocks, wide, narrow):
    assert ops._prefill_splits(1, 1, 128 * blocks, 10 ** 6, 128) == wide
    assert ops._prefill_splits(1, 1, 128 * blocks, 10 ** 6, 64) == narrow


# 8 heads of keys, 4 queries each: 10 and 11 blocks of rows a head lie on either side of 85
# blocks, 24 (of 192, with two shares) is the most
@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S,P", [(32, 900), (33, 1500), (320, 1700), (321, 1700),
                                 (768, 3100)])
def test_shares_against_float32(S, P, D):
    g = torch.Generator(device=DEV).manual_seed(S)
    T = P + S
    q = torch.randn(1, S, 32, D, generator=g, device=DEV).to(torch.bfloat16)
    k, v = (torch.randn(1, 8, T, D, generator=g, device=DEV).to(torch.bfloat16)
            for _ in range(2))
    blocks = 8 * -(-4 * S // 128)
    places = 256 if D == 128 and blocks <= 85 else 512
    assert ops._prefill_splits(1, 8, 4 * S, T, D) == min(16, T // 192, places // blocks) > 1
    pos0 = torch.tensor([P], dtype=torch.int32, device=DEV)
    got = ops.attn_prefill(q, k, v, pos0, scale=D ** -0.5).float()
    hide = torch.arange(T, device=DEV) > torch.arange(P, T, device=DEV).unsqueeze(1)
    for h in (0, 5, 31):
        s = q[0, :, h].float() @ k[0, h // 4].float().T / math.sqrt(D)
        want = torch.softmax(s.masked_fill(hide, float("-inf")), -1) @ v[0, h // 4].float()
        # weights and results are rounded to 2^-9 each; twice that
        err = (got[0, :, h] - want).norm() / want.norm()
        assert err < 2.0 ** -7, err
