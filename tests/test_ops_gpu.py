"""GPU numerics tests: each HIP kernel vs the fp32 torch reference on the
same bf16 inputs (tests/conftest.py registers the gpu marker)."""

import math

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
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(torch.bfloat16)


def test_mfma_probe_layouts(lib):
    """Falsify the assumed A/B/C fragment maps with asymmetric operands
    (guide §3: symmetric B would hide a transposed C-write)."""
    A = randbf(16, 32, seed=1)
    B = (torch.arange(32 * 16, device=DEV).float().view(32, 16) * 0.01 + 0.1).to(torch.bfloat16)
    C = lib.mfma_probe(A, B)
    ref = A.float() @ B.float()
    assert torch.allclose(C, ref, atol=1e-2, rtol=1e-2), \
        f"max err {(C - ref).abs().max().item()}"


def test_rmsnorm(lib):
    from fei_amd.ops import reference as ref
    x = randbf(33, 4096, seed=2)
    w = randbf(4096, seed=3, scale=0.5)
    out = lib.rmsnorm(x, w, 1e-5)
    expected = ref.rmsnorm(x.float(), w.float(), 1e-5)
    assert (out.float() - expected).abs().max() < 2e-2


def test_fused_add_rmsnorm(lib):
    from fei_amd.ops import reference as ref
    x = randbf(8, 4096, seed=4)
    res = randbf(8, 4096, seed=5)
    w = randbf(4096, seed=6, scale=0.5)
    res_gpu = res.clone()
    out, new_res = lib.fused_add_rmsnorm(x, res_gpu, w, 1e-5)
    exp_out, exp_res = ref.fused_add_rmsnorm(x, res.clone(), w, 1e-5)
    assert (new_res.float() - exp_res.float()).abs().max() < 2e-2
    assert (out.float() - exp_out.float()).abs().max() < 2e-2


def _mk_cache(B, Hkv, max_seq, D, seed=0):
    return randbf(B, Hkv, max_seq, D, seed=seed)


def test_rope_kv_decode(lib):
    from fei_amd.ops import reference as ref
    B, Hq, Hkv, D, MS = 2, 8, 2, 128, 64
    q = randbf(B, Hq, D, seed=7)
    k = randbf(B, Hkv, D, seed=8)
    v = randbf(B, Hkv, D, seed=9)
    kc = torch.zeros(B, Hkv, MS, D, device=DEV, dtype=torch.bfloat16)
    vc = torch.zeros_like(kc)
    pos = torch.tensor([3, 11], dtype=torch.int32, device=DEV)
    table = ref.rope_table(MS, D, device=DEV)

    kc_ref = torch.zeros_like(kc)
    vc_ref = torch.zeros_like(vc)
    q_ref = ref.rope_kv_decode(q.clone(), k, v, kc_ref, vc_ref, pos, table)

    q_gpu = q.clone()
    lib.rope_kv_decode(q_gpu, k, v, kc, vc, pos, table)
    assert (q_gpu.float() - q_ref.float()).abs().max() < 2e-2
    assert (kc.float() - kc_ref.float()).abs().max() < 2e-2
    assert torch.equal(vc, vc_ref)


def test_rope_kv_prefill_strided(lib):
    """Exercise the strided-q path: q/k/v as views into a fused qkv buffer."""
    from fei_amd.ops import reference as ref
    B, S, Hq, Hkv, D, MS = 2, 9, 4, 2, 128, 64
    W = (Hq + 2 * Hkv) * D
    qkv = randbf(B * S, W, seed=10)
    q = qkv.as_strided((B, S, Hq, D), (S * W, W, D, 1))
    k = qkv.as_strided((B, S, Hkv, D), (S * W, W, D, 1), storage_offset=Hq * D)
    v = qkv.as_strided((B, S, Hkv, D), (S * W, W, D, 1), storage_offset=(Hq + Hkv) * D)
    kc = torch.zeros(B, Hkv, MS, D, device=DEV, dtype=torch.bfloat16)
    vc = torch.zeros_like(kc)
    pos0 = torch.tensor([0, 5], dtype=torch.int32, device=DEV)
    table = ref.rope_table(MS, D, device=DEV)

    kc_ref = torch.zeros_like(kc)
    vc_ref = torch.zeros_like(vc)
    q_ref = ref.rope_kv_prefill(q.contiguous().clone(), k.contiguous(),
                                v.contiguous(), kc_ref, vc_ref, pos0, table)

    lib.rope_kv_prefill(q, k, v, kc, vc, pos0, table)
    assert (q.float() - q_ref.float()).abs().max() < 2e-2
    assert (kc.float() - kc_ref.float()).abs().max() < 2e-2
    assert torch.equal(vc, vc_ref)


@pytest.mark.parametrize("n,splits", [(1, 1), (7, 4), (300, 16), (1000, 16), (20, 32), (1000, 32)])
def test_attn_decode(lib, n, splits):
    from fei_amd.ops import reference as ref
    B, Hq, Hkv, D, MS = 2, 8, 2, 128, 1024
    q = randbf(B, Hq, D, seed=20 + n)
    kc = _mk_cache(B, Hkv, MS, D, seed=21 + n)
    vc = _mk_cache(B, Hkv, MS, D, seed=22 + n)
    pos = torch.tensor([n - 1, max(n // 2 - 1, 0)], dtype=torch.int32, device=DEV)
    out = lib.attn_decode(q, kc, vc, pos, splits=splits)
    expected = ref.attn_decode(q, kc, vc, pos + 1)
    err = (out.float() - expected.float()).abs().max().item()
    assert err < 2e-2, f"max err {err}"


@pytest.mark.parametrize("n,splits", [(2100, 32), (8100, 32), (2100, 16),
                                      (4100, 64)])
def test_attn_decode_long_context(lib, n, splits):
    """More keys than the splits' waves take in one round, beside a sequence
    of a third of them in the same launch."""
    from fei_amd.ops import reference as ref
    B, Hq, Hkv, D, MS = 2, 8, 2, 128, 8192
    q = randbf(B, Hq, D, seed=70 + n)
    kc = _mk_cache(B, Hkv, MS, D, seed=71 + n)
    vc = _mk_cache(B, Hkv, MS, D, seed=72 + n)
    pos = torch.tensor([n - 1, n // 3], dtype=torch.int32, device=DEV)
    out = lib.attn_decode(q, kc, vc, pos, splits=splits)
    expected = ref.attn_decode(q, kc, vc, pos + 1)
    err = (out.float() - expected.float()).abs().max().item()
    assert err < 2e-2, f"max err {err}"


@pytest.mark.parametrize("n,splits", [(1, 1), (7, 4), (300, 16), (1000, 32),
                                      (20, 32)])
def test_attn_decode_workspace(lib, n, splits):
    """A workspace may hold anything (here NaN, then another call's sums): what
    a call did not write it does not read. More entries than two, and a layer,
    are taken and make no difference; nor does a workspace of the call's own."""
    from fei_amd.ops import reference as ref
    B, Hq, Hkv, D, MS = 2, 8, 2, 128, 1024
    q = randbf(B, Hq, D, seed=50 + n)
    kc = _mk_cache(B, Hkv, MS, D, seed=51 + n)
    vc = _mk_cache(B, Hkv, MS, D, seed=52 + n)
    pos = torch.tensor([n - 1, max(n // 2 - 1, 0)], dtype=torch.int32,
                       device=DEV)
    ws = (torch.full((B, Hq, splits, D), float("nan"), device=DEV),
          torch.full((B, Hq, splits, 2), float("nan"), device=DEV),
          torch.zeros(B * Hkv * splits, dtype=torch.int32, device=DEV))
    expected = ref.attn_decode(q, kc, vc, pos + 1)
    own = lib.attn_decode(q, kc, vc, pos, splits=splits)
    assert (own.float() - expected.float()).abs().max() < 2e-2
    full = torch.full_like(pos, MS - 1)
    for at in (pos, full, pos):
        got = lib.attn_decode(q, kc, vc, at, splits=splits, workspace=ws,
                              layer=3)
        if at is pos:
            assert torch.equal(got, own)
    assert torch.equal(own, lib.attn_decode(q, kc, vc, pos, splits=splits,
                                            workspace=ws[:2]))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S,p0", [(16, 0), (64, 0), (129, 0), (64, 37)])
def test_attn_prefill_causal(lib, D, S, p0):
    from fei_amd.ops import reference as ref
    B, Hq, Hkv, MS = 2, 4, 2, 512
    q = randbf(B, S, Hq, D, seed=30 + S + D)
    kc = _mk_cache(B, Hkv, MS, D, seed=31 + S)
    vc = _mk_cache(B, Hkv, MS, D, seed=32 + S)
    pos0 = torch.tensor([p0, p0], dtype=torch.int32, device=DEV)
    out = lib.attn_prefill(q, kc, vc, pos0)
    expected = ref.attn_prefill(q, kc, vc, pos0)
    err = (out.float() - expected.float()).abs().max().item()
    assert err < 2e-2, f"max err {err}"


def test_attn_prefill_spiked_scores(lib):
    """Force large max jumps across KV tiles (rule 26: exercise the rescale
    path of the online softmax with an input that forces it)."""
    from fei_amd.ops import reference as ref
    B, S, Hq, Hkv, D, MS = 1, 64, 2, 1, 128, 256
    q = randbf(B, S, Hq, D, seed=40)
    kc = _mk_cache(B, Hkv, MS, D, seed=41, )
    vc = _mk_cache(B, Hkv, MS, D, seed=42)
    # spike one late key so every row's max jumps at the last tile
    kc[:, :, 60, :] = (q[0, :, 0, :].mean(0) * 8).to(torch.bfloat16)
    pos0 = torch.zeros(B, dtype=torch.int32, device=DEV)
    out = lib.attn_prefill(q, kc, vc, pos0)
    expected = ref.attn_prefill(q, kc, vc, pos0)
    err = (out.float() - expected.float()).abs().max().item()
    assert err < 3e-2, f"max err {err}"


def test_attn_prefill_bidirectional(lib):
    from fei_amd.ops import reference as ref
    B, S, Hq, Hkv, D, MS = 1, 33, 4, 4, 64, 128
    q = randbf(B, S, Hq, D, seed=50)
    kc = _mk_cache(B, Hkv, MS, D, seed=51)
    vc = _mk_cache(B, Hkv, MS, D, seed=52)
    pos0 = torch.zeros(B, dtype=torch.int32, device=DEV)
    kv_len = torch.tensor([S], dtype=torch.int32, device=DEV)
    out = lib.attn_prefill(q, kc, vc, pos0, causal=False, kv_len=kv_len)
    expected = lib._ref_bidir(q, kc, vc, kv_len, 1.0 / math.sqrt(D))
    err = (out.float() - expected.float()).abs().max().item()
    assert err < 2e-2, f"max err {err}"


def test_swiglu(lib):
    from fei_amd.ops import reference as ref
    gu = randbf(17, 2 * 14336, seed=60)
    out = lib.swiglu(gu)
    expected = ref.swiglu(gu)
    assert (out.float() - expected.float()).abs().max() < 1e-2


def test_sample_greedy(lib):
    B, V = 2, 128256
    g = torch.Generator(device=DEV).manual_seed(70)
    logits = (torch.randn(B, V, generator=g, device=DEV)).to(torch.bfloat16)
    token = torch.zeros(B, dtype=torch.int32, device=DEV)
    step = torch.zeros(1, dtype=torch.int32, device=DEV)
    out_tokens = torch.zeros(B, 8, dtype=torch.int32, device=DEV)
    ws = torch.zeros(B, 64 * 2, dtype=torch.float32, device=DEV)
    lib.sample(logits, token, step, ws, out_tokens=out_tokens, temperature=0.0)
    expected = logits.float().argmax(dim=-1)
    assert torch.equal(token.long(), expected)
    assert torch.equal(out_tokens[:, 0].long(), expected)


def test_sample_gumbel_prefers_peak(lib):
    B, V = 1, 1024
    logits = torch.full((B, V), -10.0, device=DEV).to(torch.bfloat16)
    logits[0, 123] = 10.0
    token = torch.zeros(B, dtype=torch.int32, device=DEV)
    step = torch.zeros(1, dtype=torch.int32, device=DEV)
    ws = torch.zeros(B, 64 * 2, dtype=torch.float32, device=DEV)
    hits = 0
    for s in range(20):
        step.fill_(s)
        lib.sample(logits, token, step, ws, temperature=1.0, seed=s)
        if int(token[0]) == 123:
            hits += 1
    assert hits >= 19   # peak is ~20 logits above the rest


def test_sample_gumbel_varies_with_step(lib):
    B, V = 1, 512
    g = torch.Generator(device=DEV).manual_seed(71)
    logits = torch.randn(B, V, generator=g, device=DEV).to(torch.bfloat16)
    token = torch.zeros(B, dtype=torch.int32, device=DEV)
    step = torch.zeros(1, dtype=torch.int32, device=DEV)
    ws = torch.zeros(B, 64 * 2, dtype=torch.float32, device=DEV)
    seen = set()
    for s in range(16):
        step.fill_(s)
        lib.sample(logits, token, step, ws, temperature=2.0, seed=1)
        seen.add(int(token[0]))
    assert len(seen) > 3    # high temperature must explore


def test_advance(lib):
    pos = torch.tensor([5, 9], dtype=torch.int32, device=DEV)
    step = torch.zeros(1, dtype=torch.int32, device=DEV)
    lib.advance(pos, step)
    assert pos.tolist() == [6, 10]
    assert int(step) == 1


def test_gemv_matches_linear(lib):
    import torch.nn.functional as F
    # 2 to 32 rows run in the matrix-core tile (k_skinny), one in the streaming
    # kernel (k_gemv)
    for M, N, K in [(1, 4096, 4096), (1, 6144, 4096), (2, 512, 1024),
                    (4, 128256, 4096), (8, 4096, 4096), (8, 6144, 4096),
                    (8, 4096, 14336), (5, 1024, 2048), (8, 120, 4096),
                    (8, 4096, 1536), (12, 4096, 4096), (16, 4096, 4096),
                    (4, 1024, 8192), (8, 2048, 8192)]:
        x = randbf(M, K, seed=80 + M)
        w = randbf(N, K, seed=81 + N % 97, scale=0.02)
        out = lib.linear_decode(x, w)
        ref_out = F.linear(x.float(), w.float())
        err = (out.float() - ref_out).abs().max().item()
        tol = 0.02 * max(1.0, K / 4096)
        assert err < tol, f"M{M} N{N} K{K}: max err {err}"


@pytest.mark.parametrize("M", [1, 8])
def test_gemv_swiglu_matches(lib, M):
    import torch.nn.functional as F
    from fei_amd.ops import reference as ref
    I, K = 14336, 4096
    x = randbf(M, K, seed=90)
    wgu = randbf(2 * I, K, seed=91, scale=0.02)
    out = lib.gemv_swiglu(x, wgu)
    # the kernel keeps gate/up dots in f32 through silu; compare against the
    # unrounded f32 reference (bf16-rounding g first shifts silu(g)*u by more
    # than the kernel's true error)
    gu32 = F.linear(x.float(), wgu.float())
    g, u = gu32[..., :I], gu32[..., I:]
    expected = torch.nn.functional.silu(g) * u
    # relative tolerance: outputs reach |8|, where one bf16 ulp is ~0.03
    err = ((out.float() - expected).abs() / (1 + expected.abs())).max().item()
    assert err < 2e-2, f"max rel err {err}"


@pytest.mark.parametrize("n", [1, 63, 640])
def test_attn_decode_fused(lib, n):
    """Fused rope+append+attention vs the reference pipeline."""
    from fei_amd.ops import reference as ref
    B, Hq, Hkv, D, MS = 2, 8, 2, 128, 1024
    W = (Hq + 2 * Hkv) * D
    qkv = randbf(B, W, seed=100 + n, scale=0.5)
    q = qkv.as_strided((B, Hq, D), (W, D, 1))
    k = qkv.as_strided((B, Hkv, D), (W, D, 1), storage_offset=Hq * D)
    v = qkv.as_strided((B, Hkv, D), (W, D, 1), storage_offset=(Hq + Hkv) * D)
    kc = _mk_cache(B, Hkv, MS, D, seed=101 + n)
    vc = _mk_cache(B, Hkv, MS, D, seed=102 + n)
    pos = torch.tensor([n - 1, max(n // 2 - 1, 0)], dtype=torch.int32, device=DEV)
    table = ref.rope_table(MS, D, device=DEV)

    kc_ref, vc_ref = kc.clone(), vc.clone()
    q_ref = ref.rope_kv_decode(q.contiguous().clone(), k.contiguous(),
                               v.contiguous(), kc_ref, vc_ref, pos, table)
    expected = ref.attn_decode(q_ref, kc_ref, vc_ref, pos + 1)

    out = lib.attn_decode_fused(q, k, v, kc, vc, pos, table)
    err = (out.float() - expected.float()).abs().max().item()
    assert err < 2e-2, f"n={n}: max err {err}"
    # cache rows written identically
    assert (kc.float() - kc_ref.float()).abs().max() < 2e-2
    assert torch.equal(vc, vc_ref)


def test_sample_onepass_greedy(lib):
    B, V = 2, 128256
    g = torch.Generator(device=DEV).manual_seed(170)
    logits = torch.randn(B, V, generator=g, device=DEV).to(torch.bfloat16)
    token = torch.zeros(B, dtype=torch.int32, device=DEV)
    step = torch.zeros(1, dtype=torch.int32, device=DEV)
    out_tokens = torch.zeros(B, 8, dtype=torch.int32, device=DEV)
    ws = torch.zeros(B, 64 * 2, dtype=torch.float32, device=DEV)
    lib.sample(logits, token, step, ws, out_tokens=out_tokens, temperature=0.0)
    expected = logits.float().argmax(dim=-1)
    assert torch.equal(token.long(), expected)
    assert torch.equal(out_tokens[:, 0].long(), expected)


@pytest.mark.parametrize("n,splits", [(1, 4), (70, 4), (640, 4), (300, 16), (40, 32), (1000, 32)])
def test_attn_decode_rope_fused_split(lib, n, splits):
    """Split-K attention with in-kernel RoPE+append vs the reference
    pipeline (covers owner-split cache writes and LDS new-key path)."""
    from fei_amd.ops import reference as ref
    B, Hq, Hkv, D, MS = 2, 8, 2, 128, 1024
    W = (Hq + 2 * Hkv) * D
    qkv = randbf(B, W, seed=200 + n, scale=0.5)
    q = qkv.as_strided((B, Hq, D), (W, D, 1))
    k = qkv.as_strided((B, Hkv, D), (W, D, 1), storage_offset=Hq * D)
    v = qkv.as_strided((B, Hkv, D), (W, D, 1), storage_offset=(Hq + Hkv) * D)
    kc = _mk_cache(B, Hkv, MS, D, seed=201 + n)
    vc = _mk_cache(B, Hkv, MS, D, seed=202 + n)
    pos = torch.tensor([n - 1, max(n // 2 - 1, 0)], dtype=torch.int32, device=DEV)
    table = ref.rope_table(MS, D, device=DEV)

    kc_ref, vc_ref = kc.clone(), vc.clone()
    q_ref = ref.rope_kv_decode(q.contiguous().clone(), k.contiguous(),
                               v.contiguous(), kc_ref, vc_ref, pos, table)
    expected = ref.attn_decode(q_ref, kc_ref, vc_ref, pos + 1)

    out = lib.attn_decode(q, kc, vc, pos, splits=splits, k=k, v=v, table=table)
    err = (out.float() - expected.float()).abs().max().item()
    assert err < 2e-2, f"n={n} splits={splits}: max err {err}"
    assert (kc.float() - kc_ref.float()).abs().max() < 2e-2
    assert torch.equal(vc, vc_ref)


def test_gemv_res_matches(lib):
    import torch.nn.functional as F
    M, N, K = 1, 4096, 4096
    x = randbf(M, K, seed=300)
    w = randbf(N, K, seed=301, scale=0.02)
    res = randbf(M, N, seed=302)
    expected = (res.float() + F.linear(x.float(), w.float())).to(torch.bfloat16)
    lib.gemv_res(x, w, res)
    err = ((res.float() - expected.float()).abs() /
           (1 + expected.float().abs())).max().item()
    assert err < 2e-2, f"max rel err {err}"


def test_gemv_norm_matches(lib):
    M, N, K = 1, 6144, 4096
    res = randbf(M, K, seed=310)
    wn = randbf(K, seed=311, scale=0.5)
    w = randbf(N, K, seed=312, scale=0.02)
    out = lib.gemv_norm(res, wn, w, 1e-5)
    x = lib.rmsnorm(res, wn, 1e-5)
    expected = lib.linear_decode(x, w)
    err = ((out.float() - expected.float()).abs() /
           (1 + expected.float().abs())).max().item()
    assert err < 2e-2, f"max rel err {err}"


def test_gemv_swiglu_norm_matches(lib):
    M, I, K = 1, 14336, 4096
    res = randbf(M, K, seed=320)
    wn = randbf(K, seed=321, scale=0.5)
    wgu = randbf(2 * I, K, seed=322, scale=0.02)
    out = lib.gemv_swiglu_norm(res, wn, wgu, 1e-5)
    x = lib.rmsnorm(res, wn, 1e-5)
    expected = lib.gemv_swiglu(x, wgu)
    err = ((out.float() - expected.float()).abs() /
           (1 + expected.float().abs())).max().item()
    assert err < 2e-2, f"max rel err {err}"


@pytest.mark.parametrize("n", [5, 100, 500, 1000])
def test_attn_decode_paged(lib, n):
    """Paged attention over a scrambled block table == contiguous reference.
    n=500/1000 at splits=4 -> chunk >= 125 exercises the WIDE V lane map;
    the short n cases take the pair map."""
    from fei_amd.ops import reference as ref
    B, Hq, Hkv, D, BS = 2, 8, 2, 128, 16
    max_blocks = 64
    n_phys = 256
    g = torch.Generator(device=DEV).manual_seed(400 + n)
    k_pool = (torch.randn(n_phys, Hkv, BS, D, generator=g, device=DEV)).to(torch.bfloat16)
    v_pool = (torch.randn(n_phys, Hkv, BS, D, generator=g, device=DEV)).to(torch.bfloat16)
    # scrambled, non-overlapping physical blocks per sequence
    perm = torch.randperm(n_phys, generator=g, device=DEV)[: B * max_blocks]
    bt = perm.view(B, max_blocks).to(torch.int32)
    q = randbf(B, Hq, D, seed=401 + n)
    pos = torch.tensor([n - 1, max(n // 2 - 1, 0)], dtype=torch.int32, device=DEV)

    out = lib.attn_decode_paged(q, k_pool, v_pool, bt, pos, splits=4)

    # contiguous gather reference
    max_len = max_blocks * BS
    kc = torch.zeros(B, Hkv, max_len, D, dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros_like(kc)
    for b in range(B):
        for j, blk in enumerate(bt[b].tolist()):
            kc[b, :, j * BS:(j + 1) * BS] = k_pool[blk]
            vc[b, :, j * BS:(j + 1) * BS] = v_pool[blk]
    expected = ref.attn_decode(q, kc, vc, pos + 1)
    err = (out.float() - expected.float()).abs().max().item()
    assert err < 2e-2, f"n={n}: max err {err}"


def test_layernorm_kernel(lib):
    from fei_amd.ops import reference as ref
    x = randbf(9, 768, seed=500)
    res = randbf(9, 768, seed=501)
    w = randbf(768, seed=502, scale=0.5)
    b = randbf(768, seed=503, scale=0.1)
    out = lib.layernorm(x, w, b, 1e-6)
    expected = ref.layernorm(x, w, b, 1e-6)
    assert (out.float() - expected.float()).abs().max() < 2e-2
    out = lib.layernorm(x, w, b, 1e-6, residual=res)
    expected = ref.layernorm(x, w, b, 1e-6, residual=res)
    assert (out.float() - expected.float()).abs().max() < 2e-2


def test_gelu_kernel(lib):
    from fei_amd.ops import reference as ref
    x = randbf(7, 3072, seed=510, scale=2.0)
    out = lib.gelu(x)
    expected = ref.gelu(x)
    assert (out.float() - expected.float()).abs().max() < 1e-2


def test_quant_fp8_matches_torch(lib):
    from fei_amd.ops import reference as ref
    w = randbf(64, 512, seed=600, scale=0.05)
    w8_gpu, sc_gpu = lib.quant_fp8(w)
    w8_ref, sc_ref = ref.quant_fp8(w.cpu())
    assert torch.allclose(sc_gpu.cpu(), sc_ref, rtol=1e-3)
    # decoded values must match the torch e4m3fn cast (RNE)
    deq_gpu = ref.dequant_fp8(w8_gpu.cpu(), sc_gpu.cpu())
    deq_ref = ref.dequant_fp8(w8_ref, sc_ref)
    mismatch = (deq_gpu != deq_ref).float().mean().item()
    assert mismatch < 0.01, f"{mismatch:.4f} of encodings differ"


def test_gemv_norm_fp8_matches_dequant(lib):
    from fei_amd.ops import reference as ref
    M, N, K = 1, 6144, 4096
    res = randbf(M, K, seed=610)
    wn = randbf(K, seed=611, scale=0.5)
    w = randbf(N, K, seed=612, scale=0.02)
    w8, sc = lib.quant_fp8(w)
    out = lib.gemv_norm_fp8(res, wn, w8, sc, 1e-5)
    wdq = ref.dequant_fp8(w8.cpu(), sc.cpu()).to(DEV).to(torch.bfloat16)
    expected = lib.gemv_norm(res, wn, wdq, 1e-5)
    err = ((out.float() - expected.float()).abs() /
           (1 + expected.float().abs())).max().item()
    assert err < 2e-2, f"max rel err {err}"


def test_gemv_res_fp8_matches_dequant(lib):
    from fei_amd.ops import reference as ref
    M, N, K = 1, 4096, 4096
    x = randbf(M, K, seed=620)
    w = randbf(N, K, seed=621, scale=0.02)
    res0 = randbf(M, N, seed=622)
    w8, sc = lib.quant_fp8(w)
    res_a = res0.clone()
    lib.gemv_res_fp8(x, w8, sc, res_a)
    wdq = ref.dequant_fp8(w8.cpu(), sc.cpu()).to(DEV).to(torch.bfloat16)
    res_b = res0.clone()
    lib.gemv_res(x, wdq, res_b)
    err = ((res_a.float() - res_b.float()).abs() /
           (1 + res_b.float().abs())).max().item()
    assert err < 2e-2, f"max rel err {err}"


def test_gemv_swiglu_norm_fp8_matches_dequant(lib):
    from fei_amd.ops import reference as ref
    M, I, K = 1, 14336, 4096
    res = randbf(M, K, seed=630)
    wn = randbf(K, seed=631, scale=0.5)
    wgu = randbf(2 * I, K, seed=632, scale=0.02)
    w8, sc = lib.quant_fp8(wgu)
    out = lib.gemv_swiglu_norm_fp8(res, wn, w8, sc, 1e-5)
    wdq = ref.dequant_fp8(w8.cpu(), sc.cpu()).to(DEV).to(torch.bfloat16)
    expected = lib.gemv_swiglu_norm(res, wn, wdq, 1e-5)
    err = ((out.float() - expected.float()).abs() /
           (1 + expected.float().abs())).max().item()
    assert err < 3e-2, f"max rel err {err}"


@pytest.mark.parametrize("M,K", [(1, 4096), (4, 4104), (8, 2056)])
def test_gemv_ssq_chain(lib, M, K):
    """gemv_res(ssq_out) -> gemv_norm/gemv_swiglu_norm(ssq): the sums of squares
    that the residual product adds up are those of the new rows, and the norm
    takes them. Several rows of a K that the matrix-core tile takes (a multiple
    of 64) make their norm without them."""
    N, I = 512, 1024
    x = randbf(M, K, seed=330)
    w = randbf(K, K, seed=331, scale=0.02)
    res = randbf(M, K, seed=332)
    wn = randbf(K, seed=333, scale=0.5)
    w2 = randbf(N, K, seed=334, scale=0.02)
    wgu = randbf(2 * I, K, seed=335, scale=0.02)
    assert lib._product(res, w2, M, K, N) == "gemv"

    want = res.double() + x.double() @ w.double().t()
    ssq = torch.zeros(M, dtype=torch.float32, device=res.device)
    lib.gemv_res(x, w, res, ssq_out=ssq)
    assert (res.double() - want).norm() < 2 ** -8 * want.norm()
    want_ssq = res.float().pow(2).sum(dim=-1)
    assert torch.allclose(ssq, want_ssq, rtol=1e-4), (ssq, want_ssq)

    y = res.double()
    y = y * (y.pow(2).mean(-1, keepdim=True) + 1e-5).rsqrt() * wn.double()
    # rows and results rounded once each; a SwiGLU's twice
    close = lambda a, b, tol: (a.double() - b).norm() < tol * b.norm()
    out = lib.gemv_norm(res, wn, w2, 1e-5, ssq=ssq)
    assert close(out, y @ w2.double().t(), 2 ** -7)
    # the sums it is given are the sums it uses
    half = lib.gemv_norm(res, wn, w2, 1e-5, ssq=4 * ssq)
    assert close(half, y @ w2.double().t() / 2, 2 ** -7)
    act = lib.gemv_swiglu_norm(res, wn, wgu, 1e-5, ssq=ssq)
    g, u = (y @ wgu.double().t()).split(I, 1)
    assert close(act, torch.nn.functional.silu(g) * u, 2 ** -6)


@pytest.mark.parametrize("n", [7, 100, 500, 1000])
def test_attn_decode_paged_rope_fused(lib, n):
    """Fused paged form (raw q/k/v + rope table; in-kernel RoPE + pool
    append) must equal roping torch-side, appending, then the plain
    paged kernel — the serving hot path (sessions._forward_paged)."""
    from fei_amd.ops import reference as ref
    B, Hq, Hkv, D, BS = 2, 8, 2, 128, 16
    max_blocks, n_phys = 64, 256
    g = torch.Generator(device=DEV).manual_seed(500 + n)
    k_pool = (torch.randn(n_phys, Hkv, BS, D, generator=g, device=DEV) * 0.3).to(torch.bfloat16)
    v_pool = (torch.randn(n_phys, Hkv, BS, D, generator=g, device=DEV) * 0.3).to(torch.bfloat16)
    k_pool2, v_pool2 = k_pool.clone(), v_pool.clone()
    perm = torch.randperm(n_phys, generator=g, device=DEV)[: B * max_blocks]
    bt = perm.view(B, max_blocks).to(torch.int32)
    q = randbf(B, Hq, D, seed=501 + n)
    k = randbf(B, Hkv, D, seed=502 + n)
    v = randbf(B, Hkv, D, seed=503 + n)
    pos = torch.tensor([n - 1, max(n // 2 - 1, 0)], dtype=torch.int32,
                       device=DEV)
    rope = ref.rope_table(2048, D, device=DEV)

    out_f = lib.attn_decode_paged(q.clone(), k_pool, v_pool, bt, pos,
                                  splits=4, k=k, v=v, table=rope)

    # torch-side rope + append, then the plain paged kernel
    q_r = ref.apply_rope(q.float(), pos.long(), rope).to(torch.bfloat16)
    k_r = ref.apply_rope(k.float(), pos.long(), rope).to(torch.bfloat16)
    for b in range(B):
        p = int(pos[b])
        blk = int(bt[b, p // BS])
        k_pool2[blk, :, p % BS, :] = k_r[b]
        v_pool2[blk, :, p % BS, :] = v[b]
    out_u = lib.attn_decode_paged(q_r.contiguous(), k_pool2, v_pool2, bt,
                                  pos, splits=4)
    assert (out_f.float() - out_u.float()).abs().max().item() < 2e-2
    # the appended pool rows must match too
    for b in range(B):
        p = int(pos[b])
        blk = int(bt[b, p // BS])
        dk = (k_pool[blk, :, p % BS].float()
              - k_pool2[blk, :, p % BS].float()).abs().max().item()
        dv = (v_pool[blk, :, p % BS].float()
              - v_pool2[blk, :, p % BS].float()).abs().max().item()
        assert dk < 2e-2 and dv == 0.0
