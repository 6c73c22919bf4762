"""What csrc/decode_one.hip and csrc/encoder_one.hip compute, in float64 with plain torch,
rounded to bfloat16 where they hand bfloat16 on: only the order of sums is left to differ."""

import math

import torch


def bf(x):
    return x.to(torch.bfloat16).double()


def rms(x, gain, eps):
    return bf(x * (x.square().mean() + eps).rsqrt() * gain.double())


def step(m, h, pos, k, v, fp8=False, keep=None):
    """A decoding step of one row h [1, C] at ``pos``, caches [layers, 1, Hkv, room, D]:
    logits [vocab], and the rows that go into the caches [layers, Hkv, D]. ``keep``: which
    of the keys in front of the new one are looked at."""
    s, D = m.spec, m.D
    last = min(pos, k.shape[3] - 1)
    keep = slice(0, last) if keep is None else keep
    x, rows = h[0].double(), ([], [])
    cos, sin = m.rope[last].double().unbind(-1)

    def rope(t):
        a, b = t[:, :D // 2], t[:, D // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], 1)

    def product(y, w, pair):
        if not fp8:
            return w.double() @ y
        w, scale = pair
        return w.view(torch.float8_e4m3fn).double() @ y * scale.double()
    for i, lw in enumerate(m.layers):
        q8 = m.fp8[i] if fp8 else dict.fromkeys(("wqkv", "wo", "wgu", "wdown"))
        qkv = bf(product(rms(x, lw.norm_attn, s.norm_eps), lw.wqkv, q8["wqkv"]))
        q, kn, vn = qkv.view(-1, D).split([m.hq_l, m.hkv_l, m.hkv_l])
        q, kn = rope(q), bf(rope(kn))
        att = []
        for j in range(m.hkv_l):
            keys, values = (torch.cat([c[i, 0, j, keep].double(), t[j:j + 1]])
                            for c, t in ((k, kn), (v, vn)))
            mine = q[j * (m.hq_l // m.hkv_l):(j + 1) * (m.hq_l // m.hkv_l)]
            att.append(torch.softmax(mine @ keys.T / math.sqrt(D), 1) @ values)
        x = bf(x + product(bf(torch.cat(att).view(-1)), lw.wo, q8["wo"]))
        gate, up = product(rms(x, lw.norm_mlp, s.norm_eps), lw.wgu, q8["wgu"]).chunk(2)
        act = bf(gate / (1 + torch.exp(-gate)) * up)
        x = bf(x + product(act, lw.wdown, q8["wdown"]))
        rows[0].append(kn)
        rows[1].append(vn)
    head = product(rms(x, m.norm_f, s.norm_eps), m.lm_head, m.fp8_lm_head if fp8 else None)
    return bf(head), torch.stack(rows[0]), torch.stack(rows[1])


def layernorm(x, gain, shift, eps):
    x = x - x.mean(-1, keepdim=True)
    inv = (x.square().mean(-1, keepdim=True) + eps).rsqrt()
    return bf(x * inv * gain.double() + shift.double())


def encoder(m, h, lens):
    """Embeddings [B, C] of the normed rows h [B, S, C]."""
    B, S, C = h.shape
    H, D = m.spec.num_heads, m.spec.head_dim
    h = h.double().reshape(B * S, C)
    n = [min(max(int(i), 0), S) for i in lens]

    def product(x, lw, name):
        return x @ lw["w" + name].double().T + lw["b" + name].double()
    for lw in m.layers:
        qkv = bf(product(h, lw, "qkv")).view(B, S, 3, H, D)
        att = torch.zeros(B, S, H, D, dtype=torch.float64, device=h.device)
        for b in range(B):
            for j in range(H if n[b] else 0):
                q, key, value = qkv[b, :, :, j].unbind(1)
                t = q @ key[:n[b]].T / math.sqrt(D)
                p = torch.exp(t - t.amax(1, keepdim=True))
                att[b, :, j] = bf(p) @ value[:n[b]] / p.sum(1, keepdim=True)
        mid = product(bf(att.view(B * S, H * D)), lw, "o")
        h = layernorm(h + mid, lw["ln1_w"], lw["ln1_b"], m.eps)
        t = product(h, lw, "i")
        t = bf(t * 0.5 * torch.erfc(-t / math.sqrt(2)))
        h = layernorm(h + product(t, lw, "o2"), lw["ln2_w"], lw["ln2_b"], m.eps)
    out = torch.stack([h.view(B, S, C)[b, :n[b]].sum(0) / max(n[b], 1) for b in range(B)])
    return out / out.norm(dim=1, keepdim=True).clamp_min(1e-12)
