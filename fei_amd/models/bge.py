"""Embedding encoder for memdir semantic search — bge-base architecture
(BERT-style: 12 layers, 768 hidden, 12 heads, post-LayerNorm residual
blocks, GELU MLP, biased linears).

Up to 128 rows take one launch (ops.encoder_one). Where lengths are given, of more than 640
rows only those that texts have are run (ops.encoder_packed): padding is left out on the
device. Else, up to 1024 rows, all layers are launched from one call (ops.encoder_layers).
All have their products in this library's matrix-core tiles; those of more rows without
lengths are the BLAS library's (GELU's own). Bidirectional attention runs in the HIP prompt kernel (causal=0),
LayerNorm with the residual and GELU in HIP kernels. Weights are random-init — there is no
network for checkpoints — but the architecture matches bge-base so real weights could be
loaded via the same tensors.

Output: mean-pooled last hidden state, L2-normalised — [B, hidden].
"""

from __future__ import annotations

import math
from typing import List, Optional

import torch

from fei_amd import ops
from fei_amd.engine.config import ModelSpec, get_spec

# a layer's tensors in the order in which they are used
NAMES = ("wqkv", "bqkv", "wo", "bo", "ln1_w", "ln1_b", "wi", "bi", "wo2", "bo2",
         "ln2_w", "ln2_b")


class BgeEncoder:
    # Up to 128 rows in one launch, which keeps all CUs while it runs: two encoders on
    # two streams take 239 us each of 24 tokens, 216 without. Not for those who
    # run much side by side
    one_launch = True

    def __init__(self, spec: Optional[ModelSpec] = None,
                 device: Optional[torch.device] = None,
                 dtype: Optional[torch.dtype] = None, seed: int = 42,
                 max_seq_len: int = 512):
        self.spec = spec or get_spec("bge-base")
        if device is None:
            device = torch.device("cuda:0") if torch.cuda.is_available() else torch.device("cpu")
        self.device = device
        if dtype is None:
            dtype = torch.bfloat16 if device.type == "cuda" else torch.float32
        self.dtype = dtype
        self.max_seq_len = min(max_seq_len, self.spec.max_seq_len)
        self.eps = 1e-12 if device.type == "cpu" else 1e-6   # BERT uses 1e-12
        self._init_weights(seed)

    def _init_weights(self, seed: int) -> None:
        s = self.spec
        # CPU generator: identical weights on every device for the same seed
        # (the encoder is small; cross-device reproducibility matters for
        # the GPU-vs-CPU numerics test and shared federation indexes)
        g = torch.Generator().manual_seed(seed)
        C, I = s.hidden_size, s.intermediate_size
        sc = 1.0 / math.sqrt(C)

        def rand(*shape, scale):
            w = torch.randn(*shape, generator=g, dtype=torch.float32) * scale
            return w.to(device=self.device, dtype=self.dtype)

        def zeros(*shape):
            return torch.zeros(*shape, device=self.device, dtype=self.dtype)

        def ones(*shape):
            return torch.ones(*shape, device=self.device, dtype=self.dtype)

        self.tok_emb = rand(s.vocab_size, C, scale=0.02)
        self.pos_emb = rand(self.max_seq_len, C, scale=0.02)
        self.emb_ln_w, self.emb_ln_b = ones(C), zeros(C)
        self.layers = []
        for _ in range(s.num_layers):
            self.layers.append({
                "wqkv": rand(3 * s.num_heads * s.head_dim, C, scale=sc),
                "bqkv": zeros(3 * s.num_heads * s.head_dim),
                "wo": rand(C, s.num_heads * s.head_dim, scale=sc),
                "bo": zeros(C),
                "ln1_w": ones(C), "ln1_b": zeros(C),
                "wi": rand(I, C, scale=sc),
                "bi": zeros(I),
                "wo2": rand(C, I, scale=1.0 / math.sqrt(I)),
                "bo2": zeros(C),
                "ln2_w": ones(C), "ln2_b": zeros(C),
            })

    @torch.no_grad()
    def encode_ids(self, token_ids: torch.Tensor,
                   lengths: Optional[torch.Tensor] = None) -> torch.Tensor:
        """token_ids [B, S] -> embeddings [B, C] (fp32, L2-normalised).
        BERT block: h = LN(h + Attn(h)); h = LN(h + GELU(h Wi + bi) Wo2 + bo2)."""
        return self._encode(token_ids, lengths, lengths is not None)

    def _encode(self, token_ids: torch.Tensor, lengths: Optional[torch.Tensor],
                pack: bool) -> torch.Tensor:
        """``pack``: whether padding may be left out."""
        s = self.spec
        B, S = token_ids.shape
        H, D = s.num_heads, s.head_dim
        embed = (token_ids.long().contiguous(), self.tok_emb, self.pos_emb,
                 self.emb_ln_w, self.emb_ln_b)
        kv_len = (lengths.to(torch.int32) if lengths is not None
                  else torch.full((B,), S, dtype=torch.int32, device=self.device))
        weights = [lw[n] for lw in self.layers for n in NAMES]
        # of one and two layers the one launch's start costs more than their seams:
        # captured, us, the chain's first, one layer of 768 and 8 rows 40, 40, 128 64,
        # 73, two of 128 and 64 rows 64, 62, 100 75, 83; four of 256 and 128 140, 137
        if self.one_launch and (len(self.layers) > 2 or B * S <= 32 * len(self.layers)):
            out = ops.encoder_one(*embed, weights, H, D, s.intermediate_size, kv_len,
                                  self.eps)
            if out is not None:
                return out
        if pack:
            out = ops.encoder_packed(*embed, weights, H, D, s.intermediate_size,
                                     kv_len, self.eps)
            if out is not None:
                return out
        h = ops.embed_layernorm(*embed, self.eps, self.dtype)
        pos0 = kv_len                  # of causal attention alone
        few = ops.encoder_layers(h, weights, H, D, s.intermediate_size, pos0,
                                 kv_len, self.eps)
        h = few if few is not None else self._layers(h, pos0, kv_len)
        return ops.pool_unit(h, kv_len)

    def _layers(self, h: torch.Tensor, pos0: torch.Tensor,
                kv_len: torch.Tensor) -> torch.Tensor:
        B, S = h.shape[:2]
        H, D = self.spec.num_heads, self.spec.head_dim
        scale = 1.0 / math.sqrt(D)
        for lw in self.layers:
            qkv = ops.linear_bias(h, lw["wqkv"], lw["bqkv"]) \
                .view(B, S, 3, H, D)
            # the attention reads queries, keys and values where they are
            q, k, v = qkv.unbind(2)
            att = ops.attn_prefill(q, k.transpose(1, 2), v.transpose(1, 2),
                                   pos0, scale=scale, causal=False,
                                   kv_len=kv_len)
            o = ops.linear_bias(att.reshape(B, S, H * D), lw["wo"], lw["bo"])
            h = ops.layernorm(o, lw["ln1_w"], lw["ln1_b"], self.eps,
                              residual=h)
            inner = ops.linear_bias(h, lw["wi"], lw["bi"], act_gelu=True)
            o2 = ops.linear_bias(inner, lw["wo2"], lw["bo2"])
            h = ops.layernorm(o2, lw["ln2_w"], lw["ln2_b"], self.eps,
                              residual=h)
        return h

    @torch.no_grad()
    def encode_texts(self, texts: List[str], tokenizer=None,
                     batch_size: int = 64) -> torch.Tensor:
        """Convenience: byte-tokenize + pad + encode in batches."""
        from fei_amd.engine.tokenizer import ByteTokenizer
        tok = tokenizer or ByteTokenizer()
        out = []
        for i in range(0, len(texts), batch_size):
            chunk = texts[i:i + batch_size]
            ids = [tok.encode(t)[: self.max_seq_len] for t in chunk]
            n = [len(x) for x in ids]
            lens = torch.tensor(n, device=self.device)
            S = max(*n, 1)
            padded = torch.full((len(ids), S), tok.pad_id, dtype=torch.long,
                                device=self.device)
            for j, row in enumerate(ids):
                padded[j, :len(row)] = torch.tensor(row, device=self.device)
            pack = ops.encoder_packing_pays(padded.numel(), sum(n),
                                            self.spec.intermediate_size)
            out.append(self._encode(padded, lens, pack))
        return torch.cat(out, dim=0)
