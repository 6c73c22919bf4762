// All layers of an encoder, launched from one call: over few rows its kernels take
// 4 to 10 us each, less than it takes to launch them one by one from Python.
#include "fei_epilogue.h"

extern "C" {

void fei_skinny(void* out, const void* x, const void* w, int M, int N, int K,
                int epi, const float* bias, float scale, float cap, int n_mix,
                int n_router, float* router, void* act, long as,
                const void* bias16, const void* gain, const float* sums,
                int tiles, float eps, float* sums_out, hipStream_t stream);
void fei_rows_bias(void* out, const void* x, const void* w, const void* bias,
                   int M, int N, int K, int gelu, hipStream_t stream);
void fei_attn_prefill(const void* q, const void* k_cache, const void* v_cache,
                      void* out, const int* pos0, const int* kv_len, int B,
                      int S, int Hq, int Hkv, int D, int max_seq, float scale,
                      int causal, long q_ts, int splits, float* po, float* pml,
                      long kv_b, long kv_h, long kv_t, hipStream_t stream);
void fei_add_layernorm(void* out, const void* x, const void* res,
                       const void* w, const void* b, int rows, int cols,
                       float eps, int has_res, hipStream_t stream);

// w: 12 a layer, in the order in which they are read below; h [B * S, C] is
// replaced by the layers' result; h1 and tmp as h, qkv [B * S, 3 H D],
// att [B * S, H D], inner [B * S, I]. What fei_skinny and fei_attn_prefill ask of
// their rows holds for all. splits, po, pml: see fei_attn_prefill.
void fei_encoder_layers(const void* const* w, int layers, void* h, void* h1,
                        void* tmp, void* qkv, void* att, void* inner,
                        const int* pos0, const int* kv_len, int B, int S, int H,
                        int D, int C, int I, float scale, float eps,
                        int splits, float* po, float* pml,
                        hipStream_t stream) {
  const int M = B * S, HD = H * D;
  auto product = [&](void* out, const void* x, const void* const* wb, int N,
                     int K, int epi) {
    // K shared by the waves of a block, or tiles of 64 rows: 12 layers of 768,
    // 40 rows 512 us and 788, 64 rows 571 and 800
    if (M > 64)
      return fei_rows_bias(out, x, wb[0], wb[1], M, N, K, epi == EPI_GELU,
                           stream);
    fei_skinny(out, x, wb[0], M, N, K, epi, nullptr, 1.f, 0.f, 0, 0, nullptr,
               nullptr, 0, wb[1], nullptr, nullptr, 0, 0.f, nullptr, stream);
  };
  for (int l = 0; l < layers; ++l, w += 12) {
    product(qkv, h, w, 3 * HD, C, EPI_BF16);
    fei_attn_prefill(qkv, (u16*)qkv + HD, (u16*)qkv + 2 * HD, att, pos0, kv_len,
                     B, S, H, H, D, S, scale, 0, 3L * HD, splits, po, pml,
                     3L * S * HD, D, 3L * HD, stream);
    product(tmp, att, w + 2, C, HD, EPI_BF16);
    fei_add_layernorm(h1, tmp, h, w[4], w[5], M, C, eps, 1, stream);
    product(inner, h1, w + 6, I, C, EPI_GELU);
    product(tmp, inner, w + 8, C, I, EPI_BF16);
    fei_add_layernorm(h, tmp, h1, w[10], w[11], M, C, eps, 1, stream);
  }
}

}  // extern "C"
