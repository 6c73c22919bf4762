// A layer of a Llama-style decoder over few rows, launched from one call. Its kernels
// take 4 to 15 us each over few rows of a small model, and a launch from Python, with
// what is looked at before it, 10: 4 sessions, 16 layers of 2048, spent 840 of a step's
// 976 us on 80 of them. From here one takes under 2: steps of 2, 4 and 8 sessions of 40
// to 600 keys 916 -> 753 us, 925 -> 765, 934 -> 833 (the GPU's own time is what is left
// from 8 on: 20 and 32 as before), prompts of 2 tokens 1040 -> 726, of 7 behind 300 1027
// -> 787, of 20 1037 -> 861.
#include "fei_epilogue.h"

extern "C" {

void fei_gemv(void* out, const void* x, const void* gain, const void* w,
              const float* wscale, int M, int N, int K, float eps, int epi,
              float* ssq, hipStream_t stream);
void fei_skinny(void* out, const void* x, const void* w, int M, int N, int K,
                int epi, const float* bias, float scale, float cap, int n_mix,
                int n_router, float* router, void* act, long as,
                const void* bias16, const void* gain, const float* sums,
                int tiles, float eps, float* sums_out, hipStream_t stream);
void fei_rmsnorm(void* out, const void* x, const void* w, int rows, int cols,
                 float eps, hipStream_t stream);
void fei_attn_decode(const void* q, void* kc, void* vc, const int* table,
                     float* po, float* pml, void* out, const int* pos, int B,
                     int Hq, int Hkv, int D, int max_seq, int bs_log, int W,
                     int splits, float scale, long q_bs, const void* kin,
                     const void* vin, const float* cs, long kv_bs,
                     hipStream_t stream);
void fei_attn_decode_product(const void* q, void* kc, void* vc, const int* table,
                             float* po, float* pml, void* out, const int* pos,
                             int Hq, int Hkv, int D, int max_seq, int bs_log, int W,
                             int splits, float scale, long q_bs, const void* kin,
                             const void* vin, const float* cs, long kv_bs,
                             void* res, const void* w, const float* wscale, int N,
                             hipStream_t stream);
void fei_rope_kv_prefill(void* q, const void* k, const void* v, void* k_cache,
                         void* v_cache, const float* cos_sin, const int* pos0,
                         int B, int S, int Hq, int Hkv, int D, int max_seq,
                         long q_ts, long kv_ts, hipStream_t stream);
void fei_attn_prefill(const void* q, const void* k_cache, const void* v_cache,
                      void* out, const int* pos0, const int* kv_len, int B,
                      int S, int Hq, int Hkv, int D, int max_seq, float scale,
                      int causal, long q_ts, int splits, float* po, float* pml,
                      long kv_b, long kv_h, long kv_t, hipStream_t stream);

// What the layers share. Rows are B x S; S is 0 for a decoding step, of B rows. room:
// positions of a cache row, or those that a row of ``table`` can name (a paged pool's
// blocks of 1 << bs_log).
struct FewRows {
  int B, S, C, I, Hq, Hkv, D, room, bs_log, W, splits;
  float eps, scale;
  const int *pos, *table;
  const float* cos_sin;
  float *po, *pml;
};

// w: norm, q k v, output, norm, gates and up, down, caches of k and v. h [M, C] is
// replaced by the residual behind the layer; qkv [M, (Hq + 2 Hkv) D], att [M, Hq D], act
// [M, I] and normed [M, C] are room. sums [M, tiles]: of squares of h's rows, of tiles of 8
// columns, C up to 2048, or of 16; they are there already if ``summed``, and left there;
// of one row they are not made nor used. All bfloat16 on 16 bytes but for these; C, Hq D
// and I multiples of 64, of one row of 8; M up to 32, C up to 16384.
void fei_llama_few(const void* const* w, int summed, void* h, void* qkv,
                   void* att, void* act, void* normed, float* sums,
                   const FewRows* p, hipStream_t stream) {
  constexpr int GEMV_BF16 = 0, GEMV_RES = 1, GEMV_SWIGLU = 2;
  const FewRows& a = *p;
  const int M = a.B * (a.S ? a.S : 1), C = a.C, HD = a.Hq * a.D;
  const int kv = a.Hkv * a.D, width = HD + 2 * kv;
  const int tiles = (C + (C <= 2048 ? 7 : 15)) / (C <= 2048 ? 8 : 16);
  auto normed_product = [&](void* out, const void* gain, const void* wt, int N,
                            bool swiglu) {
    if (M == 1)
      return fei_gemv(out, h, gain, wt, nullptr, 1, N, C, a.eps,
                      swiglu ? GEMV_SWIGLU : GEMV_BF16, nullptr, stream);
    if (!summed) fei_rmsnorm(normed, h, gain, M, C, a.eps, stream);
    fei_skinny(swiglu ? nullptr : out, summed ? h : normed, wt, M, N, C,
               swiglu ? EPI_SWIGLU : EPI_BF16, nullptr, 1.f, 0.f, 0, 0, nullptr,
               swiglu ? out : nullptr, swiglu ? N : 0, nullptr,
               summed ? gain : nullptr, summed ? sums : nullptr,
               summed ? tiles : 0, summed ? a.eps : 0.f, nullptr, stream);
  };
  auto add = [&](const void* x, const void* wt, int K) {
    if (M == 1)
      return fei_gemv(h, x, nullptr, wt, nullptr, 1, C, K, 0.f, GEMV_RES,
                      nullptr, stream);
    fei_skinny(h, x, wt, M, C, K, EPI_RES_BF16, nullptr, 1.f, 0.f, 0, 0, nullptr,
               nullptr, 0, nullptr, nullptr, nullptr, tiles, 0.f, sums, stream);
    summed = 1;
  };
  void *kc = (void*)w[6], *vc = (void*)w[7];
  normed_product(qkv, w[0], w[1], width, false);
  const u16 *k = (const u16*)qkv + HD, *v = k + kv;
  if (a.S) {
    fei_rope_kv_prefill(qkv, k, v, kc, vc, a.cos_sin, a.pos, a.B, a.S, a.Hq, a.Hkv,
                        a.D, a.room, width, width, stream);
    fei_attn_prefill(qkv, kc, vc, att, a.pos, a.pos, a.B, a.S, a.Hq, a.Hkv, a.D,
                     a.room, a.scale, 1, width, a.splits, a.po, a.pml,
                     (long)a.Hkv * a.room * a.D, (long)a.room * a.D, a.D, stream);
  } else if (M == 1) {
    fei_attn_decode_product(qkv, kc, vc, a.table, a.po, a.pml, att, a.pos, a.Hq,
                            a.Hkv, a.D, a.room, a.bs_log, a.W, a.splits, a.scale,
                            width, k, v, a.cos_sin, width, h, w[2], nullptr, C,
                            stream);
  } else {
    fei_attn_decode(qkv, kc, vc, a.table, a.po, a.pml, att, a.pos, a.B, a.Hq,
                    a.Hkv, a.D, a.room, a.bs_log, a.W, a.splits, a.scale, width, k,
                    v, a.cos_sin, width, stream);
  }
  if (a.S || M > 1) add(att, w[2], HD);
  normed_product(act, w[3], w[4], a.I, true);
  add(act, w[5], a.I);
}

}  // extern "C"
