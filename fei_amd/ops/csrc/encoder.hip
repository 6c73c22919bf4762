// All layers of an encoder, launched from one call: over few rows its kernels take
// 4 to 10 us each, less than it takes to launch them one by one from Python.
#include "fei_epilogue.h"

namespace {

// Mean of a text's first len rows, to length 1: out [B, C] float32. A block per
// text; a thread has 8 columns of every SIDEth row. Bound by latency, and by what
// one CU loads of a long text (256 rows of 768: 393 KB). In library operations it
// is nine launches and six passes over the rows in float32: 64 texts of 256 about
// 110 us for 8.6 here.
__global__ void __launch_bounds__(1024)
k_pool_unit(float* __restrict__ out, const u16* __restrict__ h,
            const int* __restrict__ lens, int S, int C) {
  extern __shared__ __align__(16) float part[];    // [sides][C]
  __shared__ float red[16];
  const int b = blockIdx.x, tid = threadIdx.x, nv = C >> 3;
  const int sides = 1024 / nv, side = tid / nv, c = tid - side * nv;
  const int n = min(max(lens[b], 0), S);
  const s16x8* row = (const s16x8*)(h + (long)b * S * C) + c;
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = 0.f;
  if (side < sides) {
#pragma unroll 4
    for (int s = side; s < n; s += sides) {
      const s16x8 x = row[(long)s * nv];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] += bf2f((u16)x[j]);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) part[side * C + c * 8 + j] = v[j];
  }
  __syncthreads();
  float sq = 0.f;
  for (int i = tid; i < C; i += 1024) {
    float t = 0.f;
    for (int k = 0; k < sides; ++k) t += part[k * C + i];
    t /= (float)max(n, 1);
    part[i] = t;                           // of this thread's columns alone
    sq = fmaf(t, t, sq);
  }
  sq = wave_reduce_sum(sq);
  if ((tid & 63) == 0) red[tid >> 6] = sq;
  __syncthreads();
  sq = 0.f;
#pragma unroll
  for (int k = 0; k < 16; ++k) sq += red[k];
  const float len = sqrtf(sq);
  const float norm = len < 1e-12f ? 1e-12f : len;   // NaN stays
  for (int i = tid; i < C; i += 1024) out[(long)b * C + i] = part[i] / norm;
}

}  // namespace

extern "C" {

// h [B, S, C] bfloat16 on 16 bytes, C % 8 == 0, at most 2048
void fei_pool_unit(float* out, const void* h, const int* lens, int B, int S,
                   int C, hipStream_t stream) {
  const int sides = 1024 / (C / 8);
  hipLaunchKernelGGL(k_pool_unit, dim3(B), dim3(1024), sides * C * 4, stream,
                     out, (const u16*)h, lens, S, C);
}

void fei_skinny(void* out, const void* x, const void* w, int M, int N, int K,
                int epi, const float* bias, float scale, float cap, int n_mix,
                int n_router, float* router, void* act, long as,
                const void* bias16, const void* gain, const float* sums,
                int tiles, float eps, float* sums_out, hipStream_t stream);
void fei_rows_bias(void* out, const void* x, const void* w, const void* bias,
                   int M, int N, int K, int gelu, hipStream_t stream);
void fei_rows(void* out, const void* x, long xs, const void* w, int M, int N,
              int K, int swiglu, int xj, int wide, int parts,
              hipStream_t stream);
void fei_parts_layernorm(void* out, const float* parts, int np,
                         const void* bias, const void* res, const void* gain,
                         const void* shift, int rows, int cols, float eps,
                         hipStream_t stream);
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
// their rows holds for all. splits, po, pml: see fei_attn_prefill. parts: room
// for the larger of p1 and p2 times B * S * C floats, and as many parts of the
// output and the outer product's K, for more than 64 rows (0: whole products).
void fei_encoder_layers(const void* const* w, int layers, void* h, void* h1,
                        void* tmp, void* qkv, void* att, void* inner,
                        const int* pos0, const int* kv_len, int B, int S, int H,
                        int D, int C, int I, float scale, float eps,
                        int splits, float* po, float* pml, float* parts,
                        int p1, int p2, hipStream_t stream) {
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
  // to = LayerNorm(x W^T + b + from). Few tiles: K in parts, which the norm sums
  // (12 layers of 768: 100 rows 667 us for 819, 512 848 for 954)
  auto residual = [&](void* to, const void* from, const void* x,
                      const void* const* wb, int K, int np) {
    if (np) {
      fei_rows(parts, x, K, wb[0], M, C, K, 0, 2, 0, np, stream);
      return fei_parts_layernorm(to, parts, np, wb[1], from, wb[2], wb[3], M, C,
                                 eps, stream);
    }
    product(tmp, x, wb, C, K, EPI_BF16);
    fei_add_layernorm(to, tmp, from, wb[2], wb[3], M, C, eps, 1, stream);
  };
  for (int l = 0; l < layers; ++l, w += 12) {
    product(qkv, h, w, 3 * HD, C, EPI_BF16);
    fei_attn_prefill(qkv, (u16*)qkv + HD, (u16*)qkv + 2 * HD, att, pos0, kv_len,
                     B, S, H, H, D, S, scale, 0, 3L * HD, splits, po, pml,
                     3L * S * HD, D, 3L * HD, stream);
    residual(h1, h, att, w + 2, HD, p1);
    product(inner, h1, w + 6, I, C, EPI_GELU);
    residual(h, h1, inner, w + 8, I, p2);
  }
}

}  // extern "C"
