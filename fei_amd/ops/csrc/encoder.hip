// All layers of an encoder, launched from one call: over few rows its kernels take
// 4 to 10 us each, less than it takes to launch them one by one from Python.
#include "fei_epilogue.h"
#include "fei_mma.h"

namespace {

// Mean of a text's first len rows, to length 1: out [B, C] float32. A block per
// text; a thread has 8 columns of every SIDEth row. Bound by latency, and by what
// one CU loads of a long text (256 rows of 768: 393 KB). starts: null, or the first row
// of each text, where only the rows that texts have are there. In library operations it
// is nine launches and six passes over the rows in float32: 64 texts of 256 about
// 110 us for 8.6 here.
__global__ void __launch_bounds__(1024)
k_pool_unit(float* __restrict__ out, const u16* __restrict__ h,
            const int* __restrict__ lens, const int* __restrict__ starts,
            int S, int C) {
  extern __shared__ __align__(16) float part[];    // [sides][C]
  __shared__ float red[16];
  const int b = blockIdx.x, tid = threadIdx.x, nv = C >> 3;
  const int sides = 1024 / nv, side = tid / nv, c = tid - side * nv;
  const int n = min(max(lens[b], 0), S);
  const long first = starts ? starts[b] : (long)b * S;
  const s16x8* row = (const s16x8*)(h + first * C) + c;
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

// First row of each of B texts that lie one behind another, and behind the last the
// number of rows in all. A text has lens[b] rows, at least none and at most S.
__global__ void __launch_bounds__(1024)
k_text_starts(int* __restrict__ starts, const int* __restrict__ lens, int B,
              int S) {
  __shared__ int sum[16];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  int before = 0;
  for (int b0 = 0; b0 < B; b0 += 1024) {
    const int b = b0 + tid;
    int v = b < B ? min(max(lens[b], 0), S) : 0;
    const int n = v;
#pragma unroll
    for (int i = 1; i < 64; i *= 2) {
      const int t = __shfl_up(v, i);
      if (lane >= i) v += t;
    }
    __syncthreads();                       // the sums before have been read
    if (lane == 63) sum[wid] = v;
    __syncthreads();
    int all = 0;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (k < wid) v += sum[k];
      all += sum[k];
    }
    if (b < B) starts[b] = before + v - n;
    before += all;
  }
  if (tid == 0) starts[B] = before;
}

// out = LayerNorm(x + res) W^T + bias, or GELU of it: what an encoder's layer does
// behind each of its two residual products, for up to 8 XL rows of C <= 1024. Each
// block makes the norm of all rows for itself, to LDS, in twelve waves, while four
// others have their first rows of W on the way, which they multiply as k_skinny
// (gemv.hip) does. Block b writes normed rows b, b + gridDim.x, .. to ``normed``,
// which is none of the inputs.
//
// Bound by latency and, from 32 rows on, by the norm's own work on one CU: 16 rows of
// W and 24 of x take 7 us, a launch of 3.8 for the norm and one of 5 otherwise; in
// all four waves, in front of the products, 9. Whole encoders, 12 layers of 768,
// fused and not: 8 rows 341 us, 374; 16 383, 392; 24 392, 411; of more rows, in variants
// that are not kept, 32 448, 443; 64 661, 513.
constexpr int NORM_WAVES = 12;             // beside four that multiply

template <int XL, bool GELU>
__global__ void __launch_bounds__(64 * (4 + NORM_WAVES))
k_norm_product(u16* __restrict__ out, const u16* __restrict__ x,
               const u16* __restrict__ res, const u16* __restrict__ gain,
               const u16* __restrict__ shift, u16* __restrict__ normed,
               const u16* __restrict__ w, const u16* __restrict__ bias, int M,
               int N, int C, float eps) {
  constexpr int MT = (XL + 1) / 2, R = XL * 8, S = 3;
  constexpr int NR = (R + NORM_WAVES - 1) / NORM_WAVES;  // a wave's rows
  extern __shared__ __align__(16) u16 buf[];             // rows of w, of x
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, lg = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int r8 = lane >> 3, c8 = ((lane & 7) ^ r8) * 8;
  const int steps = C / 64, per = (steps + 3) / 4;
  const int lo = min(wid * per, steps - 1);
  const int n = wid < 4 ? max(min(steps, (wid + 1) * per) - wid * per, 0) : 0;
  const int turn = n ? blockIdx.x * 3 % n : 0;
  auto at = [&](int s) {
    const int t = s + turn;
    return lo + (t < n ? t : t - n);
  };
  const u16* src[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
    src[i] = w + (long)min(n0 + i * 8 + r8, N - 1) * C + c8;
  u16* mine = buf + wid * S * 1024;
  u16* xs = buf + 4 * S * 1024;
  const u32 lds = (u32)(uintptr_t)(__attribute__((address_space(3))) u16*)mine;
  auto load = [&](int step, int b) {
    if (step >= n) return;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      load_lds(src[i] + at(step) * 64, lds + (b * 1024 + i * 512) * 2);
  };
  const int nv = C >> 3;
  if (wid < 4) {
#pragma unroll
    for (int s = 0; s < S; ++s) load(s, s);
  } else {
    // rows wid - 4 and every 12th on; 8 columns lane and lane + 64 of each
    s16x8 xv[NR][2], rv[NR][2], gv[2], sv[2];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const long row = min(wid - 4 + NORM_WAVES * i, M - 1);
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        const int c = min(lane + 64 * v, nv - 1);
        xv[i][v] = ((const s16x8*)(x + row * C))[c];
        rv[i][v] = ((const s16x8*)(res + row * C))[c];
      }
    }
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      const int c = min(lane + 64 * v, nv - 1);
      gv[v] = ((const s16x8*)gain)[c];
      sv[v] = ((const s16x8*)shift)[c];
    }
    const bool both = lane + 64 < nv, one = lane < nv;
    float f[NR][2][8], sum[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      float t = 0.f, t0 = 0.f;             // in the order of k_layernorm_wave
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        t0 = t;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          f[i][v][j] = bf2f((u16)xv[i][v][j]) + bf2f((u16)rv[i][v][j]);
          t += f[i][v][j];
        }
      }
      sum[i] = wave_sum(both ? t : one ? t0 : 0.f);
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const float mean = sum[i] / (float)C;
      float t = 0.f, t0 = 0.f;
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        t0 = t;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          f[i][v][j] -= mean;
          t = fmaf(f[i][v][j], f[i][v][j], t);
        }
      }
      sum[i] = wave_sum(both ? t : one ? t0 : 0.f);
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const float inv = rsqrtf(sum[i] / (float)C + eps);
      const int row = wid - 4 + NORM_WAVES * i;
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        const int c = lane + 64 * v;
        s16x8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          o[j] = (short)El<u16>::st(fmaf(f[i][v][j] * inv,
                                         bf2f((u16)gv[v][j]),
                                         bf2f((u16)sv[v][j])));
        if (c < nv && row < R) {
          st8(xs + ((c >> 3) * R + row) * 64 + ((c & 7) ^ (row & 7)) * 8, o);
          if (row < M && row % gridDim.x == blockIdx.x)
            st8(normed + (long)row * C + c * 8, o);
        }
      }
    }
  }
  // not __syncthreads: the rows of w stay on the way
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  f32x4 acc[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  int b = 0;
  for (int s = 0; s < n; ++s) {
    if (n - s > 2) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    else if (n - s > 1) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const u16* bw = mine + b * 1024;
    const u16* bx = xs + at(s) * R * 64;
    s16x8 fa[2], fb[2][MT];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int c = ((kk * 4 + lg) ^ (l15 & 7)) * 8;
      fa[kk] = ld8(bw + l15 * 64 + c);
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        // an odd group of 8 rows stands in for the one after it
        const int r = XL >= 2 * j + 2 ? l15 : l15 & 7;
        fb[kk][j] = ld8(bx + (j * 16 + r) * 64 + c);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    load(s + S, b);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[j] = mma(fa[kk], fb[kk][j], acc[j]);
    b = b == S - 1 ? 0 : b + 1;
  }
  __syncthreads();
  f32x4* red = (f32x4*)buf;
#pragma unroll
  for (int j = 0; j < MT; ++j)
    if (wid < 4) red[(j * 4 + wid) * 64 + lane] = acc[j];
  __syncthreads();
  for (int t = wid; t < MT; t += 4 + NORM_WAVES) {
    const f32x4* p = red + t * 256 + lane;
    f32x4 v = p[0];
#pragma unroll
    for (int k = 1; k < 4; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += p[k * 64][e];
    const int m = t * 16 + l15, c = n0 + 4 * lg;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (m >= M || c + e >= N) break;
      const float y = v[e] + bf2f(bias[c + e]);
      out[(long)m * N + c + e] = f2bf(GELU ? gelu_erf(y) : y);
    }
  }
}

template <bool GELU>
void norm_product(u16* out, const u16* x, const u16* res, const u16* gain,
                  const u16* shift, u16* normed, const u16* w, const u16* bias,
                  int M, int N, int C, float eps, hipStream_t stream) {
  auto go = [&](auto kernel, int xl) {
    const int lds = 24576 + xl * 8 * C * 2;
    allow_lds(kernel, lds);
    hipLaunchKernelGGL(kernel, dim3((N + 15) / 16),
                       dim3(64 * (4 + NORM_WAVES)), lds, stream, out, x, res,
                       gain, shift, normed, w, bias, M, N, C, eps);
  };
  if (M <= 8) go(k_norm_product<1, GELU>, 1);
  else if (M <= 16) go(k_norm_product<2, GELU>, 2);
  else go(k_norm_product<3, GELU>, 3);
}

}  // namespace

extern "C" {

// h [B, S, C] bfloat16 on 16 bytes, C % 8 == 0, at most 2048
void fei_pool_unit(float* out, const void* h, const int* lens, int B, int S,
                   int C, hipStream_t stream) {
  const int sides = 1024 / (C / 8);
  hipLaunchKernelGGL(k_pool_unit, dim3(B), dim3(1024), sides * C * 4, stream,
                     out, (const u16*)h, lens, nullptr, S, C);
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

void fei_rows_bias_of(void* out, const void* x, const void* w, const void* bias,
                      int M, int N, int K, int gelu, const int* count,
                      hipStream_t stream);
void fei_rows_parts_of(float* out, const void* x, const void* w, int M, int N,
                       int K, int parts, const int* count, hipStream_t stream);
void fei_parts_layernorm_of(void* out, const float* parts, int np,
                            const void* bias, const void* res, const void* gain,
                            const void* shift, int rows, int cols, float eps,
                            const int* count, hipStream_t stream);
void fei_tile_counted(void* out, long os, const void* x, long xs, const void* w,
                      const void* bias, int M, int N, int K, int epi, int parts,
                      const int* count, hipStream_t stream);
void fei_attn_packed(const void* qkv, void* out, const int* kv_len,
                     const int* starts, int B, int S, int H, int D, float scale,
                     hipStream_t stream);
void fei_layernorm_packed(void* out, const void* x, const void* res,
                          const void* w, const void* bias, int texts, int S,
                          int cols, float eps, const int* starts,
                          hipStream_t stream);

void fei_embed_layernorm(void* out, const long* ids, const void* tok, const void* pos,
                         const void* w, const void* bias, int texts, int S, int cols,
                         int vocab, float eps, const int* starts,
                         hipStream_t stream);

// An encoder over the rows that its texts have, one behind another: out [B, C] float32.
// ids [B, S] of tok [vocab, C]; pos [S, C]; gain and shift of the first norm; w: 12 a layer, as in
// fei_encoder_layers; h, h1 and tmp have room for B * S rows of C, qkv of 3 H D, att of
// H D, inner of I; starts for B + 1. How many rows there are only the device knows: grids
// are made for all B * S, and blocks that have none leave. many: whether
// products are fei_tile_counted's, else in tiles of 64 x 64. p1, p2 and parts as in
// fei_encoder_layers. All on 16 bytes, C and H D and I
// multiples of 64, C <= 2048.
//
// 64 texts of 64 to 256 tokens, 10336 rows of 16384, 12 layers of 768: 2565 us; all
// rows, with the library's products, 3750. Texts of one length, for which the library's
// tiles are better: 32 x 128 to 64 x 256 2 to 6 % slower. Bound by the products, at 0.7 to
// 1 PFLOP/s of tiles that fill the chip one and a half times. To find the number costs each kernel
// a load before its first, 30 us of the 570 that 320 rows take in all.
void fei_encoder_packed(const void* const* w, int layers, float* out,
                        const long* ids, const void* tok, const void* pos,
                        int vocab, const void* gain, const void* shift, void* h,
                        void* h1, void* tmp, void* qkv, void* att,
                        void* inner, const int* lens, int* starts, int B, int S,
                        int H, int D, int C, int I, float scale, float eps,
                        int many, float* parts, int p1, int p2,
                        hipStream_t stream) {
  const int M = B * S, HD = H * D;
  const int* count = starts + B;
  hipLaunchKernelGGL(k_text_starts, dim3(1), dim3(1024), 0, stream, starts,
                     lens, B, S);
  fei_embed_layernorm(h, ids, tok, pos, gain, shift, B, S, C, vocab, eps, starts,
                      stream);
  auto product = [&](void* to, const void* x, const void* const* wb, int N, int K,
                     bool gelu) {
    constexpr int TILE_GELU = 2, TILE_BIAS = 5;
    if (!many)
      return fei_rows_bias_of(to, x, wb[0], wb[1], M, N, K, gelu, count, stream);
    fei_tile_counted(to, N, x, K, wb[0], wb[1], M, N, K,
                     gelu ? TILE_GELU : TILE_BIAS, 1, count, stream);
  };
  auto residual = [&](void* to, const void* from, const void* x,
                      const void* const* wb, int K, int np) {
    if (np) {
      constexpr int TILE_PARTS = 4;
      if (many)
        fei_tile_counted(parts, C, x, K, wb[0], nullptr, M, C, K, TILE_PARTS, np,
                         count, stream);
      else
        fei_rows_parts_of(parts, x, wb[0], M, C, K, np, count, stream);
      return fei_parts_layernorm_of(to, parts, np, wb[1], from, wb[2], wb[3], M,
                                    C, eps, count, stream);
    }
    product(tmp, x, wb, C, K, false);
    fei_layernorm_packed(to, tmp, from, wb[2], wb[3], B, S, C, eps, starts,
                         stream);
  };
  for (int l = 0; l < layers; ++l, w += 12) {
    product(qkv, h, w, 3 * HD, C, false);
    fei_attn_packed(qkv, att, lens, starts, B, S, H, D, scale, stream);
    residual(h1, h, att, w + 2, HD, p1);
    product(inner, h1, w + 6, I, C, true);
    residual(h, h1, inner, w + 8, I, p2);
  }
  hipLaunchKernelGGL(k_pool_unit, dim3(B), dim3(1024), 1024 / (C / 8) * C * 4,
                     stream, out, (const u16*)h, lens, starts, S, C);
}

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
  if (M <= 24 && C <= 1024) {
    // The norms inside the products behind them, but the last. What comes here is what the
    // one launch of encoder_one.hip does not take: widths beyond 768 (inner ones 3072, 12
    // heads), more than 32 layers, models that are to leave CUs to others, fewer CUs
    auto behind = [&](void* out, const void* res, const void* const* norm,
                      void* normed, const void* const* wb, int N, bool gelu) {
      auto run = [&](auto launch) {
        launch((u16*)out, (const u16*)tmp, (const u16*)res,
               (const u16*)norm[0], (const u16*)norm[1], (u16*)normed,
               (const u16*)wb[0], (const u16*)wb[1], M, N, C, eps, stream);
      };
      if (gelu) run(norm_product<true>);
      else run(norm_product<false>);
    };
    for (int l = 0; l < layers; ++l, w += 12) {
      if (l) behind(qkv, h1, w - 2, h, w, 3 * HD, false);
      else product(qkv, h, w, 3 * HD, C, EPI_BF16);
      fei_attn_prefill(qkv, (u16*)qkv + HD, (u16*)qkv + 2 * HD, att, pos0,
                       kv_len, B, S, H, H, D, S, scale, 0, 3L * HD, splits, po,
                       pml, 3L * S * HD, D, 3L * HD, stream);
      product(tmp, att, w + 2, C, HD, EPI_BF16);
      behind(inner, h, w + 4, h1, w + 6, I, true);
      product(tmp, inner, w + 8, C, I, EPI_BF16);
    }
    if (layers)
      fei_add_layernorm(h, tmp, h1, w[-2], w[-1], M, C, eps, 1, stream);
    return;
  }
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
