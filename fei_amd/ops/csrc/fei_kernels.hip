// fei_amd gfx950 kernels: RMSNorm, RoPE+KV-append, decode attention
// (split-K online-softmax), SwiGLU, sampling (argmax / Gumbel), position
// advance. Semantics match fei_amd/ops/reference.py; numerics tests compare
// against the fp32 torch reference (tests/test_ops_gpu.py).
//
// Design notes (per /opt/skills/guides/cdna_hip_programming.md):
//  - every memory-bound kernel loads bf16 as 16-byte vectors (Guideline 13)
//  - decode attention reads the length from a DEVICE tensor so the whole
//    decode step is hipGraph-capturable with a static grid
//  - block sizes are multiples of 64 (wave64)
#include "fei_epilogue.h"
#include "fei_mma.h"

// a logit as float: bfloat16 bits or float
__device__ __forceinline__ float logit(u16 v) { return bf2f(v); }
__device__ __forceinline__ float logit(float v) { return v; }

extern "C" {

// ---------------------------------------------------------------------------
// RMSNorm: out[r,:] = x[r,:] * rsqrt(mean(x^2)+eps) * w ; bf16 I/O, f32 acc.
// One block per row (grid-stride); cols % 8 == 0; cols/8 <= 256*MAX_V8.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
k_rmsnorm(u16* __restrict__ out, const u16* __restrict__ x,
          const u16* __restrict__ w, int rows, int cols, float eps) {
  __shared__ float red[4];
  const int nv = cols >> 3;                       // vec8 per row
  for (int row = blockIdx.x; row < rows; row += gridDim.x) {
    const s16x8* xr = (const s16x8*)(x + (long)row * cols);
    float ss = 0.f;
    for (int i = threadIdx.x; i < nv; i += blockDim.x) {
      s16x8 v = xr[i];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float f = bf2f((u16)v[j]);
        ss = fmaf(f, f, ss);
      }
    }
    ss = block_reduce_sum(ss, red);
    const float inv = rsqrtf(ss / (float)cols + eps);
    s16x8* orow = (s16x8*)(out + (long)row * cols);
    const s16x8* wv = (const s16x8*)w;
    // second read hits L1/L2 (a row is tiny vs 32 MB L2) — avoids a
    // runtime-indexed register array (guide rule 20: scratch).
    for (int i = threadIdx.x; i < nv; i += blockDim.x) {
      s16x8 v = xr[i];
      s16x8 wvv = wv[i];
      s16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        o[j] = (short)f2bf(bf2f((u16)v[j]) * inv * bf2f((u16)wvv[j]));
      orow[i] = o;
    }
    __syncthreads();
  }
}

void fei_rmsnorm(void* out, const void* x, const void* w, int rows, int cols,
                 float eps, hipStream_t stream) {
  int grid = rows < 2048 ? rows : 2048;
  hipLaunchKernelGGL(k_rmsnorm, dim3(grid), dim3(256), 0, stream,
                     (u16*)out, (const u16*)x, (const u16*)w, rows, cols, eps);
}

// ---------------------------------------------------------------------------
// Fused residual-add + RMSNorm: res = res + x ; out = rmsnorm(res) * w.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
k_add_rmsnorm(u16* __restrict__ out, u16* __restrict__ res,
              const u16* __restrict__ x, const u16* __restrict__ w,
              int rows, int cols, float eps) {
  __shared__ float red[4];
  const int nv = cols >> 3;
  for (int row = blockIdx.x; row < rows; row += gridDim.x) {
    const s16x8* xr = (const s16x8*)(x + (long)row * cols);
    s16x8* rr = (s16x8*)(res + (long)row * cols);
    float ss = 0.f;
    for (int i = threadIdx.x; i < nv; i += blockDim.x) {
      s16x8 xv = xr[i];
      s16x8 rv = rr[i];
      s16x8 nr;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float f = bf2f((u16)rv[j]) + bf2f((u16)xv[j]);
        u16 b = f2bf(f);
        nr[j] = (short)b;
        f = bf2f(b);                                // match reference rounding
        ss = fmaf(f, f, ss);
      }
      rr[i] = nr;
    }
    ss = block_reduce_sum(ss, red);
    const float inv = rsqrtf(ss / (float)cols + eps);
    s16x8* orow = (s16x8*)(out + (long)row * cols);
    const s16x8* wv = (const s16x8*)w;
    // re-read the just-written residual (L1/L2-hot; rule 20: no runtime-
    // indexed register array).
    for (int i = threadIdx.x; i < nv; i += blockDim.x) {
      s16x8 rv = rr[i];
      s16x8 wvv = wv[i];
      s16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        o[j] = (short)f2bf(bf2f((u16)rv[j]) * inv * bf2f((u16)wvv[j]));
      orow[i] = o;
    }
    __syncthreads();
  }
}

void fei_add_rmsnorm(void* out, void* res, const void* x, const void* w,
                     int rows, int cols, float eps, hipStream_t stream) {
  int grid = rows < 2048 ? rows : 2048;
  hipLaunchKernelGGL(k_add_rmsnorm, dim3(grid), dim3(256), 0, stream,
                     (u16*)out, (u16*)res, (const u16*)x, (const u16*)w,
                     rows, cols, eps);
}

// ---------------------------------------------------------------------------
// RoPE (decode) + KV append. q [B,Hq,D] roped in place at pos[b]; k,v
// [B,Hkv,D]: k roped and written with v into caches [B,Hkv,max_seq,D].
// Half-split pairing (Llama): pair (d, d+D/2). cos_sin: [max_seq, D/2, 2] f32.
// Grid: (Hq+Hkv, B); block D/2 threads (<=64 -> one wave for D=128).
// ---------------------------------------------------------------------------
__global__ void k_rope_kv_decode(u16* __restrict__ q, const u16* __restrict__ k,
                                 const u16* __restrict__ v,
                                 u16* __restrict__ kc, u16* __restrict__ vc,
                                 const float* __restrict__ cos_sin,
                                 const int* __restrict__ pos,
                                 int B, int Hq, int Hkv, int D, int max_seq,
                                 long q_bs, long kv_bs) {
  const int h = blockIdx.x;
  const int b = blockIdx.y;
  const int i = threadIdx.x;               // pair index in [0, D/2)
  const int p = pos[b];
  const float c = cos_sin[((long)p * (D / 2) + i) * 2 + 0];
  const float s = cos_sin[((long)p * (D / 2) + i) * 2 + 1];
  if (h < Hq) {
    u16* qp = q + (long)b * q_bs + (long)h * D;
    float x1 = bf2f(qp[i]), x2 = bf2f(qp[i + D / 2]);
    qp[i] = f2bf(x1 * c - x2 * s);
    qp[i + D / 2] = f2bf(x2 * c + x1 * s);
  } else {
    const int hk = h - Hq;
    const u16* kp = k + (long)b * kv_bs + (long)hk * D;
    const u16* vp = v + (long)b * kv_bs + (long)hk * D;
    u16* kcp = kc + (((long)b * Hkv + hk) * max_seq + p) * D;
    u16* vcp = vc + (((long)b * Hkv + hk) * max_seq + p) * D;
    float x1 = bf2f(kp[i]), x2 = bf2f(kp[i + D / 2]);
    kcp[i] = f2bf(x1 * c - x2 * s);
    kcp[i + D / 2] = f2bf(x2 * c + x1 * s);
    vcp[i] = vp[i];
    vcp[i + D / 2] = vp[i + D / 2];
  }
}

void fei_rope_kv_decode(void* q, const void* k, const void* v, void* k_cache,
                        void* v_cache, const float* cos_sin, const int* pos,
                        int B, int Hq, int Hkv, int D, int max_seq,
                        long q_bs, long kv_bs, hipStream_t stream) {
  hipLaunchKernelGGL(k_rope_kv_decode, dim3(Hq + Hkv, B), dim3(D / 2), 0,
                     stream, (u16*)q, (const u16*)k, (const u16*)v,
                     (u16*)k_cache, (u16*)v_cache, cos_sin, pos,
                     B, Hq, Hkv, D, max_seq, q_bs, kv_bs);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// RoPE (prefill) + KV append for S tokens. q [B,S,Hq,D] roped in place;
// k [B,S,Hkv,D] roped + appended with v at pos0[b]+s.
// A thread takes dimensions 8 i .. 8 i + 7 of a head and their partners D/2 on,
// 16 bytes each. Bound by HBM: 6 x 1001 tokens, 32/8 heads of 64: 60 -> 17 us
// (a thread per pair, 2 bytes a load, before), 2048 tokens, 32/8 of 128:
// 21 -> 14. VEC = false: D is no multiple of 16, or rows lie unaligned.
// ---------------------------------------------------------------------------
template <bool VEC>
__global__ void __launch_bounds__(256)
k_rope_kv_prefill(u16* __restrict__ q, const u16* __restrict__ k,
                  const u16* __restrict__ v, u16* __restrict__ kc,
                  u16* __restrict__ vc, const float* __restrict__ cos_sin,
                  const int* __restrict__ pos0, long units, int S, int Hq,
                  int Hkv, int D, int max_seq, long q_ts, long kv_ts) {
  constexpr int E = VEC ? 8 : 1;
  const int per = D / (2 * E), heads = Hq + Hkv;
  for (long u = (long)blockIdx.x * 256 + threadIdx.x; u < units;
       u += (long)gridDim.x * 256) {
    const int i = (int)(u % per) * E;
    const long th = u / per;
    const int h = (int)(th % heads);
    const long tok = th / heads;
    const int b = (int)(tok / S);
    const int p = pos0[b] + (int)(tok - (long)b * S);
    const float* cs = cos_sin + ((long)p * (D / 2) + i) * 2;
    const u16* src = h < Hq ? q + tok * q_ts + (long)h * D + i
                            : k + tok * kv_ts + (long)(h - Hq) * D + i;
    const long at = (((long)b * Hkv + h - Hq) * max_seq + p) * D + i;
    u16* dst = h < Hq ? (u16*)src : kc + at;
    u16 x1[E], x2[E], o1[E], o2[E];
    float t[2 * E];
    __builtin_memcpy(x1, src, sizeof(x1));
    __builtin_memcpy(x2, src + D / 2, sizeof(x2));
#pragma unroll
    for (int j = 0; j < 2 * E; ++j) t[j] = cs[j];
#pragma unroll
    for (int j = 0; j < E; ++j) {
      const float a = bf2f(x1[j]), c = bf2f(x2[j]);
      o1[j] = f2bf(a * t[2 * j] - c * t[2 * j + 1]);
      o2[j] = f2bf(c * t[2 * j] + a * t[2 * j + 1]);
    }
    __builtin_memcpy(dst, o1, sizeof(o1));
    __builtin_memcpy(dst + D / 2, o2, sizeof(o2));
    if (h >= Hq) {
      const u16* vp = v + tok * kv_ts + (long)(h - Hq) * D + i;
      __builtin_memcpy(o1, vp, sizeof(o1));
      __builtin_memcpy(o2, vp + D / 2, sizeof(o2));
      __builtin_memcpy(vc + at, o1, sizeof(o1));
      __builtin_memcpy(vc + at + D / 2, o2, sizeof(o2));
    }
  }
}

extern "C" void fei_rope_kv_prefill(void* q, const void* k, const void* v,
                                    void* k_cache, void* v_cache,
                                    const float* cos_sin, const int* pos0,
                                    int B, int S, int Hq, int Hkv, int D,
                                    int max_seq, long q_ts, long kv_ts,
                                    hipStream_t stream) {
  const bool vec = D % 16 == 0 && q_ts % 8 == 0 && kv_ts % 8 == 0 &&
                   (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v |
                     (uintptr_t)k_cache | (uintptr_t)v_cache) & 15) == 0;
  const long units = (long)B * S * (Hq + Hkv) * (D / (vec ? 16 : 2));
  const int grid = (int)min((units + 255) / 256, (long)65536);
#define GO(V)                                                                \
  hipLaunchKernelGGL(k_rope_kv_prefill<V>, dim3(grid), dim3(256), 0, stream, \
                     (u16*)q, (const u16*)k, (const u16*)v, (u16*)k_cache,   \
                     (u16*)v_cache, cos_sin, pos0, units, S, Hq, Hkv, D,     \
                     max_seq, q_ts, kv_ts)
  if (vec) GO(true); else GO(false);
#undef GO
}

extern "C" {

// ---------------------------------------------------------------------------
// SwiGLU: gate_up [rows, 2*inter] -> out [rows, inter]; silu(g)*u, f32 math.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
k_swiglu(u16* __restrict__ out, const u16* __restrict__ gu, long rows,
         int inter) {
  const long nvec = rows * (inter >> 3);
  const int iv = inter >> 3;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < nvec;
       idx += (long)gridDim.x * blockDim.x) {
    const long row = idx / iv;
    const int col = (int)(idx % iv);
    const s16x8* gp = (const s16x8*)(gu + row * 2 * inter) + col;
    const s16x8* up = (const s16x8*)(gu + row * 2 * inter + inter) + col;
    s16x8 g8 = *gp, u8 = *up;
    s16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float g = bf2f((u16)g8[j]);
      float u = bf2f((u16)u8[j]);
      float silu = g / (1.f + __expf(-g));
      o[j] = (short)f2bf(silu * u);
    }
    ((s16x8*)(out + row * inter))[col] = o;
  }
}

void fei_swiglu(void* out, const void* gate_up, long rows, int inter,
                hipStream_t stream) {
  long nvec = rows * (inter >> 3);
  int grid = (int)min((nvec + 255) / 256, (long)2048);
  if (grid < 1) grid = 1;
  hipLaunchKernelGGL(k_swiglu, dim3(grid), dim3(256), 0, stream,
                     (u16*)out, (const u16*)gate_up, rows, inter);
}

// ---------------------------------------------------------------------------
// Sampling. Stage 1: per (b, chunk) partial argmax of logits/T + Gumbel
// noise (temperature<=0 -> greedy, no noise). Stage 2: final reduce, write
// token[b], out_tokens[b, step]. `step` lives on device so the sequence of
// kernels is hipGraph-replayable.
// ws: [B, nchunks, 2] f32 (value, idx-as-float-bits via int store).
// ---------------------------------------------------------------------------
}  // extern "C"

template <typename T>
__global__ void __launch_bounds__(256)
k_sample_partial(const T* __restrict__ logits, float* __restrict__ ws,
                 int B, int vocab, int nchunks, float temperature,
                 u64 seed, const int* __restrict__ step) {
  const int chunk = blockIdx.x;
  const int b = blockIdx.y;
  const int chunk_size = (vocab + nchunks - 1) / nchunks;
  const int start = chunk * chunk_size;
  const int end = min(start + chunk_size, vocab);
  const u64 st = (u64)(*step);
  float best = -1.0f / 0.0f;
  int besti = start;
  const float invT = temperature > 0.f ? 1.f / temperature : 1.f;
  for (int i = start + threadIdx.x; i < end; i += blockDim.x) {
    float v = logit(logits[(long)b * vocab + i]) * invT;
    if (temperature > 0.f) {
      float u = hash_uniform(seed ^ (st * 0x51ed27f1ull) ^ ((u64)b << 40) ^ (u64)i);
      v += -__logf(-__logf(u));
    }
    if (v > best) { best = v; besti = i; }
  }
  // wave then block reduce of (best, besti)
#pragma unroll
  for (int off = 32; off; off >>= 1) {
    float ov = __shfl_xor(best, off);
    int oi = __shfl_xor(besti, off);
    if (ov > best || (ov == best && oi < besti)) { best = ov; besti = oi; }
  }
  __shared__ float rv[4];
  __shared__ int ri[4];
  const int wid = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { rv[wid] = best; ri[wid] = besti; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < (int)(blockDim.x >> 6); ++i)
      if (rv[i] > best || (rv[i] == best && ri[i] < besti)) { best = rv[i]; besti = ri[i]; }
    ws[((long)b * nchunks + chunk) * 2] = best;
    ((int*)ws)[((long)b * nchunks + chunk) * 2 + 1] = besti;
  }
}

extern "C" {

__global__ void k_sample_final(const float* __restrict__ ws,
                               int* __restrict__ token,
                               int* __restrict__ out_tokens,
                               const int* __restrict__ step,
                               int B, int nchunks, int max_new) {
  // one wave, parallel chunk loads + shfl argmax (a serial thread-0 loop
  // cost ~8 us at nchunks=64)
  const int b = blockIdx.x;
  const int lane = threadIdx.x & 63;
  float best = -1.0f / 0.0f;
  int besti = 0x7fffffff;
  for (int c = lane; c < nchunks; c += 64) {
    const float v = ws[((long)b * nchunks + c) * 2];
    const int i = ((const int*)ws)[((long)b * nchunks + c) * 2 + 1];
    if (v > best || (v == best && i < besti)) { best = v; besti = i; }
  }
#pragma unroll
  for (int off = 32; off; off >>= 1) {
    const float ov = __shfl_xor(best, off);
    const int oi = __shfl_xor(besti, off);
    if (ov > best || (ov == best && oi < besti)) { best = ov; besti = oi; }
  }
  if (lane == 0) {
    token[b] = besti;
    const int st = *step;
    if (out_tokens && st < max_new) out_tokens[(long)b * max_new + st] = besti;
  }
}

void fei_sample(const void* logits, int* token, int* out_tokens,
                const int* step, float* ws, int B, int vocab, int nchunks,
                float temperature, u64 seed, int max_new, int f32,
                hipStream_t stream) {
  if (f32)
    hipLaunchKernelGGL(k_sample_partial<float>, dim3(nchunks, B), dim3(256), 0,
                       stream, (const float*)logits, ws, B, vocab, nchunks,
                       temperature, seed, step);
  else
    hipLaunchKernelGGL(k_sample_partial<u16>, dim3(nchunks, B), dim3(256), 0,
                       stream, (const u16*)logits, ws, B, vocab, nchunks,
                       temperature, seed, step);
  hipLaunchKernelGGL(k_sample_final, dim3(B), dim3(64), 0, stream,
                     ws, token, out_tokens, step, B, nchunks, max_new);
}

// advance: pos[b]+=1 ; step+=1  (runs after sampling inside the graph)
// max_pos clamps the position at cache capacity: a caller decoding past
// max_seq would otherwise index the RoPE table / KV cache out of bounds
// from inside the graph (memory corruption, not an exception). Clamped
// steps overwrite the last slot — wrong results but memory-safe; the
// python loops stop at capacity before this matters.
__global__ void k_advance(int* pos, int* step, int B, int max_pos) {
  if ((int)threadIdx.x < B)
    pos[threadIdx.x] = min(pos[threadIdx.x] + 1, max_pos);
  if (threadIdx.x == 0 && step) *step += 1;
}

void fei_advance(int* pos, int* step, int B, int max_pos,
                 hipStream_t stream) {
  hipLaunchKernelGGL(k_advance, dim3(1), dim3(max(B, 64)), 0, stream,
                     pos, step, B, max_pos);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// First place of the largest value of each row (NaN above all, as in torch's
// argmax): ordered bits above the inverted place, so that one maximum of whole
// numbers decides. A row in chunks, a block each, then a wave per row. 20 x 128256
// bfloat16: 4.6 + 4.5 us, torch 41.
// ---------------------------------------------------------------------------
__device__ __forceinline__ u64 rank_of(float v, int i) {
  u32 u = __builtin_bit_cast(u32, v + 0.f);          // -0 counts as 0
  u = v != v ? ~0u : u & 0x80000000u ? ~u : u | 0x80000000u;
  return (u64)u << 32 | (u32)~i;
}
__device__ __forceinline__ u64 wave_max(u64 v) {
#pragma unroll
  for (int off = 32; off; off >>= 1) {
    const u64 o = __shfl_xor(v, off);
    v = o > v ? o : v;
  }
  return v;
}

template <typename T, bool VEC>
__global__ void __launch_bounds__(256)
k_argmax_chunk(u64* __restrict__ part, const T* __restrict__ x, int cols,
               int per) {
  constexpr int E = VEC ? 16 / sizeof(T) : 1;
  const T* row = x + (long)blockIdx.y * cols;
  const int lo = blockIdx.x * per, hi = min(cols, lo + per);
  u64 best = 0;
#pragma unroll 4
  for (int i = lo + threadIdx.x * E; i < hi; i += 256 * E) {
    T v[E];
    __builtin_memcpy(v, VEC ? __builtin_assume_aligned(row + i, 16) : row + i,
                     sizeof(v));
#pragma unroll
    for (int j = 0; j < E; ++j) {
      const u64 r = rank_of(logit(v[j]), i + j);
      best = r > best ? r : best;
    }
  }
  __shared__ u64 red[4];
  best = wave_max(best);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x) return;
  for (int i = 1; i < 4; ++i) best = red[i] > best ? red[i] : best;
  part[(long)blockIdx.y * gridDim.x + blockIdx.x] = best;
}

__global__ void __launch_bounds__(64)
k_argmax_row(long* __restrict__ out, const u64* __restrict__ part, int chunks) {
  const u64* p = part + (long)blockIdx.x * chunks;
  u64 best = 0;
  for (int i = threadIdx.x; i < chunks; i += 64) best = p[i] > best ? p[i] : best;
  best = wave_max(best);
  if (threadIdx.x == 0) out[blockIdx.x] = (u32)~(u32)best;
}

// x [rows, cols] -> out [rows]; part [rows, chunks]
extern "C" void fei_argmax(long* out, u64* part, const void* x, int rows,
                           int cols, int chunks, int f32, hipStream_t stream) {
  const int per = (cols + chunks * 8 - 1) / (chunks * 8) * 8;
  const dim3 grid(chunks, rows);
  const bool vec = cols % 8 == 0 && (uintptr_t)x % 16 == 0;
#define GO(T, V)                                                           \
  hipLaunchKernelGGL((k_argmax_chunk<T, V>), grid, dim3(256), 0, stream,   \
                     part, (const T*)x, cols, per)
  if (f32) {
    if (vec) GO(float, true); else GO(float, false);
  } else {
    if (vec) GO(u16, true); else GO(u16, false);
  }
#undef GO
  hipLaunchKernelGGL(k_argmax_row, dim3(rows), dim3(64), 0, stream, out, part,
                     chunks);
}

// ---------------------------------------------------------------------------
// One-pass sampler for small B: grid (B), block 1024 = 16 waves streaming
// the whole vocab row; replaces the partial+final pair (one node, no
// workspace round trip).
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(1024)
k_sample_onepass(const T* __restrict__ logits, int* __restrict__ token,
                 int* __restrict__ out_tokens, const int* __restrict__ step,
                 int B, int vocab, float temperature, u64 seed, int max_new) {
  const int b = blockIdx.x;
  const int tid = threadIdx.x;
  const u64 st = (u64)(*step);
  const float invT = temperature > 0.f ? 1.f / temperature : 1.f;
  float best = -1.0f / 0.0f;
  int besti = 0x7fffffff;
  const T* row = logits + (long)b * vocab;
  // rows of a vocabulary that is no multiple of 8 are not 16-byte aligned
  const int nv = (vocab & 7) ? 0 : vocab >> 3;
  for (int i = tid; i < nv; i += blockDim.x) {
    T v8[8];
    __builtin_memcpy(v8, __builtin_assume_aligned(row + i * 8, 16),
                     sizeof(v8));
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int idx = i * 8 + j;
      float v = logit(v8[j]) * invT;
      if (temperature > 0.f) {
        float u = hash_uniform(seed ^ (st * 0x51ed27f1ull) ^ ((u64)b << 40) ^ (u64)idx);
        v += -__logf(-__logf(u));
      }
      if (v > best || (v == best && idx < besti)) { best = v; besti = idx; }
    }
  }
  // tail (vocab % 8)
  for (int idx = nv * 8 + tid; idx < vocab; idx += blockDim.x) {
    float v = logit(row[idx]) * invT;
    if (temperature > 0.f) {
      float u = hash_uniform(seed ^ (st * 0x51ed27f1ull) ^ ((u64)b << 40) ^ (u64)idx);
      v += -__logf(-__logf(u));
    }
    if (v > best || (v == best && idx < besti)) { best = v; besti = idx; }
  }
#pragma unroll
  for (int off = 32; off; off >>= 1) {
    const float ov = __shfl_xor(best, off);
    const int oi = __shfl_xor(besti, off);
    if (ov > best || (ov == best && oi < besti)) { best = ov; besti = oi; }
  }
  __shared__ float rv[16];
  __shared__ int ri[16];
  const int wid = tid >> 6;
  if ((tid & 63) == 0) { rv[wid] = best; ri[wid] = besti; }
  __syncthreads();
  if (tid == 0) {
    const int nw = blockDim.x >> 6;
    for (int i = 1; i < nw; ++i)
      if (rv[i] > best || (rv[i] == best && ri[i] < besti)) {
        best = rv[i]; besti = ri[i];
      }
    token[b] = besti;
    if (out_tokens && (int)st < max_new)
      out_tokens[(long)b * max_new + (int)st] = besti;
  }
}

extern "C" {

void fei_sample_onepass(const void* logits, int* token, int* out_tokens,
                        const int* step, int B, int vocab, float temperature,
                        u64 seed, int max_new, int f32, hipStream_t stream) {
  if (f32)
    hipLaunchKernelGGL(k_sample_onepass<float>, dim3(B), dim3(1024), 0, stream,
                       (const float*)logits, token, out_tokens, step, B, vocab,
                       temperature, seed, max_new);
  else
    hipLaunchKernelGGL(k_sample_onepass<u16>, dim3(B), dim3(1024), 0, stream,
                       (const u16*)logits, token, out_tokens, step, B, vocab,
                       temperature, seed, max_new);
}

// Shard sampler for tensor-parallel decode: each rank samples over its OWN
// lm_head shard [B, vocab_local] and emits (best value, best GLOBAL index)
// into out[b] = {f32 val, i32 idx}; the ranks then all-gather 8 bytes per
// sequence instead of the full vocab row (replaces the 513 KB logits
// all-gather per step at Llama-3 vocab). Gumbel noise is keyed by the
// GLOBAL index, so the sharded sample is bit-identical to the full-vocab
// k_sample_onepass on the gathered logits.
__global__ void __launch_bounds__(1024)
k_sample_shard(const u16* __restrict__ logits, float* __restrict__ out,
               const int* __restrict__ step, int B, int vocab_local,
               int v_offset, float temperature, u64 seed) {
  const int b = blockIdx.x;
  const int tid = threadIdx.x;
  const u64 st = (u64)(*step);
  const float invT = temperature > 0.f ? 1.f / temperature : 1.f;
  float best = -1.0f / 0.0f;
  int besti = 0x7fffffff;
  const s16x8* row = (const s16x8*)(logits + (long)b * vocab_local);
  const int nv = vocab_local >> 3;
  for (int i = tid; i < nv; i += blockDim.x) {
    s16x8 v8 = row[i];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int idx = v_offset + i * 8 + j;
      float v = bf2f((u16)v8[j]) * invT;
      if (temperature > 0.f) {
        float u = hash_uniform(seed ^ (st * 0x51ed27f1ull) ^ ((u64)b << 40) ^ (u64)idx);
        v += -__logf(-__logf(u));
      }
      if (v > best || (v == best && idx < besti)) { best = v; besti = idx; }
    }
  }
  for (int k = nv * 8 + tid; k < vocab_local; k += blockDim.x) {
    const int idx = v_offset + k;
    float v = bf2f(logits[(long)b * vocab_local + k]) * invT;
    if (temperature > 0.f) {
      float u = hash_uniform(seed ^ (st * 0x51ed27f1ull) ^ ((u64)b << 40) ^ (u64)idx);
      v += -__logf(-__logf(u));
    }
    if (v > best || (v == best && idx < besti)) { best = v; besti = idx; }
  }
#pragma unroll
  for (int off = 32; off; off >>= 1) {
    const float ov = __shfl_xor(best, off);
    const int oi = __shfl_xor(besti, off);
    if (ov > best || (ov == best && oi < besti)) { best = ov; besti = oi; }
  }
  __shared__ float rv[16];
  __shared__ int ri[16];
  const int wid = tid >> 6;
  if ((tid & 63) == 0) { rv[wid] = best; ri[wid] = besti; }
  __syncthreads();
  if (tid == 0) {
    const int nw = blockDim.x >> 6;
    for (int i = 1; i < nw; ++i)
      if (rv[i] > best || (rv[i] == best && ri[i] < besti)) {
        best = rv[i]; besti = ri[i];
      }
    out[(long)b * 2] = best;
    ((int*)out)[(long)b * 2 + 1] = besti;
  }
}

void fei_sample_shard(const void* logits, float* out, const int* step,
                      int B, int vocab_local, int v_offset, float temperature,
                      u64 seed, hipStream_t stream) {
  hipLaunchKernelGGL(k_sample_shard, dim3(B), dim3(1024), 0, stream,
                     (const u16*)logits, out, step, B, vocab_local, v_offset,
                     temperature, seed);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// LayerNorm (+ optional fused residual add) and bias+GELU — the encoder-side
// kernels (BERT/bge architecture: post-LN residual blocks, GELU MLP).
// bf16 I/O, f32 statistics. Rows of up to 2048 columns: a wave each, kept in
// registers between the passes, no barrier. Bound by HBM (16384 rows of 768 with
// residual: 41 us with a block per row that read it three times, 16 so). Wider
// rows: one block per row.
// ---------------------------------------------------------------------------
namespace {

// PACK: text b of at most S rows has rows starts[b] to starts[b + 1] - 1 of ``out``.
// ALL_ROWS: x is [texts, S, cols], and the rows that a text has not are left out;
// PACKED_ROWS: x and res are packed already.
// EMBED: of text b's token s x has row ids[b, s], and res row s; their sum is rounded to
// bfloat16. Two launches less: an encoder of 24 tokens 388 -> 382 us.
enum { NO_PACK, ALL_ROWS, PACKED_ROWS };
template <int V, bool RES, int PACK = NO_PACK, bool EMBED = false>
__global__ void __launch_bounds__(256)               // V loads of 8 columns a lane
k_layernorm_wave(u16* __restrict__ out, const u16* __restrict__ x,
                 const u16* __restrict__ res, const u16* __restrict__ w,
                 const u16* __restrict__ bias, int rows, int cols, float eps,
                 const int* __restrict__ starts, int S,
                 const long* __restrict__ ids, int vocab) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  int to = row;
  if (PACK == ALL_ROWS) {
    const int b = row / S;
    to = starts[b] + row - b * S;
    if (to >= starts[b + 1]) return;
  }
  if (PACK == PACKED_ROWS && row >= starts[rows / S]) return;
  const int nv = cols >> 3;
  long from = row;
  if (EMBED) {
    from = ids[row];
    if (from < 0 || from >= vocab) __builtin_trap();   // as torch's embedding does
  }
  const s16x8* xr = (const s16x8*)(x + from * cols);
  const s16x8* rr = (const s16x8*)(res + (long)(EMBED ? row % S : row) * cols);
  s16x8 xv[V], rv[RES ? V : 1], wv[V], bv[V];
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int at = min(lane + 64 * i, nv - 1);
    xv[i] = xr[at];
    if (RES) rv[i] = rr[at];
  }
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int at = min(lane + 64 * i, nv - 1);
    wv[i] = ((const s16x8*)w)[at];
    bv[i] = ((const s16x8*)bias)[at];
  }
  float f[V][8], sum = 0.f;
#pragma unroll
  for (int i = 0; i < V; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      f[i][j] = bf2f((u16)xv[i][j]);
      if (RES) f[i][j] += bf2f((u16)rv[i][j]);
      if (EMBED) f[i][j] = bf2f(f2bf(f[i][j]));
      if (lane + 64 * i < nv) sum += f[i][j];
    }
  const float mean = wave_reduce_sum(sum) / (float)cols;
  float var = 0.f;
#pragma unroll
  for (int i = 0; i < V; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      f[i][j] -= mean;
      if (lane + 64 * i < nv) var = fmaf(f[i][j], f[i][j], var);
    }
  const float inv = rsqrtf(wave_reduce_sum(var) / (float)cols + eps);
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int at = lane + 64 * i;
    if (at >= nv) break;
    s16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      o[j] = (short)f2bf(f[i][j] * inv * bf2f((u16)wv[i][j]) +
                         bf2f((u16)bv[i][j]));
    ((s16x8*)(out + (long)to * cols))[at] = o;
  }
}

}  // namespace

extern "C" {

__global__ void __launch_bounds__(256)
k_add_layernorm(u16* __restrict__ out, const u16* __restrict__ x,
                const u16* __restrict__ res, const u16* __restrict__ w,
                const u16* __restrict__ bias, int rows, int cols, float eps,
                int has_res) {
  __shared__ float red[4];
  const int nv = cols >> 3;
  for (int row = blockIdx.x; row < rows; row += gridDim.x) {
    const s16x8* xr = (const s16x8*)(x + (long)row * cols);
    const s16x8* rr = (const s16x8*)(res + (long)row * cols);
    float sum = 0.f;
    for (int i = threadIdx.x; i < nv; i += blockDim.x) {
      s16x8 xv = xr[i];
      s16x8 rv = has_res ? rr[i] : xv;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float f = bf2f((u16)xv[j]) + (has_res ? bf2f((u16)rv[j]) : 0.f);
        sum += f;
      }
    }
    sum = block_reduce_sum(sum, red);
    const float mean = sum / (float)cols;
    float var = 0.f;
    for (int i = threadIdx.x; i < nv; i += blockDim.x) {
      s16x8 xv = xr[i];
      s16x8 rv = has_res ? rr[i] : xv;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float f = bf2f((u16)xv[j]) + (has_res ? bf2f((u16)rv[j]) : 0.f) - mean;
        var = fmaf(f, f, var);
      }
    }
    var = block_reduce_sum(var, red);
    const float inv = rsqrtf(var / (float)cols + eps);
    s16x8* orow = (s16x8*)(out + (long)row * cols);
    const s16x8* wv8 = (const s16x8*)w;
    const s16x8* bv8 = (const s16x8*)bias;
    for (int i = threadIdx.x; i < nv; i += blockDim.x) {
      s16x8 xv = xr[i];
      s16x8 rv = has_res ? rr[i] : xv;
      s16x8 wv = wv8[i];
      s16x8 bv = bv8[i];
      s16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float f = bf2f((u16)xv[j]) + (has_res ? bf2f((u16)rv[j]) : 0.f);
        o[j] = (short)f2bf((f - mean) * inv * bf2f((u16)wv[j]) +
                           bf2f((u16)bv[j]));
      }
      orow[i] = o;
    }
    __syncthreads();
  }
}

void fei_add_layernorm(void* out, const void* x, const void* res,
                       const void* w, const void* bias, int rows, int cols,
                       float eps, int has_res, hipStream_t stream) {
  const int nv = cols >> 3;
  auto by_wave = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((rows + 3) / 4), dim3(256), 0, stream,
                       (u16*)out, (const u16*)x, (const u16*)res,
                       (const u16*)w, (const u16*)bias, rows, cols, eps,
                       nullptr, 0, nullptr, 0);
  };
  if (nv >= 1 && nv <= 64)
    return by_wave(has_res ? k_layernorm_wave<1, true>
                           : k_layernorm_wave<1, false>);
  if (nv > 64 && nv <= 128)
    return by_wave(has_res ? k_layernorm_wave<2, true>
                           : k_layernorm_wave<2, false>);
  if (nv > 128 && nv <= 256)
    return by_wave(has_res ? k_layernorm_wave<4, true>
                           : k_layernorm_wave<4, false>);
  int grid = rows < 2048 ? rows : 2048;
  hipLaunchKernelGGL(k_add_layernorm, dim3(grid), dim3(256), 0, stream,
                     (u16*)out, (const u16*)x, (const u16*)res,
                     (const u16*)w, (const u16*)bias, rows, cols, eps,
                     has_res);
}

// LayerNorm of packed x + res: of the rows that texts have; starts has texts + 1 values.
// cols % 8 == 0, at most 2048.
void fei_layernorm_packed(void* out, const void* x, const void* res,
                          const void* w, const void* bias, int texts, int S,
                          int cols, float eps, const int* starts,
                          hipStream_t stream) {
  const int rows = texts * S, nv = cols >> 3;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((rows + 3) / 4), dim3(256), 0, stream,
                       (u16*)out, (const u16*)x, (const u16*)res,
                       (const u16*)w, (const u16*)bias, rows, cols, eps,
                       starts, S, nullptr, 0);
  };
  if (nv <= 64) go(k_layernorm_wave<1, true, PACKED_ROWS>);
  else if (nv <= 128) go(k_layernorm_wave<2, true, PACKED_ROWS>);
  else go(k_layernorm_wave<4, true, PACKED_ROWS>);
}

// LayerNorm of the sum of the rows of tok [vocab, cols] that ids [texts, S] name and of
// pos [S, cols]: of all, or with starts those that texts have, packed. All bfloat16 on 16
// bytes, cols % 8 == 0, at most 2048.
void fei_embed_layernorm(void* out, const long* ids, const void* tok, const void* pos,
                         const void* w, const void* bias, int texts, int S, int cols,
                         int vocab, float eps, const int* starts,
                         hipStream_t stream) {
  const int rows = texts * S, nv = cols >> 3;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((rows + 3) / 4), dim3(256), 0, stream,
                       (u16*)out, (const u16*)tok, (const u16*)pos,
                       (const u16*)w, (const u16*)bias, rows, cols, eps,
                       starts, S, ids, vocab);
  };
#define GO(V) go(starts ? k_layernorm_wave<V, true, ALL_ROWS, true>           \
                        : k_layernorm_wave<V, true, NO_PACK, true>)
  if (nv <= 64) GO(1);
  else if (nv <= 128) GO(2);
  else GO(4);
#undef GO
}

// GELU, erf form (torch's default). 16384 x 3072: 50 us with erff, 41 with
// gelu_erf, which keeps the vector units less busy; memory would take 31.
__global__ void __launch_bounds__(256)
k_gelu(u16* __restrict__ out, const u16* __restrict__ x, long n8) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n8;
       i += (long)gridDim.x * blockDim.x) {
    s16x8 v = ((const s16x8*)x)[i];
    s16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      o[j] = (short)El<u16>::st(gelu_erf(bf2f((u16)v[j])));
    ((s16x8*)out)[i] = o;
  }
}

void fei_gelu(void* out, const void* x, long n, hipStream_t stream) {
  long n8 = n >> 3;
  int grid = (int)((n8 + 255) / 256);
  if (grid > 2048) grid = 2048;
  if (grid < 1) grid = 1;
  hipLaunchKernelGGL(k_gelu, dim3(grid), dim3(256), 0, stream,
                     (u16*)out, (const u16*)x, n8);
}

}  // extern "C"
