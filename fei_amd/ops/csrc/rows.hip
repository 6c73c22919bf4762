// Products of tens to hundreds of rows with a weight matrix (gfx950):
// out[M, N] = x[M, K] @ W[N, K]^T in bfloat16 with float32 sums, where a library
// product leaves the chip half idle or makes a result that takes another pass.
#include <type_traits>

#include "fei_epilogue.h"
#include "fei_mma.h"

namespace {

enum {
  ROWS_PARTS = 0,      // float32 sums of a part of K, [parts][M][N]
  ROWS_SWIGLU = 1,     // W has N rows of gates, then N of up; bfloat16
  ROWS_BIAS = 2,       // with a bias per column; bfloat16
  ROWS_GELU = 3,       // of that
};

// Tiles of 32 XJ rows x 32 WI rows of W (SWIGLU: half of them gates, the others
// the same of up), 4 waves of half by half, S LDS buffers of 64 steps of K filled
// by direct loads. The 16-byte places of a row are permuted by the row, in the
// address that a lane reads, so that the fragment reads of 16 rows spread over the
// banks. Fragments of 32 steps are read ahead of the products with the 32 before;
// reads and loads go out between the matrix instructions.
//
// blockIdx.y: a part of K. Column tiles start at different steps of their part:
// rows of W often lie a multiple of 4 KB apart, and the same columns of all of
// them would be on the same memory channels; not where x is more than an L2 holds,
// which all tiles of columns read together then. An XCD gets consecutive tiles, four
// of rows times all of columns, rows first, so that its L2 holds what they share.
//
// Bound by HBM for one tile of rows, by the loads to LDS (36 to 43 bytes a clock
// and CU go through them) for more. Cold weights, 75 rows, against the library:
// 4096 x 14336 in 8 parts 27 us (50), 4096 x 4096 in 4 11.4 (16.2), 6144 x 4096 in
// 4 15.8 (23.8), 2 x 14336 x 4096 with SwiGLU 48 (53 + 4.5), 58 with all tiles
// starting at the same step. Two buffers instead of four: 71. Among the other
// kernels of a layer the four take 29.7, 13.4, 17.2 and 49.8.
//
// ONCE: there is one tile of rows, so that w is read once and need not push x out of
// the L2: 75 rows 26.6 -> 24.3, 14.9 -> 14.4, 45.9 -> 44.8, 40 rows of the last 43.7
// -> 38.3; two tiles share what they read (200 rows, 2 x 14336 x 4096 in tiles of
// 64 columns 92 -> 117).
//
// COUNTED: only the device knows how many of the ``room`` rows there are, and finds the
// number at ``count``; blocks without a tile leave at once. The others are told their
// tiles of rows, nm: to look at count and reckon cost 75 rows 0.4 us a launch.
template <int XJ, int WI, int S, int EPI, bool ONCE, bool COUNTED>
__global__ void __launch_bounds__(256, S * (XJ + WI) <= 20 ? 2 : 1)
k_rows(void* __restrict__ outp, const u16* __restrict__ x, long xs,
       const u16* __restrict__ w, const u16* __restrict__ bias, int room, int N,
       int K, int nx, int all_nm, const int* __restrict__ count) {
  constexpr int TM = 32 * XJ, TN = 32 * WI, MX = XJ > WI ? XJ : WI;
  constexpr int CN = EPI == ROWS_SWIGLU ? TN / 2 : TN;   // columns of out
  // whether nothing is asked for past the end, so that 16 steps do not become 20. Else
  // the last step is read again, into a buffer that is free: the second loop costs
  // registers, and more than it gains where steps are many (2 x 14336 x 4096 with
  // SwiGLU, 96 rows 45.1 us, 46.0 with one loop; 128 53.4, 50.3; 256 99.7, 86.7; parts
  // of 4096 x 14336, 128 rows 30.1, 31.9; 200 50.7, 46.9; 256 52.2, 49.8)
  constexpr bool EXACT =
      WI == 2 || (ONCE && (XJ < 4 || EPI != ROWS_SWIGLU));
  constexpr int BUF = (TM + TN) * 64, LOADS = XJ + WI;
  extern __shared__ __align__(16) u16 buf[];
  const int M =
      COUNTED ? __builtin_amdgcn_readfirstlane(min(*count, room)) : room;
  const int nm = COUNTED ? (M + TM - 1) / TM : all_nm, total = nx * nm, per = (total + 7) / 8;
  const int id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || id >= total) return;
  const int g0 = id / (4 * nx) * 4, gm = min(4, nm - g0), gr = id - g0 * nx;
  const int tile = gr / gm, n0 = tile * CN;
  const int m0 = (g0 + gr % gm) * TM, cnt = min(TM, M - m0);
  const int all = K / 64, first = (int)(blockIdx.y * (long)all / gridDim.y);
  const int steps = (int)((blockIdx.y + 1) * (long)all / gridDim.y) - first;
  const int turn = (long)M * K <= 2 << 20 ? tile * 3 % steps : 0;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, lg = lane >> 4;
  // 8 rows a load; the place of a row's 8 values depends on the row
  const int r8 = lane >> 3, c8 = ((lane & 7) ^ r8) * 8 + first * 64;
  const u16* src[LOADS];
#pragma unroll
  for (int i = 0; i < XJ; ++i)
    src[i] = x + (long)(m0 + min((wid * XJ + i) * 8 + r8, cnt - 1)) * xs + c8;
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    int r = (wid * WI + i) * 8 + r8;       // row of the tile
    long n;
    if (EPI == ROWS_SWIGLU) {              // a wave's half: gates, then up
      const int half = r / (TN / 2), q = r % (TN / 2), up = q / (TN / 4);
      n = min(n0 + half * (TN / 4) + q % (TN / 4), N - 1) + (long)up * N;
    } else {
      n = min(n0 + r, N - 1);
    }
    src[XJ + i] = w + n * K + c8;
  }
  const u32 lds = (u32)(uintptr_t)(__attribute__((address_space(3))) u16*)buf;
  auto load = [&](int step, int b, int i) {
    int t = (EXACT ? step : min(step, steps - 1)) + turn;
    t = t < steps ? t : t - steps;
    const u32 to = lds + b * BUF * 2 +
                   (i < XJ ? (wid * XJ + i) * 1024
                           : TM * 128 + (wid * WI + i - XJ) * 1024);
    if (ONCE && i >= XJ) load_lds_nt(src[i] + t * 64, to);
    else load_lds(src[i] + t * 64, to);
  };
  const int xm = (wid & 1) * 16 * XJ, wm = (wid >> 1) * 16 * WI;
  struct Frags {
    s16x8 w[WI], x[XJ];
  };
  auto read = [&](Frags& f, int b, int kk, int i) {
    const int c = ((kk * 4 + lg) ^ (l15 & 7)) * 8;
    const u16* bx = buf + b * BUF;
    if (i < XJ) f.x[i] = ld8(bx + (xm + i * 16 + l15) * 64 + c);
    if (i < WI) f.w[i] = ld8(bx + (TM + wm + i * 16 + l15) * 64 + c);
  };
  f32x4 acc[WI][XJ];
#pragma unroll
  for (int i = 0; i < WI; ++i)
#pragma unroll
    for (int j = 0; j < XJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto product = [&](const Frags& f, int i) {
    if (i >= WI) return;
#pragma unroll
    for (int j = 0; j < XJ; ++j) acc[i][j] = mma(f.w[i], f.x[j], acc[i][j]);
    __builtin_amdgcn_sched_barrier(0);
  };
  // until ``ahead`` steps of those asked for, the last, are still on the way
  auto wait = [&](int ahead) {
    if (S > 3 && ahead > 2)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * LOADS) : "memory");
    else if (S > 2 && ahead > 1)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LOADS) : "memory");
    else if (ahead > 0)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (!EXACT || s < steps)
#pragma unroll
      for (int i = 0; i < LOADS; ++i) load(s, s, i);
  wait(EXACT ? min(S, steps) - 1 : S - 1);
  asm volatile("s_barrier" ::: "memory");
  Frags f0, f1;
#pragma unroll
  for (int i = 0; i < MX; ++i) read(f0, 0, 0, i);
  int b = 0;                               // buffer of step k
  auto step = [&](int k, auto more) {
#pragma unroll
    for (int i = 0; i < MX; ++i) {
      read(f1, b, 1, i);
      product(f0, i);
    }
    // all waves have the second half of buffer b, which can be filled again,
    // and the loads of the next one have arrived
    if (more.value) wait(S - 2);
    else wait(min(S - 2, steps - 2 - k));
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int nb = b == S - 1 ? 0 : b + 1;
#pragma unroll
    for (int i = 0; i < MX; ++i) {
      read(f0, nb, 0, i);
      if (more.value) {
        load(k + S, b, i);
        if (MX + i < LOADS) load(k + S, b, MX + i);
      }
      product(f1, i);
    }
    b = nb;
  };
  int k = 0;
  for (; EXACT ? k + S < steps : k < steps; ++k) step(k, std::true_type{});
  if (EXACT)
    for (; k < steps; ++k) step(k, std::false_type{});
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // results 4 lg + 0..3 of a column group, of row l15
  constexpr int CI = EPI == ROWS_SWIGLU ? WI / 2 : WI;
#pragma unroll
  for (int j = 0; j < XJ; ++j) {
    const int r = xm + j * 16 + l15;
    if (r >= cnt) continue;
#pragma unroll
    for (int i = 0; i < CI; ++i) {
      const int n = n0 + (wid >> 1) * 16 * CI + i * 16 + 4 * lg;
      if (n >= N) continue;
      const long at = (long)(m0 + r) * N + n;
      if (EPI == ROWS_SWIGLU) {
        u16 v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float g = acc[i][j][e];
          v[e] = f2bf(g / (1.f + __expf(-g)) * acc[CI + i][j][e]);
        }
        __builtin_memcpy((u16*)outp + at, v, sizeof(v));
      } else if (EPI >= ROWS_BIAS) {
        u16 v[4], add[4];
        __builtin_memcpy(add, bias + n, sizeof(add));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float y = acc[i][j][e] + bf2f(add[e]);
          v[e] = f2bf(EPI == ROWS_GELU ? gelu_erf(y) : y);
        }
        __builtin_memcpy((u16*)outp + at, v, sizeof(v));
      } else {
        *(f32x4*)((float*)outp + (long)blockIdx.y * room * N + at) = acc[i][j];
      }
    }
  }
}

template <int XJ, int WI, int S, int EPI, bool ONCE, bool COUNTED = false>
void launch(void* out, const void* x, long xs, const void* w, int M, int N,
            int K, int parts, hipStream_t stream, const void* bias = nullptr,
            const int* count = nullptr) {
  constexpr int lds = S * 32 * (XJ + WI) * 128;
  constexpr int CN = EPI == ROWS_SWIGLU ? 16 * WI : 32 * WI;
  allow_lds(k_rows<XJ, WI, S, EPI, ONCE, COUNTED>, lds);
  const int nx = (N + CN - 1) / CN, nm = (M + 32 * XJ - 1) / (32 * XJ);
  hipLaunchKernelGGL((k_rows<XJ, WI, S, EPI, ONCE, COUNTED>),
                     dim3((nx * nm + 7) / 8 * 8, parts), dim3(256), lds, stream,
                     out, (const u16*)x, xs, (const u16*)w, (const u16*)bias, M,
                     N, K, nx, nm, count);
}

// Four buffers, but three for 128 rows of x and 64 of w, of which two blocks fit a
// CU then. 75 rows, 64 of w, three -> four: 4096 x 4096 in 4 parts 10.8 -> 10.0 us,
// 2 x 8192 x 2048 with SwiGLU 17.4 -> 15.4; 128 rows 7.6 -> 7.8 of 2048 x 2048.
template <int WI, int EPI>
void by_rows(int xj, void* out, const void* x, long xs, const void* w, int M,
             int N, int K, int parts, hipStream_t stream) {
#define GO(XJ, S)                                                             \
  M <= 32 * XJ                                                                \
      ? launch<XJ, WI, S, EPI, true>(out, x, xs, w, M, N, K, parts, stream)   \
      : launch<XJ, WI, S, EPI, false>(out, x, xs, w, M, N, K, parts, stream)
  if (xj == 2) GO(2, 4);
  else if (xj == 3) GO(3, 4);
  else GO(4, (WI == 2 ? 3 : 4));
#undef GO
}

// The sums of the parts of a product, added to a bfloat16 residual, and its RMS
// norm: what follows a product inside a layer. A row a block, 8 columns a thread
// at a time. 75 rows of 4096, 8 parts: 5.0 us, as long as the norm of a whole
// product took; latency of a launch and two passes over a row.
__global__ void __launch_bounds__(512)
k_parts_norm(u16* __restrict__ out, u16* __restrict__ res,
             const float* __restrict__ parts, int np,
             const u16* __restrict__ gain, int rows, int cols, float eps) {
  __shared__ float red[8];
  const int tid = threadIdx.x, nv = cols >> 3;
  const long row = blockIdx.x, step = (long)rows * cols;
  s16x8* rr = (s16x8*)(res + row * cols);
  float ss = 0.f;
  for (int i = tid; i < nv; i += 512) {
    const s16x8 old = rr[i];
    const float* p = parts + row * cols + i * 8;
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = 0.f;
#pragma unroll 4
    for (int k = 0; k < np; ++k) {
      const f32x8 q = ld8(p + k * step);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] += q[j];
    }
    s16x8 y;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const u16 b = f2bf(bf2f((u16)old[j]) + v[j]);
      y[j] = (short)b;
      ss = fmaf(bf2f(b), bf2f(b), ss);
    }
    rr[i] = y;
  }
  ss = wave_reduce_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  ss = 0.f;
#pragma unroll
  for (int k = 0; k < 8; ++k) ss += red[k];
  const float inv = rsqrtf(ss / (float)cols + eps);
  for (int i = tid; i < nv; i += 512) {
    const s16x8 v = rr[i], g = ((const s16x8*)gain)[i];
    s16x8 y;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      y[j] = (short)f2bf(bf2f((u16)v[j]) * inv * bf2f((u16)g[j]));
    ((s16x8*)(out + row * cols))[i] = y;
  }
}

// LayerNorm of the sum of the parts, a bias and a residual: what follows an
// encoder's product. A wave per row, V times 8 columns a lane; bound by the latency
// of a launch and of the parts, as the norm of a whole product is.
template <int V>
__global__ void __launch_bounds__(256)
k_parts_layernorm(u16* __restrict__ out, const float* __restrict__ parts, int np,
                  const u16* __restrict__ bias, const u16* __restrict__ res,
                  const u16* __restrict__ gain, const u16* __restrict__ shift,
                  int rows, int cols, float eps, const int* __restrict__ count) {
  const int lane = threadIdx.x & 63, nv = cols >> 3;
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= (count ? min(*count, rows) : rows)) return;
  const long step = (long)rows * cols;
  float v[V][8], sum = 0.f;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = lane + 64 * i;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[i][j] = 0.f;
    if (c >= nv) continue;
    const s16x8 r = ((const s16x8*)(res + row * cols))[c];
    const s16x8 b = ((const s16x8*)bias)[c];
    const float* p = parts + row * cols + c * 8;
#pragma unroll 4
    for (int k = 0; k < np; ++k) {
      const f32x8 q = ld8(p + k * step);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[i][j] += q[j];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[i][j] += bf2f((u16)b[j]) + bf2f((u16)r[j]);
      sum += v[i][j];
    }
  }
  const float mean = wave_reduce_sum(sum) / (float)cols;
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < V; ++i)
    if (lane + 64 * i < nv)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[i][j] -= mean;
        sq = fmaf(v[i][j], v[i][j], sq);
      }
  const float inv = rsqrtf(wave_reduce_sum(sq) / (float)cols + eps);
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = lane + 64 * i;
    if (c >= nv) continue;
    const s16x8 g = ((const s16x8*)gain)[c], b = ((const s16x8*)shift)[c];
    s16x8 y;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      y[j] = (short)f2bf(fmaf(v[i][j] * inv, bf2f((u16)g[j]), bf2f((u16)b[j])));
    ((s16x8*)(out + row * cols))[c] = y;
  }
}

// The parts of a product with the projections of q, k and v: q to rows of its own
// and k to the cache under RoPE, v to the cache. A thread takes dimensions
// 8 i .. 8 i + 7 of a head and their partners D/2 on; D % 16 == 0. 75 tokens, 32/8
// heads of 128, 4 parts: 4.8 us, for 3.4 to sum the parts and 3.5 for RoPE.
__global__ void __launch_bounds__(256)
k_rope_kv_parts(u16* __restrict__ q, const float* __restrict__ parts, int np,
                u16* __restrict__ kc, u16* __restrict__ vc,
                const float* __restrict__ cos_sin, const int* __restrict__ pos0,
                long units, long step, int S, int Hq, int Hkv, int D,
                int max_seq) {
  const int per = D / 16, heads = Hq + 2 * Hkv;
  const long u = (long)blockIdx.x * 256 + threadIdx.x;
  if (u >= units) return;
  const int i = (int)(u % per) * 8;
  const long th = u / per;                 // token and head
  const int h = (int)(th % heads);
  const long tok = th / heads;
  const int b = (int)(tok / S), p = pos0[b] + (int)(tok - (long)b * S);
  const float* src = parts + th * D + i;
  float x1[8], x2[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) x1[j] = x2[j] = 0.f;
#pragma unroll 4
  for (int k = 0; k < np; ++k) {
    const f32x8 a = ld8(src + k * step), c = ld8(src + k * step + D / 2);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      x1[j] += a[j];
      x2[j] += c[j];
    }
  }
  u16* dst;
  if (h < Hq) {
    dst = q + (tok * Hq + h) * D + i;
  } else {
    const int hk = h - Hq;
    dst = (hk < Hkv ? kc : vc) +
          (((long)b * Hkv + hk % Hkv) * max_seq + p) * D + i;
  }
  if (h < Hq + Hkv) {
    const float* cs = cos_sin + ((long)p * (D / 2) + i) * 2;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float a = x1[j], c = x2[j];
      x1[j] = a * cs[2 * j] - c * cs[2 * j + 1];
      x2[j] = c * cs[2 * j] + a * cs[2 * j + 1];
    }
  }
  s16x8 y1, y2;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    y1[j] = (short)f2bf(x1[j]);
    y2[j] = (short)f2bf(x2[j]);
  }
  *(s16x8*)dst = y1;
  *(s16x8*)(dst + D / 2) = y2;
}

// The sums of the parts, times a scale, added to float32.
__global__ void __launch_bounds__(256)
k_parts_add(float* __restrict__ out, const float* __restrict__ parts, int np,
            long n4, float scale) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < np; ++k) {
    const f32x4 q = ((const f32x4*)parts)[k * n4 + i];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += q[e];
  }
  f32x4 y = ((f32x4*)out)[i];
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = fmaf(scale, v[e], y[e]);
  ((f32x4*)out)[i] = y;
}

// The same, and both norms of the new rows (o2 may be null): what follows the product
// that ends a layer. A row a block, four columns a thread and turn, of which four turns
// stay in registers. 1301 rows of 2048, 4 parts: in two launches 11 us and 7; bound by
// reading the parts, at 5 TB/s.
__global__ void __launch_bounds__(256)
k_parts_add_norms(u16* __restrict__ o1, u16* __restrict__ o2,
                  float* __restrict__ x, const float* __restrict__ parts, int np,
                  const float* __restrict__ w1, const float* __restrict__ w2,
                  long step, int C, float scale, float eps) {
  constexpr int KEEP = 4;
  __shared__ float red[4];
  const int tid = threadIdx.x, nv = C >> 2;
  const long row = blockIdx.x;
  f32x4* xr = (f32x4*)(x + row * C);
  const f32x4* pr = (const f32x4*)(parts + row * C);
  float ss = 0.f;
  auto add = [&](int i) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int k = 0; k < np; ++k) {
      const f32x4 q = pr[k * (step >> 2) + i];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += q[e];
    }
    f32x4 y = xr[i];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[e] = fmaf(scale, v[e], y[e]);
      ss = fmaf(y[e], y[e], ss);
    }
    xr[i] = y;
    return y;
  };
  f32x4 y[KEEP];
#pragma unroll
  for (int k = 0; k < KEEP; ++k)
    if (tid + k * 256 < nv) y[k] = add(tid + k * 256);
  for (int i = tid + KEEP * 256; i < nv; i += 256) add(i);
  ss = block_reduce_sum(ss, red);
  const float inv = 1.f / sqrtf(ss / (float)C + eps);
  auto norm = [&](int i, f32x4 v) {
    const f32x4 a = ((const f32x4*)w1)[i];
    u16 t[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) t[e] = El<u16>::st(v[e] * inv * a[e]);
    __builtin_memcpy(o1 + row * C + i * 4, t, sizeof(t));
    if (o2) {
      const f32x4 b = ((const f32x4*)w2)[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) t[e] = El<u16>::st(v[e] * inv * b[e]);
      __builtin_memcpy(o2 + row * C + i * 4, t, sizeof(t));
    }
  };
#pragma unroll
  for (int k = 0; k < KEEP; ++k)
    if (tid + k * 256 < nv) norm(tid + k * 256, y[k]);
  for (int i = tid + KEEP * 256; i < nv; i += 256) norm(i, xr[i]);
}

}  // namespace

extern "C" {

// K % 64 == 0 and at least 64 a part, N % 4 == 0; rows of x (xs apart) and w on 16
// bytes. xj: 32 rows of x a tile, 2 to 4; wide: 128 rows of w a tile, else 64.
// swiglu: bfloat16 [M, N] of one part; else float32 [parts, M, N].
void fei_rows(void* out, const void* x, long xs, const void* w, int M, int N,
              int K, int swiglu, int xj, int wide, int parts,
              hipStream_t stream) {
#define ROWS(E)                                                            \
  wide ? by_rows<4, E>(xj, out, x, xs, w, M, N, K, parts, stream)       \
       : by_rows<2, E>(xj, out, x, xs, w, M, N, K, parts, stream)
  if (swiglu) ROWS(ROWS_SWIGLU);
  else ROWS(ROWS_PARTS);
#undef ROWS
}

// The same sizes; out [M, N] bfloat16 with a bias per column, and GELU of it. Tiles
// of 64 x 64: an encoder's products are small (12 to 48 of these tiles for 64
// rows), and what counts is that many CUs load.
void fei_rows_bias(void* out, const void* x, const void* w, const void* bias,
                   int M, int N, int K, int gelu, hipStream_t stream) {
  if (gelu)
    launch<2, 2, 3, ROWS_GELU, false>(out, x, K, w, M, N, K, 1, stream, bias);
  else
    launch<2, 2, 3, ROWS_BIAS, false>(out, x, K, w, M, N, K, 1, stream, bias);
}

// Of as many of the M rows as the device finds at ``count``.
void fei_rows_bias_of(void* out, const void* x, const void* w, const void* bias,
                      int M, int N, int K, int gelu, const int* count,
                      hipStream_t stream) {
  if (gelu)
    launch<2, 2, 3, ROWS_GELU, false, true>(out, x, K, w, M, N, K, 1, stream,
                                            bias, count);
  else
    launch<2, 2, 3, ROWS_BIAS, false, true>(out, x, K, w, M, N, K, 1, stream,
                                            bias, count);
}

// Float32 [parts, M, N] of as many, in tiles of 64 x 64.
void fei_rows_parts_of(float* out, const void* x, const void* w, int M, int N,
                       int K, int parts, const int* count, hipStream_t stream) {
  launch<2, 2, 4, ROWS_PARTS, false, true>(out, x, K, w, M, N, K, parts, stream,
                                           nullptr, count);
}

void fei_parts_norm(void* out, void* res, const float* parts, int np,
                    const void* gain, int rows, int cols, float eps,
                    hipStream_t stream) {
  hipLaunchKernelGGL(k_parts_norm, dim3(rows), dim3(512), 0, stream, (u16*)out,
                     (u16*)res, parts, np, (const u16*)gain, rows, cols, eps);
}

// cols % 8 == 0, at most 2048; out may be none of the inputs; count as above
void fei_parts_layernorm_of(void* out, const float* parts, int np,
                            const void* bias, const void* res, const void* gain,
                            const void* shift, int rows, int cols, float eps,
                            const int* count, hipStream_t stream) {
#define GO(V)                                                                \
  hipLaunchKernelGGL(k_parts_layernorm<V>, dim3((rows + 3) / 4), dim3(256), 0, \
                     stream, (u16*)out, parts, np, (const u16*)bias,          \
                     (const u16*)res, (const u16*)gain, (const u16*)shift,    \
                     rows, cols, eps, count)
  if (cols <= 1024) GO(2); else GO(4);
#undef GO
}

void fei_parts_layernorm(void* out, const float* parts, int np,
                         const void* bias, const void* res, const void* gain,
                         const void* shift, int rows, int cols, float eps,
                         hipStream_t stream) {
  fei_parts_layernorm_of(out, parts, np, bias, res, gain, shift, rows, cols, eps,
                         nullptr, stream);
}

// parts [np][B * S][(Hq + 2 Hkv) * D], q [B * S][Hq][D]; D % 16 == 0, all on 16
// bytes
void fei_rope_kv_parts(void* q, const float* parts, int np, void* k_cache,
                       void* v_cache, const float* cos_sin, const int* pos0,
                       int B, int S, int Hq, int Hkv, int D, int max_seq,
                       hipStream_t stream) {
  const long rows = (long)B * S * (Hq + 2 * Hkv), units = rows * (D / 16);
  hipLaunchKernelGGL(k_rope_kv_parts, dim3((units + 255) / 256), dim3(256), 0,
                     stream, (u16*)q, parts, np, (u16*)k_cache, (u16*)v_cache,
                     cos_sin, pos0, units, rows * D, S, Hq, Hkv, D, max_seq);
}

// out += scale * the sums; n % 4 == 0 values a part, all on 16 bytes
void fei_parts_add(float* out, const float* parts, int np, long n, float scale,
                   hipStream_t stream) {
  hipLaunchKernelGGL(k_parts_add, dim3((n / 4 + 255) / 256), dim3(256), 0,
                     stream, out, parts, np, n / 4, scale);
}

// x [rows, C] float32 += scale * the sums, and its norms with gains w1 and w2 in
// bfloat16 (o2, w2 may be null); C % 4 == 0, all on 16 bytes, o1 and o2 on 8
void fei_parts_add_norms(void* o1, void* o2, float* x, const float* parts,
                         int np, const float* w1, const float* w2, int rows,
                         int C, float scale, float eps, hipStream_t stream) {
  hipLaunchKernelGGL(k_parts_add_norms, dim3(rows), dim3(256), 0, stream,
                     (u16*)o1, (u16*)o2, x, parts, np, w1, w2, (long)rows * C, C,
                     scale, eps);
}

}  // extern "C"
