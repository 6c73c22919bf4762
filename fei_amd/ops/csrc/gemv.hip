// Products of few rows with a weight matrix, the decode step's (gfx950):
// out[M, N] = x[M, K] @ W[N, K]^T, F.linear's layout.
//
// k_gemv streams the weights, bfloat16 or fp8 (e4m3fn, a scale per row), through
// the vector units; from M = 2 on k_skinny (below) uses the matrix units.
#include <type_traits>

#include "fei_epilogue.h"
#include "fei_mma.h"

namespace {


enum { GEMV_BF16 = 0, GEMV_RES = 1, GEMV_SWIGLU = 2 };

// Decode attention of one row that its product sums itself: what the splits of the keys
// left (attn_decode.hip), [heads][splits][D] and their maxima (of exponents of 2) and sums,
// [heads][splits][2]; keys: of a split. Of so few keys that one split had them all, x
// has the result.
struct Splits {
  const float *po, *pml;
  const int* pos;
  int splits, room, keys, D;
};

// A wave streams two rows of w, 4 loads of 16 bytes a lane from each at a time
// and the next 4 before it uses them; all waves of a product are on the chip at
// once, so what counts is how soon their loads are out and how many. x goes to
// LDS meanwhile: its loads are issued first (loads come back in order), and the
// barriers leave the weights in flight. NORM: x is a residual under an RMS norm
// with gains, which the block takes on the way to LDS (rounded to bfloat16 there,
// as a norm kernel's result is). KS = 4: the block's waves share two rows. LDS = false:
// x from L1/L2, for rows that LDS has no room for. GEMV_RES adds to out in
// place; GEMV_SWIGLU: w has N rows of gates, then N of up, a wave takes a pair.
// ssq (may be null): with GEMV_RES gets the sums of squares of the new rows
// added, with NORM has those of x.
//
// Bound by HBM and, at decode sizes, by the 3 us that a launch and the first
// loads take. In a graph of launches over cold weights, M = 1, against two rows
// a wave in plain loops (and for NORM a norm's launch of 4.6 us in front):
// 6144 x 4096 with norm 10.8 us (9.7 + 4.6), 4096 x 4096 7.8 (7.9),
// 2 x 14336 x 4096 SwiGLU with norm 36.8 (36.3 + 4.6), 4096 x 14336 20.8
// (24.9), 128256 x 4096 151 (165). fp8: 7.1 (10), 5.7 (6.5), 20.4 (44.5),
// 13.7 (13). Two or eight loads a row in flight, four rows a wave, or rows
// shared by 2 waves are slower at nearly every size.
//
// NS: x is the sum of up to NS splits of the keys, which every block makes for itself:
// a launch less, and the weights are on the way meanwhile. For up to XS * 2048 columns.
// All blocks read all splits, 4 bytes a column, from the L2s: whole decoding steps, us, 16
// layers of 2048, 300 keys (3 splits) 685 -> 652, 1000 (8) 703 -> 670, 2000 (16) 702 ->
// 692; 32 layers of 4096, three runs of either in turn, which differ by 2 to 4, 300 keys
// 2889 -> 2871, 512 (5) 2896 -> 2887, 600 2896 -> 2890, 700 (6) 2890 -> 2899, which is left
// to the launch; fp8 weights, 300 keys 1889 -> 1849, 512 1892 -> 1864.
template <int M, int KS, bool NORM, int EPI, bool FP8, bool LDS, int NS = 0,
          int XS = 1>
__device__ __forceinline__ void
gemv(u16* __restrict__ out, const u16* __restrict__ x,
     const u16* __restrict__ gain, const void* __restrict__ wp,
     const float* __restrict__ wscale, int N, int K, float eps,
     float* __restrict__ ssq, const Splits* sp) {
  constexpr int E = FP8 ? 16 : 8;          // weights of a 16-byte load
  constexpr int U = KS > 1 ? 2 : 4;        // loads of a row in flight
  constexpr int R = 2;                     // rows of w
  constexpr int WV = 4 / KS;               // waves side by side
  extern __shared__ __align__(16) u16 xs[];   // the rows, normed
  __shared__ float red[4][M];
  __shared__ float part[KS > 1 ? 4 : 1][R][M];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ks = KS > 1 ? wid % KS : 0;
  // SWIGLU: half of a wave's rows are gates, the others the same of up
  constexpr int RO = EPI == GEMV_SWIGLU ? R / 2 : R;     // results per wave
  const int n0 = (blockIdx.x * WV + wid / KS) * RO;
  const u32x4* w[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    long n = min(n0 + r % RO, N - 1);
    if (EPI == GEMV_SWIGLU && r >= RO) n += N;
    w[r] = (const u32x4*)((const char*)wp + n * K * (FP8 ? 1 : 2));
  }
  const int nv = K / E;                    // loads of a row
  const int per = KS > 1 ? ((nv + 63) / 64 + KS - 1) / KS * 64 : nv;
  const int lo = ks * per, hi = KS > 1 ? min(nv, lo + per) : nv;
  // x first: loads come back in order
  constexpr int XV = NS ? XS : NORM && M == 1 ? 4 : 8;
  const int nx = M * (K / 8);
  s16x8 x0[XV], g0[NORM ? XV : 1];
  auto gain_at = [&](int c) {
    return ((const s16x8*)gain)[M == 1 ? c : c % (K / 8)];
  };
  f32x4 po[NS ? XS : 1][NS ? NS : 1][2];
  f32x2 ml[NS ? XS : 1][NS ? NS : 1];
  int used = 0;
  if constexpr (NS > 0) {
#pragma unroll
    for (int i = 0; i < XS; ++i) {
      const int c = min(tid + i * 256, nx - 1), head = c * 8 / sp->D;
      x0[i] = ((const s16x8*)x)[c];
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const long at = (long)head * sp->splits + min(s, sp->splits - 1);
        ml[i][s] = ((const f32x2*)sp->pml)[at];
        const f32x4* p = (const f32x4*)(sp->po + at * sp->D + (c * 8 & (sp->D - 1)));
        po[i][s][0] = p[0];
        po[i][s][1] = p[1];
      }
    }
    const int n = min(*sp->pos + 1, sp->room);
    used = min(sp->splits, (n + sp->keys - 1) / sp->keys);
  } else {
#pragma unroll
    for (int i = 0; LDS && i < XV; ++i) {
      const int c = min(tid + i * 256, nx - 1);
      x0[i] = ((const s16x8*)x)[c];
      if (NORM) g0[i] = gain_at(c);
    }
  }
  u32x4 v[U][R], nxt[U][R];
  auto fetch = [&](u32x4 (&d)[U][R], int i0) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int r = 0; r < R; ++r)
        d[u][r] = __builtin_nontemporal_load(w[r] + i0 + u * 64 + lane);
  };
  auto fetch_tail = [&](u32x4 (&d)[U][R], int i0) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (i0 + u * 64 + lane < hi)
          d[u][r] = __builtin_nontemporal_load(w[r] + i0 + u * 64 + lane);
  };
  auto get = [&](u32x4 (&d)[U][R], int i0) {
    if (i0 + U * 64 <= hi) fetch(d, i0);
    else if (i0 < hi) fetch_tail(d, i0);
  };
  get(v, lo);
  float inv[M];
  if (NORM) {
    float ss[M];
#pragma unroll
    for (int m = 0; m < M; ++m) ss[m] = 0.f;
    auto square = [&](int c, s16x8 xv) {
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float f = bf2f((u16)xv[j]);
        s = fmaf(f, f, s);
      }
#pragma unroll
      for (int m = 0; m < M; ++m)
        ss[m] += M == 1 || c / (K / 8) == m ? s : 0.f;
    };
#pragma unroll
    for (int i = 0; i < XV; ++i)
      if (tid + i * 256 < nx) square(tid + i * 256, x0[i]);
    for (int c = tid + XV * 256; c < nx; c += 256)
      square(c, ((const s16x8*)x)[c]);
#pragma unroll
    for (int m = 0; m < M; ++m) {
      ss[m] = wave_sum(ss[m]);
      if (lane == 0) red[wid][m] = ss[m];
    }
    // not __syncthreads: the weights stay in flight
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int m = 0; m < M; ++m)
      inv[m] = rsqrtf((ssq ? ssq[m] : red[0][m] + red[1][m] + red[2][m] +
                                          red[3][m]) / (float)K + eps);
  }
  if constexpr (NS > 0) {
    if (used != 1)
#pragma unroll
      for (int i = 0; i < XS; ++i) {
        float m = -3.0e38f, l = 0.f, v[8];
#pragma unroll
        for (int s = 0; s < NS; ++s)
          if (s < used) m = fmaxf(m, ml[i][s][0]);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = 0.f;
#pragma unroll
        for (int s = 0; s < NS; ++s)
          if (s < used) {                  // what lies there else is not used
            const float f = __builtin_amdgcn_exp2f(ml[i][s][0] - m);
            l = fmaf(f, ml[i][s][1], l);
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = fmaf(f, po[i][s][j >> 2][j & 3], v[j]);
          }
        const float r = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) x0[i][j] = (short)El<u16>::st(v[j] * r);
      }
  }
  auto stage = [&](int c, s16x8 xv, s16x8 gv) {
    if (NORM) {
      float f = inv[0];
#pragma unroll
      for (int m = 1; m < M; ++m) f = c / (K / 8) == m ? inv[m] : f;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        xv[j] = (short)El<u16>::st(bf2f((u16)xv[j]) * f * bf2f((u16)gv[j]));
    }
    ((s16x8*)xs)[c] = xv;
  };
#pragma unroll
  for (int i = 0; LDS && i < XV; ++i)
    if (tid + i * 256 < nx) stage(tid + i * 256, x0[i], g0[NORM ? i : 0]);
  for (int c = tid + XV * 256; LDS && c < nx; c += 256)
    stage(c, ((const s16x8*)x)[c], NORM ? gain_at(c) : x0[0]);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

  float acc[R][M];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int m = 0; m < M; ++m) acc[r][m] = 0.f;
  auto dot = [&](const u32x4 (&d)[R], int i) {
#pragma unroll
    for (int m = 0; m < M; ++m) {
      s16x8 xv[E / 8];
#pragma unroll
      for (int q = 0; q < E / 8; ++q)
        xv[q] = ld8((LDS ? xs : x) + (long)m * K + i * E + q * 8);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (FP8) {
          float s = 0.f;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const u32 t = d[r][q];
            const f32x2 a = __builtin_amdgcn_cvt_pk_f32_fp8(t, false);
            const f32x2 b = __builtin_amdgcn_cvt_pk_f32_fp8(t, true);
            const s16x8 y = xv[q / 2 * (E / 8 - 1)];
            s = fmaf(a[0], bf2f((u16)y[q % 2 * 4]), s);
            s = fmaf(a[1], bf2f((u16)y[q % 2 * 4 + 1]), s);
            s = fmaf(b[0], bf2f((u16)y[q % 2 * 4 + 2]), s);
            s = fmaf(b[1], bf2f((u16)y[q % 2 * 4 + 3]), s);
          }
          acc[r][m] += s;
        } else {
          acc[r][m] += dot8_bf16(xv[0], __builtin_bit_cast(s16x8, d[r]));
        }
      }
    }
  };
  for (int i0 = lo; i0 < hi; i0 += U * 64) {
    get(nxt, i0 + U * 64);
    if (i0 + U * 64 <= hi) {
#pragma unroll
      for (int u = 0; u < U; ++u) dot(v[u], i0 + u * 64 + lane);
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (i0 + u * 64 + lane < hi) dot(v[u], i0 + u * 64 + lane);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int r = 0; r < R; ++r) v[u][r] = nxt[u][r];
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int m = 0; m < M; ++m) acc[r][m] = wave_sum(acc[r][m]);
  if (KS > 1) {
    if (lane == 0) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) part[wid][r][m] = acc[r][m];
    }
    __syncthreads();
    if (ks) return;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int m = 0; m < M; ++m) {
        acc[r][m] = part[wid][r][m];
#pragma unroll
        for (int k = 1; k < KS; ++k) acc[r][m] += part[wid + k][r][m];
      }
  }
  if (lane) return;
  float sq[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    sq[m] = 0.f;
#pragma unroll
    for (int r = 0; r < RO; ++r) {
      const int n = n0 + r;
      if (n >= N) break;
      float y = acc[r][m];
      if (FP8) y *= wscale[n];
      u16* o = out + (long)m * N + n;
      if (EPI == GEMV_SWIGLU) {
        float u = acc[r + R - RO][m];
        if (FP8) u *= wscale[n + N];
        *o = f2bf(y / (1.f + __expf(-y)) * u);
      } else if (EPI == GEMV_RES) {
        const u16 t = f2bf(bf2f(*o) + y);
        *o = t;
        sq[m] = fmaf(bf2f(t), bf2f(t), sq[m]);
      } else {
        *o = f2bf(y);
      }
    }
    if (EPI == GEMV_RES && ssq) atomicAdd(&ssq[m], sq[m]);
  }
}

template <int M, int KS, bool NORM, int EPI, bool FP8, bool LDS>
__global__ void __launch_bounds__(256)
k_gemv(u16* __restrict__ out, const u16* __restrict__ x,
       const u16* __restrict__ gain, const void* __restrict__ wp,
       const float* __restrict__ wscale, int N, int K, float eps,
       float* __restrict__ ssq) {
  gemv<M, KS, NORM, EPI, FP8, LDS>(out, x, gain, wp, wscale, N, K, eps, ssq,
                                   nullptr);
}

// The output product of an attention, added to a residual: see Splits.
template <bool FP8, int NS, int XS>
__global__ void __launch_bounds__(256)
k_gemv_splits(u16* __restrict__ out, const u16* __restrict__ x,
              const void* __restrict__ wp, const float* __restrict__ wscale, int N,
              int K, const Splits sp) {
  gemv<1, 1, false, GEMV_RES, FP8, true, NS, XS>(out, x, nullptr, wp, wscale, N, K,
                                                 0.f, nullptr, &sp);
}

template <int M, bool NORM, int EPI, bool FP8>
void launch_gemv(void* out, const void* x, const void* gain, const void* w,
                 const float* wscale, int N, int K, float eps, float* ssq,
                 hipStream_t stream) {
  const size_t lds = (size_t)M * K * 2;
  auto go = [&](auto kernel, int blocks, size_t bytes) {
    allow_lds(kernel, bytes);
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), bytes, stream,
                       (u16*)out, (const u16*)x, (const u16*)gain, w, wscale,
                       N, K, eps, ssq);
  };
  const int per = EPI == GEMV_SWIGLU ? 4 : 8;          // results per block
  if constexpr (!NORM) {
    if (lds > 65536)
      return go(k_gemv<M, 1, false, EPI, FP8, false>, (N + per - 1) / per, 0);
    // Few long rows: a wave per two rows would be one per SIMD. 2048 x 8192:
    // 8.4 us against 9.1 (fp8 5.7, 6.8); 2048 x 2048: 4.5 against 4.3.
    if constexpr (EPI != GEMV_SWIGLU)
      if (N <= 2048 && K >= 4096)
        return go(k_gemv<M, 4, false, EPI, FP8, true>, (N + 1) / 2, lds);
  }
  go(k_gemv<M, 1, NORM, EPI, FP8, true>, (N + per - 1) / per, lds);
}

// Cache prefetch: stream a weight region through normal (cache-filling)
// loads so a LATER kernel's reads hit L2/L3 instead of HBM. Launched on a
// side stream during low-bandwidth phases (decode attention) to convert
// idle HBM cycles into prefill of the next GEMV's operand. The impossible
// store defeats dead-code elimination; nothing is written in practice.
__global__ void __launch_bounds__(256)
k_prefetch(const u16* __restrict__ w, long n_vec8, float* __restrict__ sink) {
  float acc = 0.f;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n_vec8;
       i += (long)gridDim.x * blockDim.x) {
    const s16x8 v = ((const s16x8*)w)[i];
    acc += (float)(short)v[0];
  }
  if (acc == 1.0f / 0.0f) sink[0] = acc;
}

}  // namespace

extern "C" {

// epi: what becomes of the sums (see above). gain null: no norm. wscale null:
// bfloat16 weights. M is 1, 2, 3, 4 or 8; with a norm M * K * 2 is at most
// 128 KB (the callers see to both).
void fei_gemv(void* out, const void* x, const void* gain, const void* w,
              const float* wscale, int M, int N, int K, float eps, int epi,
              float* ssq, hipStream_t stream) {
  auto run = [&](auto m, auto norm, auto e, auto fp8) {
    launch_gemv<m.value, norm.value, e.value, fp8.value>(
        out, x, gain, w, wscale, N, K, eps, ssq, stream);
  };
  auto by_weights = [&](auto m, auto norm, auto e) {
    if (wscale) run(m, norm, e, std::true_type{});
    else run(m, norm, e, std::false_type{});
  };
  auto by_rows = [&](auto norm, auto e) {
    switch (M) {
      case 1: return by_weights(std::integral_constant<int, 1>{}, norm, e);
      case 2: return by_weights(std::integral_constant<int, 2>{}, norm, e);
      case 3: return by_weights(std::integral_constant<int, 3>{}, norm, e);
      case 4: return by_weights(std::integral_constant<int, 4>{}, norm, e);
      case 8: return by_weights(std::integral_constant<int, 8>{}, norm, e);
      default: return;
    }
  };
  auto by_epi = [&](auto norm) {
    if (epi == GEMV_RES)
      by_rows(norm, std::integral_constant<int, GEMV_RES>{});
    else if (epi == GEMV_SWIGLU)
      by_rows(norm, std::integral_constant<int, GEMV_SWIGLU>{});
    else
      by_rows(norm, std::integral_constant<int, GEMV_BF16>{});
  };
  if (gain) by_epi(std::true_type{});
  else by_epi(std::false_type{});
}

// out [1, N] += the attention that ``left`` splits of ``keys`` keys each left in po and
// pml, where each head has room for ``splits``, (or, one that had all keys, in x) times w
// [N, K], heads of D one behind another. K up to 2048 and 16 left, or up to 4096 and 5
// (which fei_attn_decode_product sees to). K % 8 == 0, D a power of two.
void fei_gemv_splits(void* out, const void* x, const void* w, const float* wscale,
                     int N, int K, const float* po, const float* pml,
                     const int* pos, int splits, int left, int room, int keys,
                     int D, hipStream_t stream) {
  const Splits sp{po, pml, pos, splits, room, keys, D};
  auto run = [&](auto ns, auto xs) {
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((N + 7) / 8), dim3(256), K * 2, stream,
                         (u16*)out, (const u16*)x, w, wscale, N, K, sp);
    };
    if (wscale) go(k_gemv_splits<true, ns.value, xs.value>);
    else go(k_gemv_splits<false, ns.value, xs.value>);
  };
  const std::integral_constant<int, 1> one{};
  const std::integral_constant<int, 2> two{};
  const std::integral_constant<int, 4> four{};
  if (K <= 2048) {
    if (left <= 2) run(two, one);
    else if (left <= 4) run(four, one);
    else if (left <= 8) run(std::integral_constant<int, 8>{}, one);
    else run(std::integral_constant<int, 16>{}, one);
  } else {
    if (left <= 2) run(two, two);
    else if (left <= 4) run(four, two);
    else run(std::integral_constant<int, 5>{}, two);
  }
}

void fei_prefetch(const void* w, long bytes, void* sink, int n_blocks,
                  hipStream_t stream) {
  const long n_vec8 = bytes / 16;
  if (n_vec8 <= 0) return;
  hipLaunchKernelGGL(k_prefetch, dim3(n_blocks), dim3(256), 0, stream,
                     (const u16*)w, n_vec8, (float*)sink);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// The same for 2 to 64 rows on the matrix units. The block's four waves share K;
// a wave streams 16 RT rows of w and the rows of x, 64 of K a stage, S stages
// ahead, by direct loads into LDS of its own, so that nothing but the sum at the
// end has a barrier. A load takes 8 whole lines of 128 bytes (fragments read
// from memory directly, 16 lanes on 16 rows, come one lane a cycle: 4096 x 4096
// in 9.6 us, 28672 x 4096 in 52); the 16-byte places of a row are permuted by
// the row, so that the fragment reads spread over the banks.
//
// Bound by HBM, and with many rows by the loads of x, of which a block repeats
// all. Measured with cold weights in a graph, 8 rows, against tiles through
// registers with 4 KB a wave in flight: 6144 x 4096 16.0 -> 10.6 us, 4096 x 4096
// 10.3 -> 7.8, 28672 x 4096 53 -> 41, 4096 x 14336 29 -> 20.2, 128256 x 4096 190
// -> 172. 20 rows, against the library: 3072 x 2048 11.9 -> 5.8, 2048 x 2048
// 10.9 -> 5.5, 16384 x 2048 17.6 -> 14.6, 2048 x 8192 14.9 -> 13.7.
namespace {

// The RMS norm of x inside the product, from the sums of squares that the
// product before left.
struct SkinnyNorm {
  const u16* gain;     // null: none
  const float* sums;   // [M, tiles], together of all columns of x
  int tiles;
  float eps;
  float* sums_out;     // EPI_RES_BF16: the same of the new rows; may be null. With
                       // tiles of N / 8 they are of 8 columns each
};

// XL: groups of 8 rows of x. N: results a row of x; with EPI_SWIGLU w has N
// rows of gates, then N of up, and half of a wave's tiles are either. NORM: x is
// a residual; its fragments take the gains on the way to the matrix units (rounded
// then, as a norm kernel would), the sums the root mean square. 8 rows, 28672 x
// 4096: 42 us for 41 and a norm's launch of 4.8; normed in full before the
// products, with the root mean square waited for, it was 46; with the gains
// through registers, before the first stages could be asked for, 43.
template <int EPI, int XL, int RT, int S, bool NORM>
__global__ void __launch_bounds__(256)
k_skinny(void* __restrict__ outp, const u16* __restrict__ x,
         const u16* __restrict__ w, int M, int N, int K, Epilogue ep,
         SkinnyNorm nm) {
  constexpr int MT = (XL + 1) / 2;
  constexpr int WL = RT ? 2 * RT : 1, FR = RT ? RT : 1;  // loads, fragments of w
  constexpr int LOADS = WL + XL, STAGE = LOADS * 512;
  constexpr int RO = EPI == EPI_SWIGLU ? RT / 2 : FR;
  extern __shared__ __align__(16) u16 buf[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, lg = lane >> 4;
  const int n0 = blockIdx.x * (RT ? 16 * RO : 8);
  const int r8 = lane >> 3, c8 = ((lane & 7) ^ r8) * 8;
  const int steps = K / 64, per = (steps + 3) / 4;
  const int lo = min(wid * per, steps - 1);
  const int n = max(min(steps, (wid + 1) * per) - wid * per, 0);
  // blocks start at different steps: rows often lie a multiple of 4 KB apart,
  // and the same columns of all of them would be on the same memory channels (a
  // decoding step of 8 rows, 32 layers of 4096: 3669 -> 3422 us). Two blocks of 8 columns
  // start where one of 16 does, so that either gives the same bits
  const int turn = n ? blockIdx.x / (RT ? 1 : 2) * 3 % n : 0;
  auto at = [&](int s) {
    const int t = s + turn;
    return lo + (t < n ? t : t - n);
  };
  const u16* src[LOADS];
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    long row = min(n0 + i % (2 * RO) * 8 + r8, N - 1);
    if (i >= 2 * RO) row += N;
    src[i] = w + row * K + c8;
  }
#pragma unroll
  for (int i = 0; i < XL; ++i)
    src[WL + i] = x + (long)min(i * 8 + r8, M - 1) * K + c8;
  u16* mine = buf + wid * S * STAGE;
  const u32 lds = (u32)(uintptr_t)(__attribute__((address_space(3))) u16*)mine;
  // nothing is asked for past the end: a wave often has few more stages than it asks
  // for at first, and stages read again there are waited for in the end (32 layers of
  // 4096, 8 rows: 3410 -> 3260 us a step; 16 of 2048, 20 rows: 1178 -> 1124)
  auto load = [&](int step, int b) {
    if (step >= n) return;
    const int k = at(step) * 64;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const u32 to = lds + (b * STAGE + i * 512) * 2;
      if (i < WL) load_lds_nt(src[i] + k, to);
      else load_lds(src[i] + k, to);
    }
  };
  f32x4 acc[FR][MT];
#pragma unroll
  for (int i = 0; i < FR; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // NORM: the gains go behind the stages; the sums of squares (of rows wid, wid
  // + 4, ..) are asked for first and used last
  const u16* gs = buf + 4 * S * STAGE;
  constexpr int NR = NORM ? 2 * XL : 1;
  float raw[NR][4];
  if (NORM) {
#pragma unroll
    for (int i = 0; i < NR; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        raw[i][t] = nm.sums[(long)min(wid + 4 * i, M - 1) * nm.tiles +
                            min(lane + 64 * t, nm.tiles - 1)];
    // 1 KB a load, to the end of a whole one
    const u32 to = (u32)(uintptr_t)(__attribute__((address_space(3))) u16*)gs;
    for (int i = wid * 512; i < K; i += 2048)
      load_lds(nm.gain + min(i + lane * 8, K - 8), to + i * 2);
  }
#pragma unroll
  for (int s = 0; s < S; ++s) load(s, s);
  // until ``stages`` of those asked for, the last, are still on the way
  auto wait = [&](int stages) {
    if (S > 3 && stages > 2)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * LOADS) : "memory");
    else if (S > 2 && stages > 1)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LOADS) : "memory");
    else if (stages > 0)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };
  // the gains of all waves; the stages stay in flight
  if (NORM) {
    if (n >= S)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S * LOADS) : "memory");
    else
      wait(n);
    asm volatile("s_barrier" ::: "memory");
  }
  int b = 0;
  for (int s = 0; s < n; ++s) {
    wait(min(S, n - s) - 1);
    const u16* bw = mine + b * STAGE;
    const u16* bx = bw + WL * 512;
    s16x8 fa[2][FR], fb[2][MT];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int c = ((kk * 4 + lg) ^ (l15 & 7)) * 8;
#pragma unroll
      for (int i = 0; i < FR; ++i)     // 8 rows stand for the next 8 as well
        fa[kk][i] = ld8(bw + (i * 16 + (RT ? l15 : l15 & 7)) * 64 + c);
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        // an odd group of 8 rows stands in for the one after it
        const int r = XL >= 2 * j + 2 ? l15 : l15 & 7;
        fb[kk][j] = ld8(bx + (j * 16 + r) * 64 + c);
      }
    }
    s16x8 fg[2];
    if (NORM)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
        fg[kk] = ld8(gs + at(s) * 64 + (kk * 4 + lg) * 8);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    load(s + S, b);
    if (NORM)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
          for (int e = 0; e < 8; e += 2) {
            typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
            typedef __attribute__((ext_vector_type(2))) short s16x2;
            const f32x2 v = {bf2f((u16)fb[kk][j][e]) * bf2f((u16)fg[kk][e]),
                             bf2f((u16)fb[kk][j][e + 1]) *
                                 bf2f((u16)fg[kk][e + 1])};
            const s16x2 y = __builtin_bit_cast(
                s16x2, __builtin_convertvector(v, bf16x2));
            fb[kk][j][e] = y[0];
            fb[kk][j][e + 1] = y[1];
          }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int i = 0; i < FR; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j)
          acc[i][j] = mma(fa[kk][i], fb[kk][j], acc[i][j]);
    b = b == S - 1 ? 0 : b + 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __shared__ float sinv[NORM ? XL * 8 : 1];
  if (NORM) {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      float ss = 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (lane + 64 * t < nm.tiles) ss += raw[i][t];
      for (int t = lane + 256; t < nm.tiles; t += 64)
        ss += nm.sums[(long)min(wid + 4 * i, M - 1) * nm.tiles + t];
      ss = wave_sum(ss);
      if (lane == 0) sinv[wid + 4 * i] = rsqrtf(ss / (float)K + nm.eps);
    }
  }
  __syncthreads();
  f32x4* red = (f32x4*)buf;
#pragma unroll
  for (int i = 0; i < FR; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j)
      red[((i * MT + j) * 4 + wid) * 64 + lane] = acc[i][j];
  __syncthreads();
  auto sum = [&](int t) {
    const f32x4* p = red + t * 256 + lane;
    f32x4 v = p[0];
#pragma unroll
    for (int k = 1; k < 4; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += p[k * 64][e];
    return v;
  };
  // results 4 lg + 0..3 of a tile, of row l15
  for (int t = wid; t < RO * MT; t += 4) {
    const int m = t % MT * 16 + l15, n = n0 + t / MT * 16 + 4 * lg;
    f32x4 v = sum(t);
    const float inv = NORM ? sinv[min(m, XL * 8 - 1)] : 1.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] *= inv;
    if (EPI == EPI_SWIGLU) {
      const f32x4 u = sum(t + RO * MT);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[e] = v[e] / (1.f + __expf(-v[e])) * (u[e] * inv);
    }
    float sq = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (m >= M || n + e >= N || (!RT && lg > 1)) break;
      if (EPI == EPI_SWIGLU) ep.act[m * ep.as + n + e] = f2bf(v[e]);
      else epilogue<EPI>(outp, m, N, n + e, v[e], ep);
      if (EPI == EPI_RES_BF16) {
        const float y = bf2f(((u16*)outp)[(long)m * N + n + e]);
        sq = fmaf(y, y, sq);
      }
    }
    if (EPI == EPI_RES_BF16 && nm.sums_out) {
      sq += __shfl_xor(sq, 16);
      sq += __shfl_xor(sq, 32);
      const int tile = n0 / (RT ? 16 : 8) + t / MT;
      if (lg == 0 && m < M && tile < nm.tiles)
        nm.sums_out[(long)m * nm.tiles + tile] = sq;
    }
  }
}

template <int EPI, int XL, int RT, int S>
void launch_skinny(void* out, const void* x, const void* w, int M, int N,
                   int K, const Epilogue& ep, const SkinnyNorm& nm,
                   hipStream_t stream) {
  constexpr int MT = (XL + 1) / 2;
  constexpr int WL = RT ? 2 * RT : 1, sums = (RT ? RT : 1) * MT * 4;
  constexpr int stages = 4 * S * (WL + XL);
  constexpr int lds = (stages > sums ? stages : sums) * 1024;
  constexpr int cols = EPI == EPI_SWIGLU ? 8 * RT : 8 * WL;
  auto go = [&](auto kernel, int bytes) {
    allow_lds(kernel, bytes);
    hipLaunchKernelGGL(kernel, dim3((N + cols - 1) / cols), dim3(256),
                       bytes, stream, out, (const u16*)x, (const u16*)w, M, N,
                       K, ep, nm);
  };
  if constexpr ((EPI == EPI_BF16 || EPI == EPI_SWIGLU) && XL <= 4)
    if (nm.gain)
      return go(k_skinny<EPI, XL, RT, S, true>,
                max(lds, stages * 1024 + (K + 511) / 512 * 1024));
  go(k_skinny<EPI, XL, RT, S, false>, lds);
}

// Rows of w for 128 tiles of 16 and fewer: tiles of 8 (RT = 0), half of whose products
// are for nothing, but which twice as many CUs load. 2048 x 8192, 8 rows 11.4 -> 9.0 us,
// 20 14.3 -> 11.6, 64 24.1 -> 21.6; 2048 x 2048, 20 rows 6.1 -> 5.5; 768 x 3072, 24 rows
// 6.8 -> 5.8. What a CU gets through is 60 KB a us of w and x together, whatever the
// stages in flight (2 to 8), waves (4 to 16) and first steps. The sums of squares that
// these leave are of 8 columns, for which the caller has to have room.
// Few rows of w (under 320 tiles, little more than one a CU): small tiles, so
// that all CUs load. 4096 rows, 8 of x: 7.8 us against 9.9; 6144: 12.1, 10.6.
// Many with more than 24 rows of x: wide tiles, so that x is repeated less.
// 28672 x 4096, 32 rows: 46 us against 50; 64: 55, 66.
template <int EPI, int XL>
void by_tiles(void* out, const void* x, const void* w, int M, int N, int K,
              const Epilogue& ep, const SkinnyNorm& nm, hipStream_t stream) {
  const int rows = EPI == EPI_SWIGLU ? 2 * N : N;
  if constexpr (XL >= 4)
    if (rows >= 16384)
      return launch_skinny<EPI, XL, 4, 2>(out, x, w, M, N, K, ep, nm, stream);
  if constexpr (EPI != EPI_SWIGLU) {
    if (rows <= 2048 && (!nm.sums_out || nm.tiles >= (N + 7) / 8))
      return launch_skinny<EPI, XL, 0, (XL < 4 ? 4 : 3)>(out, x, w, M, N, K, ep,
                                                         nm, stream);
    if (rows < 5120)
      return launch_skinny<EPI, XL, 1, (XL < 4 ? 3 : 2)>(out, x, w, M, N, K,
                                                         ep, nm, stream);
  }
  launch_skinny<EPI, XL, 2, 2>(out, x, w, M, N, K, ep, nm, stream);
}

template <int EPI>
void by_rows(void* out, const void* x, const void* w, int M, int N, int K,
             const Epilogue& ep, const SkinnyNorm& nm, hipStream_t stream) {
  if (M <= 8) by_tiles<EPI, 1>(out, x, w, M, N, K, ep, nm, stream);
  else if (M <= 16) by_tiles<EPI, 2>(out, x, w, M, N, K, ep, nm, stream);
  else if (M <= 24) by_tiles<EPI, 3>(out, x, w, M, N, K, ep, nm, stream);
  else if (M <= 32) by_tiles<EPI, 4>(out, x, w, M, N, K, ep, nm, stream);
  else if (M <= 48) by_tiles<EPI, 6>(out, x, w, M, N, K, ep, nm, stream);
  else by_tiles<EPI, 8>(out, x, w, M, N, K, ep, nm, stream);
}

}  // namespace

// 1 to 64 rows, K % 64 == 0, rows of x and w 16-byte aligned. See Epilogue for
// what becomes of the sums and which of the arguments that takes. gain (up to 32
// rows, EPI_BF16 and EPI_SWIGLU; 16-byte aligned): x under an RMS norm with the
// sums [M, tiles]. sums_out (EPI_RES_BF16): [M, tiles], tiles = N / 16 up, or, of N up
// to 2048, N / 8 up.
extern "C" void fei_skinny(void* out, const void* x, const void* w, int M,
                           int N, int K, int epi, const float* bias,
                           float scale, float cap, int n_mix, int n_router,
                           float* router, void* act, long as,
                           const void* bias16, const void* gain,
                           const float* sums, int tiles, float eps,
                           float* sums_out, hipStream_t stream) {
  const Epilogue ep{bias,   scale,     cap, n_mix,              n_router,
                    router, (u16*)act, as,  (const u16*)bias16};
  const SkinnyNorm nm{(const u16*)gain, sums, tiles, eps, sums_out};
  switch (epi) {
#define CASE(E)                                                      \
  case E: return by_rows<E>(out, x, w, M, N, K, ep, nm, stream)
    CASE(EPI_BF16);
    CASE(EPI_F32);
    CASE(EPI_RES);
    CASE(EPI_PARALLEL);
    CASE(EPI_RES_BF16);
    CASE(EPI_SWIGLU);
    CASE(EPI_GELU);
#undef CASE
    default: return;
  }
}
