// Products of few rows with a weight matrix, the decode step's (gfx950):
// out[M, N] = x[M, K] @ W[N, K]^T, F.linear's layout.
//
// k_gemv streams the weights, bfloat16 or fp8 (e4m3fn, a scale per row), through
// the vector units; from M = 4 on k_gemm_m8 (below) uses the matrix units.
#include <type_traits>

#include "fei_epilogue.h"
#include "fei_mma.h"

namespace {

typedef __attribute__((ext_vector_type(4))) u32 u32x4;

enum { GEMV_BF16 = 0, GEMV_RES = 1, GEMV_SWIGLU = 2 };

// Sum over a wave, added in the order of a butterfly from lane ^ 32 down to
// lane ^ 1, without LDS.
__device__ __forceinline__ float wave_sum(float v) {
  const u32 a = __builtin_bit_cast(u32, v);
  const auto p = __builtin_amdgcn_permlane32_swap(a, a, false, false);
  const u32 p0 = p[0], p1 = p[1];
  v = __builtin_bit_cast(float, p0) + __builtin_bit_cast(float, p1);
  const u32 b = __builtin_bit_cast(u32, v);
  const auto q = __builtin_amdgcn_permlane16_swap(b, b, false, false);
  const u32 q0 = q[0], q1 = q[1];
  return row16_sum(__builtin_bit_cast(float, q0) +
                   __builtin_bit_cast(float, q1));
}

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
template <int M, int KS, bool NORM, int EPI, bool FP8, bool LDS>
__global__ void __launch_bounds__(256)
k_gemv(u16* __restrict__ out, const u16* __restrict__ x,
       const u16* __restrict__ gain, const void* __restrict__ wp,
       const float* __restrict__ wscale, int N, int K, float eps,
       float* __restrict__ ssq) {
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
  constexpr int XV = NORM && M == 1 ? 4 : 8;
  const int nx = M * (K / 8);
  s16x8 x0[XV], g0[NORM ? XV : 1];
  auto gain_at = [&](int c) {
    return ((const s16x8*)gain)[M == 1 ? c : c % (K / 8)];
  };
#pragma unroll
  for (int i = 0; LDS && i < XV; ++i) {
    const int c = min(tid + i * 256, nx - 1);
    x0[i] = ((const s16x8*)x)[c];
    if (NORM) g0[i] = gain_at(c);
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

template <int M, bool NORM, int EPI, bool FP8>
void launch_gemv(void* out, const void* x, const void* gain, const void* w,
                 const float* wscale, int N, int K, float eps, float* ssq,
                 hipStream_t stream) {
  const size_t lds = (size_t)M * K * 2;
  auto go = [&](auto kernel, int blocks, size_t bytes) {
    // beyond 64 KB a kernel has to ask
    if (bytes > 65536)
      (void)hipFuncSetAttribute((const void*)kernel,
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)bytes);
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

void fei_prefetch(const void* w, long bytes, void* sink, int n_blocks,
                  hipStream_t stream) {
  const long n_vec8 = bytes / 16;
  if (n_vec8 <= 0) return;
  hipLaunchKernelGGL(k_prefetch, dim3(n_blocks), dim3(256), 0, stream,
                     (const u16*)w, n_vec8, (float*)sink);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// MFMA M<=8 GEMM: out[M, N] = x[M, K] @ W[N, K]^T for the decode batch
// path. Four VALU-kernel variants measured slower than the pipelined
// k_gemv<8> (profiles/r02_batch_attention.md); this MFMA tile beats it
// on every llama shape (qkv 1.45x, o 1.43x, down 1.27x, stacked gate/up
// 1.65x — experimental/gemv_mfma.hip, numerics exact vs the VALU form).
// Structure: 16 n-rows per workgroup, each of NW waves owns K/NW with
// wave-private double-buffered LDS staging (register prefetch overlaps
// the next tile's loads with the current tile's MFMAs; same-wave ds
// ordering needs no barriers), one end-of-kernel cross-wave C reduce.
// A-fragment rows clamp to M-1: the duplicate rows only produce C rows
// >= M, which are never written. Requires K % 1024 == 0, N % 16 == 0
// (the wrapper routes other shapes to k_gemv).
#define GEMM_NT 16
#define GEMM_KC 128
#define GSWZ(row, col8) ((col8) ^ ((row) & 7))

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4_g;

template <bool NTW, int EPI, int NW = 4>
__global__ void __launch_bounds__(NW * 64)
k_gemm_m8(void* __restrict__ outp, const u16* __restrict__ x,
          const u16* __restrict__ w, int M, int N, int K, Epilogue ep) {
  const int n0 = blockIdx.x * GEMM_NT;
  const int tid = threadIdx.x;
  const int wv = tid >> 6;
  const int lane = tid & 63;
  const int l15 = lane & 15, lg = lane >> 4;
  __shared__ u16 wt[NW][2][GEMM_NT * GEMM_KC];
  __shared__ float cred[NW][16][16];

  f32x4_g acc = {0.f, 0.f, 0.f, 0.f};
  const int kq = K / NW;
  const int nv8 = GEMM_KC / 8;
  const int k_lo = wv * kq, k_hi = (wv + 1) * kq;
  const int arow = l15 < M ? l15 : M - 1;
  const int srow = lane / 4, scol8 = (lane % 4) * 4;
  auto fetch = [&](int k0, s16x8 r[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const s16x8* p = (const s16x8*)(w + (long)(n0 + srow) * K + k0 +
                                      (scol8 + j) * 8);
      r[j] = NTW ? __builtin_nontemporal_load(p) : *p;
    }
  };
  auto put = [&](int buf, s16x8 r[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      ((s16x8*)wt[wv][buf])[srow * nv8 + GSWZ(srow, scol8 + j)] = r[j];
  };
  s16x8 pre[4];
  fetch(k_lo, pre);
  put(0, pre);
  int buf = 0;
  for (int k0 = k_lo; k0 < k_hi; k0 += GEMM_KC) {
    if (k0 + GEMM_KC < k_hi) fetch(k0 + GEMM_KC, pre);
#pragma unroll
    for (int kb = 0; kb < GEMM_KC / 32; ++kb) {
      const s16x8 a_frag =
          *(const s16x8*)(x + (long)arow * K + k0 + kb * 32 + lg * 8);
      const int col8 = kb * 4 + lg;
      const s16x8 b_frag =
          ((s16x8*)wt[wv][buf])[l15 * nv8 + GSWZ(l15, col8)];
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_frag, b_frag, acc,
                                                    0, 0, 0);
    }
    if (k0 + GEMM_KC < k_hi) put(buf ^ 1, pre);
    buf ^= 1;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) cred[wv][lg * 4 + r][l15] = acc[r];
  __syncthreads();
  if (wv == 0) {
    for (int i = lane; i < M * 16; i += 64) {
      const int m = i / 16, n = i % 16;
      float v = cred[0][m][n] + cred[1][m][n] + cred[2][m][n] + cred[3][m][n];
#pragma unroll
      for (int c = 4; c < NW; ++c) v += cred[c][m][n];
      epilogue<EPI>(outp, m, N, n0 + n, v, ep);
    }
  }
}

}  // namespace

// float32 results: residual != 0 adds to out, otherwise out is
// softcap(acc * scale, cap) + bias (cap 0: none; bias may be null). With few
// columns more waves share out K, so that the weight stream fills the chip.
extern "C" void fei_gemm_m8_f32(void* out, const void* x, const void* w,
                                const float* bias, int M, int N, int K,
                                int residual, float scale, float cap,
                                hipStream_t stream) {
  dim3 grid(N / GEMM_NT);
  const Epilogue ep{bias, scale, cap};
#define M8(EPI, NW)                                                         \
  hipLaunchKernelGGL((k_gemm_m8<false, EPI, NW>), grid, dim3(NW * 64), 0,   \
                     stream, out, (const u16*)x, (const u16*)w, M, N, K, ep)
#define BY_NW(EPI)                                                          \
  do {                                                                      \
    if (N <= 4096 && K % 2048 == 0) M8(EPI, 16);                            \
    else if (N <= 8192) M8(EPI, 8);                                         \
    else M8(EPI, 4);                                                        \
  } while (0)
  if (residual) BY_NW(EPI_RES); else BY_NW(EPI_F32);
#undef BY_NW
#undef M8
}

// All products of a parallel layer's input (see EPI_PARALLEL).
extern "C" void fei_gemm_m8_parallel_in(void* out, float* router,
                                        const void* x, const void* w,
                                        void* act, long as, int M, int n_mix,
                                        int n_router, int N, int K,
                                        hipStream_t stream) {
  const Epilogue ep{nullptr, 1.f,    0.f,       n_mix,
                    n_router, router, (u16*)act, as};
  if (N <= 8192)
    hipLaunchKernelGGL((k_gemm_m8<false, EPI_PARALLEL, 8>),
                       dim3(N / GEMM_NT), dim3(512), 0, stream, out,
                       (const u16*)x, (const u16*)w, M, N, K, ep);
  else
    hipLaunchKernelGGL((k_gemm_m8<false, EPI_PARALLEL, 4>),
                       dim3(N / GEMM_NT), dim3(256), 0, stream, out,
                       (const u16*)x, (const u16*)w, M, N, K, ep);
}

extern "C" void fei_gemm_m8(void* out, const void* x, const void* w, int M,
                            int N, int K, int nontemporal,
                            hipStream_t stream) {
  dim3 grid(N / GEMM_NT);
  if (nontemporal)
    hipLaunchKernelGGL((k_gemm_m8<true, EPI_BF16>), grid, dim3(256), 0,
                       stream, out, (const u16*)x, (const u16*)w, M, N, K,
                       Epilogue{});
  else
    hipLaunchKernelGGL((k_gemm_m8<false, EPI_BF16>), grid, dim3(256), 0,
                       stream, out, (const u16*)x, (const u16*)w, M, N, K,
                       Epilogue{});
}
