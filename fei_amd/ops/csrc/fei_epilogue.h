// What a skinny matrix product does with its float32 sums.
#pragma once
#include "fei_common.h"

enum {
  EPI_BF16 = 0,
  EPI_F32 = 1,
  EPI_RES = 2,        // added to float32
  EPI_PARALLEL = 3,
  EPI_RES_BF16 = 4,   // added to bfloat16
  EPI_SWIGLU = 5,     // of a gate and an up product, to act
  EPI_GELU = 6,       // bfloat16
};

struct Epilogue {
  const float* bias;   // per column, may be null
  float scale;
  float cap;           // 0: no softcap
  // EPI_SWIGLU: rows of act are ``as`` apart. EPI_PARALLEL: n_mix columns go to
  // out, the next n_router to router, of the rest relu(.)^2 to act, whose rows
  // are ``as`` apart
  int n_mix, n_router;
  float* router;
  u16* act;
  long as;
  const u16* bias16;   // EPI_BF16, EPI_GELU: per column, may be null
};

__device__ __forceinline__ float softcap(float v, float scale, float cap) {
  v *= scale;
  return cap > 0.f ? cap * tanhf(v / cap) : v;
}

// x Phi(x). Half of erfc(z), z = |x| / sqrt 2, is exp(-z^2) times a polynomial in t =
// 1 / (1 + 0.38 z) (the form of Abramowitz and Stegun, Handbook of Mathematical
// Functions, 7.1.26, with nine terms for five, fitted to the smallest relative
// error, 2.2e-8). Taken from the side of the tail, so that nothing cancels there.
// Off by 3e-8 of normal inputs' results and 2e-6 of any one down to x = -6; with
// 1 + erff(z) it was 4e-8, 5e-2 at -5. The square under the exponential is of x
// itself; t gets a Newton step, since rcp's last bit would show.
__device__ __forceinline__ float gelu_erf(float x) {
  const float z = fminf(fabsf(x), 20.f);           // 0 beyond, and no inf
  const float d = fmaf(z, 0.38f * 0.70710678118654752f, 1.f);
  float t = __builtin_amdgcn_rcpf(d);
  t = fmaf(fmaf(-d, t, 1.f), t, t);
  float p = fmaf(t, 0.029382409527897835f, -0.13070568442344666f);
  p = fmaf(t, p, 0.1811504364013672f);
  p = fmaf(t, p, -0.07997459173202515f);
  p = fmaf(t, p, 0.11458776146173477f);
  p = fmaf(t, p, 0.06946393847465515f);
  p = fmaf(t, p, 0.1019287258386612f);
  p = fmaf(t, p, 0.10696154087781906f);
  p = fmaf(t, p, 0.10720546543598175f);
  // half of erfc(z)
  const float q =
      t * p * __builtin_amdgcn_exp2f(x * -0.72134752044448170f * x);
  return x < 0.f ? x * q : fmaf(-z, q, x);
}

// silu(g) * u. The quotient is one of a reciprocal, corrected by what it leaves: as
// good as a division's, and the same of infinities, NaN and all normal numbers.
// Both sides are taken at an eighth, so that denominators up to 2^128 (g to -88.7) have
// a reciprocal that is not flushed. Of a division's 11 instructions, most of which scale
// such operands, 6 are left.
__device__ __forceinline__ float swiglu(float g, float u) {
  const float d = fmaf(__expf(-g), 0.125f, 0.125f), h = g * 0.125f;
  const float t = __builtin_amdgcn_rcpf(d), q = h * t;
  return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, h), t, q), d, h) * u;
}

__device__ __forceinline__ float relu2(float v) {
  v = fmaxf(v, 0.f);
  return v * v;
}

// N: columns of out
template <int EPI>
__device__ __forceinline__ void epilogue(void* out, int row, int N, int col,
                                         float v, const Epilogue& ep) {
  const long at = (long)row * N + col;
  if (EPI == EPI_BF16 || EPI == EPI_GELU) {
    if (ep.bias16) v += bf2f(ep.bias16[col]);
    ((u16*)out)[at] = f2bf(EPI == EPI_GELU ? gelu_erf(v) : v);
  } else if (EPI == EPI_RES_BF16) {
    ((u16*)out)[at] = f2bf(bf2f(((u16*)out)[at]) + v);
  } else if (EPI == EPI_RES) {
    ((float*)out)[at] += v * ep.scale;
  } else if (EPI == EPI_F32) {
    v = softcap(v, ep.scale, ep.cap);
    ((float*)out)[at] = ep.bias ? v + ep.bias[col] : v;
  } else if (col < ep.n_mix) {
    ((u16*)out)[(long)row * ep.n_mix + col] = f2bf(v);
  } else if (col < ep.n_mix + ep.n_router) {
    ep.router[(long)row * ep.n_router + col - ep.n_mix] = v;
  } else {
    ep.act[row * ep.as + col - ep.n_mix - ep.n_router] = f2bf(relu2(v));
  }
}
