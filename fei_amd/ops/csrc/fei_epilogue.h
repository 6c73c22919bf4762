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
  // EPI_SWIGLU: rows of act are ``as`` apart. EPI_PARALLEL: n_mix columns go to out, the next n_router to router, of
  // the rest relu(.)^2 to act, whose rows are ``as`` apart
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

// x Phi(x), erf by its rational approximation times exp(-x^2 / 2) (Abramowitz and
// Stegun, Handbook of Mathematical Functions, 7.1.26; 1.5e-7 at most). Taken from
// the side of the tail, so that nothing cancels there.
__device__ __forceinline__ float gelu_erf(float x) {
  const float z = fabsf(x) * 0.70710678118654752f;
  const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, z, 1.f));
  float p = fmaf(t, 1.061405429f, -1.453152027f);
  p = fmaf(t, p, 1.421413741f);
  p = fmaf(t, p, -0.284496736f);
  p = fmaf(t, p, 0.254829592f);
  // half of erfc(z)
  const float q = 0.5f * t * p * __expf(-z * z);
  return x * (x < 0.f ? q : 1.f - q);
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
