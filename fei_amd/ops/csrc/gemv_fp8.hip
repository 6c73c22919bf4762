// Quantization of weights to FP8 (OCP e4m3fn, gfx950's) with one float32 scale
// per output row (absmax / 448), once at load time. The products that read them
// are k_gemv's (gemv.hip).
#include "fei_common.h"

namespace {

// quantize bf16 rows -> e4m3fn + per-row scale (absmax/448), RNE on the
// mantissa via float rounding: encode(w / scale).
__device__ __forceinline__ unsigned char e4m3_encode(float f) {
  if (f != f) return 0x7F;                  // NaN
  const unsigned int bits = __float_as_uint(f);
  const unsigned int s = bits >> 31;
  float a = fabsf(f);
  if (a > 448.f) a = 448.f;                 // saturate (no inf in e4m3fn)
  // round to the e4m3 grid: scale into [1,2), round mantissa to 3 bits
  if (a < 0.001953125f * 0.5f) return (unsigned char)(s << 7);  // -> 0
  int e;
  float mant = frexpf(a, &e);               // a = mant * 2^e, mant in [0.5,1)
  mant *= 2.f; e -= 1;                      // mant in [1,2)
  if (e < -6) {                             // subnormal: units of 2^-9
    const int mi = (int)rintf(a * 512.f);   // a / 2^-9, RNE
    if (mi > 7)                             // rounds up to the min normal
      return (unsigned char)((s << 7) | (1 << 3));
    return (unsigned char)((s << 7) | mi);
  }
  int mi = (int)rintf((mant - 1.f) * 8.f);  // 3-bit mantissa, RNE via rintf
  if (mi == 8) { mi = 0; e += 1; }
  if (e > 8) { e = 8; mi = 6; }             // clamp to 448 = 1.75*2^8
  return (unsigned char)((s << 7) | ((e + 7) << 3) | mi);
}

__global__ void __launch_bounds__(256)
k_quant_fp8_rows(unsigned char* __restrict__ w8, float* __restrict__ wscale,
                 const u16* __restrict__ w, int N, int K) {
  __shared__ float red[4];
  for (int n = blockIdx.x; n < N; n += gridDim.x) {
    const u16* row = w + (long)n * K;
    float amax = 0.f;
    for (int i = threadIdx.x; i < K; i += blockDim.x)
      amax = fmaxf(amax, fabsf(bf2f(row[i])));
    amax = block_reduce_max(amax, red);
    const float scale = amax > 0.f ? amax / 448.f : 1.f;
    const float inv = 1.f / scale;
    if (threadIdx.x == 0) wscale[n] = scale;
    for (int i = threadIdx.x; i < K; i += blockDim.x)
      w8[(long)n * K + i] = e4m3_encode(bf2f(row[i]) * inv);
    __syncthreads();
  }
}

}  // namespace

extern "C" {

void fei_quant_fp8_rows(void* w8, float* wscale, const void* w, int N, int K,
                        hipStream_t stream) {
  int grid = N < 2048 ? N : 2048;
  hipLaunchKernelGGL(k_quant_fp8_rows, dim3(grid), dim3(256), 0, stream,
                     (unsigned char*)w8, wscale, (const u16*)w, N, K);
}

}  // extern "C"
