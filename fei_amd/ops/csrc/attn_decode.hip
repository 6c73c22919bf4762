// Decode attention: one new token per sequence over its cached keys, split over
// the keys, all heads of a group together; caches [B,Hkv,max_seq,D] or paged
// pools [blocks,Hkv,BS,D] behind a block table. n = pos[b] + 1 keys, read on
// the device, so that a captured launch serves every length. With cos_sin the
// step's RoPE and the cache row of the new token are made here too.
//
// A wave takes chunks of 32 keys by itself. Scores are computed transposed (K
// times Q^T, 16x16x32: a lane has 8 scores of ONE head), so that the weights
// lie in the registers as the second operand of V^T times P^T; a lane loads 8
// keys x D/16 columns of V and turns them in registers. Keys and values never
// pass LDS, and nothing but the end of a block has a barrier. Roped queries and
// weights enter the bfloat16 products as three parts, whose sum is the float32
// value: 3e-7 of a row's float32 result is what the whole is off by, as much as
// products on the vector units (4e-7); with two parts it was 3e-6, 6 % faster. An
// infinite key or value gives NaN (0 times it, in a part).
// The chunks go to the blocks' waves in order, so that short contexts end in
// few blocks (one: it writes the result), and the rest leave at once.
//
// Bound by latency (position, table, rows, combine) up to some MB of keys, by
// HBM beyond. Per layer with the combine in a graph of 16, against a thread per
// key with the products on the vector units and the scores exchanged through LDS:
// 300 keys, 32/8 heads of 64: 13.5 -> 6.1 us; 512, 3400 and 8000 keys, 32/8 of
// 128: 15.7 -> 8.2, 21.4 -> 9.7 and 25.3 -> 13.7; 8 sequences of 2047: 32.5 ->
// 20.4; 32 of 500: 72 -> 21.2; 20 of 600, heads of 64: 49 -> 12.4. The combine is
// 3.3 (heads of 64) to 5 of it, a launch's least.
#include "fei_attn.h"

namespace {

typedef __attribute__((ext_vector_type(2))) u32 u32x2;

constexpr float M_NONE = -3.0e38f;       // maximum of no keys
constexpr int CHUNK = 32;                // keys of a wave at a time
constexpr int SHARE = 4;                 // waves of a block where keys are split
// of one that has all keys of a head: as many as the registers allow
constexpr int whole_waves(int D) { return D == 64 ? 16 : 8; }

struct DecodeAttn {
  const u16* q;
  u16 *kc, *vc;
  const int* table;                      // paged: [B, W]
  float *po, *pml;                       // [B,Hq,splits,D], [B,Hq,splits,2]
  u16* out;
  const int* pos;
  const u16 *kin, *vin;
  const float* cs;
  int G, Hkv, max_seq, bs_log, W, splits;
  float scale;
  long q_bs, kv_bs;
};

__device__ __forceinline__ int keys_at(const DecodeAttn& a, int b) {
  return min(a.pos[b] + 1, a.max_seq);
}
// Splits that have keys.
template <int WAVES>
__device__ __forceinline__ int used_splits(const DecodeAttn& a, int n) {
  return min(a.splits, (n + CHUNK * WAVES - 1) / (CHUNK * WAVES));
}

// x1 and x2: dimensions d .. d + 7 and d + D/2 .. of a head; cs: their pairs.
__device__ __forceinline__ void rope8(float (&x1)[8], float (&x2)[8],
                                      const float* cs) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x4 t = *(const f32x4*)(cs + 4 * i);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float u = x1[2 * i + j], w = x2[2 * i + j];
      x1[2 * i + j] = u * t[2 * j] - w * t[2 * j + 1];
      x2[2 * i + j] = w * t[2 * j] + u * t[2 * j + 1];
    }
  }
}

template <int N>
__device__ __forceinline__ void rope_row(float (&x)[N][8], const float* cs,
                                         int lg) {
#pragma unroll
  for (int k = 0; k < N / 2; ++k)
    rope8(x[k], x[k + N / 2], cs + (k * 32 + 8 * lg) * 2);
}

// Of roped queries of 128 dimensions two parts wait in LDS: in registers, of which
// three blocks a CU leave 168, 8 spilled (8 x 2047 keys 23.8 us for 20.4).
constexpr bool parts_in_lds(int D, bool rope) { return rope && D > 64; }
// A wave's floats in LDS: its sums at the end, those parts before.
template <int D, bool ROPE>
__host__ __device__ constexpr int wave_floats(int G) {
  return parts_in_lds(D, ROPE) && G * D < D / 32 * 2 * 256 ? D / 32 * 2 * 256
                                                           : G * D;
}

template <int D, bool PAGED, bool ROPE, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, D == 64 ? 4 : WAVES > 4 ? 2 : 3)
k_attn_decode(const DecodeAttn a) {
  constexpr int KS = D / 32;             // steps of a score product
  constexpr int VC = D / 16;             // columns of V a lane loads
  typedef __attribute__((ext_vector_type(VC / 2))) u32 vrow;
  extern __shared__ __align__(16) float so[];      // [WAVES][G][D], m and l
  const int side = gridDim.x / a.Hkv, hkv = blockIdx.x / side;
  const int split = blockIdx.z * side + blockIdx.x - hkv * side;
  const int b = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, lg = lane >> 4;
  const int n = keys_at(a, b), last = n - 1;
  const int chunks = (n + CHUNK - 1) / CHUNK, used = used_splits<WAVES>(a, n);
  const int G = a.G, Hq = a.Hkv * G;
  if (split >= used) {
    if (used <= 0 && split == 0)         // no key: zeros
      for (int i = tid; i < G * D; i += 64 * WAVES)
        a.out[((long)b * Hq + hkv * G) * D + i] = 0;
    return;
  }

  auto row = [&](int key) {
    if (PAGED) {
      const int blk = a.table[(long)b * a.W + (key >> a.bs_log)];
      return ((((long)blk * a.Hkv + hkv) << a.bs_log) +
              (key & ((1 << a.bs_log) - 1))) * D;
    }
    return (((long)b * a.Hkv + hkv) * a.max_seq + key) * D;
  };
  const float* cs = ROPE ? a.cs + (long)last * D : nullptr;

  // queries, head lane % 16 (what the lanes past the last head compute is not
  // used)
  constexpr int NQ = ROPE ? 3 : 1;       // parts; an unroped query is one
  constexpr int NR = parts_in_lds(D, ROPE) ? 1 : NQ;   // of them in registers
  int mine = wid * (wave_floats<D, ROPE>(G) / 4) + lane;
  s16x8 qf[KS][NR];
  {
    const u16* qp = a.q + (long)b * a.q_bs +
                    (long)(hkv * G + min(l15, G - 1)) * D + 8 * lg;
#pragma unroll
    for (int k = 0; k < KS; ++k) qf[k][0] = ld8(qp + k * 32);
    if constexpr (ROPE) {
      float x[KS][8];
#pragma unroll
      for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int j = 0; j < 8; ++j) x[k][j] = bf2f((u16)qf[k][0][j]);
      rope_row(x, cs, lg);
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        s16x8 p[3];
        parts3(x[k], p);
#pragma unroll
        for (int i = 0; i < NR; ++i) qf[k][i] = p[i];
#pragma unroll
        for (int i = NR; i < NQ; ++i) ((s16x8*)so)[mine + (k * 2 + i - 1) * 64] = p[i];
      }
    }
  }
  const float c = a.scale * El<u16>::base;
  // The wave with the last chunk makes the new token's row, for the cache and
  // for itself; no other wave reads it.
  __shared__ __align__(16) u16 fresh[2][D];
  if (ROPE && (chunks - 1) % (a.splits * WAVES) == split * WAVES + wid &&
      lane < D / 2) {
    const u16* kp = a.kin + (long)b * a.kv_bs + (long)hkv * D + lane;
    const u16* vp = a.vin + (long)b * a.kv_bs + (long)hkv * D + lane;
    const f32x2 t = *(const f32x2*)(cs + 2 * lane);
    const float u = bf2f(kp[0]), w = bf2f(kp[D / 2]);
    const u16 row0[2] = {El<u16>::st(u * t[0] - w * t[1]), vp[0]};
    const u16 row1[2] = {El<u16>::st(w * t[0] + u * t[1]), vp[D / 2]};
    const long at = row(last) + lane;
    a.kc[at] = fresh[0][lane] = row0[0];
    a.kc[at + D / 2] = fresh[0][lane + D / 2] = row1[0];
    a.vc[at] = fresh[1][lane] = row0[1];
    a.vc[at + D / 2] = fresh[1][lane + D / 2] = row1[1];
  }

  float m = M_NONE, l = 0.f;
  f32x4 o[VC];
#pragma unroll
  for (int e = 0; e < VC; ++e) o[e] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int ch = split * WAVES + wid; ch < chunks; ch += a.splits * WAVES) {
    const int k0 = ch * CHUNK;
    s16x8 kf[2][KS];
    vrow vf[8];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const u16* kp = a.kc + row(min(k0 + 16 * t + l15, last)) + 8 * lg;
#pragma unroll
      for (int k = 0; k < KS; ++k) kf[t][k] = ld8(kp + k * 32);
    }
#pragma unroll
    for (int r = 0; r < 8; ++r)
      vf[r] = *(const vrow*)(
          a.vc + row(min(k0 + (r & 4) * 4 + 4 * lg + (r & 3), last)) +
          VC * l15);
    if (ROPE && ch == chunks - 1) {      // the new token's row is in LDS
#pragma unroll
      for (int t = 0; t < 2; ++t)
        if (k0 + 16 * t + l15 == last)
#pragma unroll
          for (int k = 0; k < KS; ++k) kf[t][k] = ld8(fresh[0] + 8 * lg + k * 32);
#pragma unroll
      for (int r = 0; r < 8; ++r)
        if (k0 + (r & 4) * 4 + 4 * lg + (r & 3) == last)
          vf[r] = *(const vrow*)(fresh[1] + VC * l15);
    }
    if (k0 + CHUNK > n) {                // what lies past the keys counts 0
#pragma unroll
      for (int r = 0; r < 8; ++r)
        if (k0 + (r & 4) * 4 + 4 * lg + (r & 3) > last)
#pragma unroll
          for (int e = 0; e < VC / 2; ++e) vf[r][e] = 0;
    }
    if (NR < NQ) asm volatile("" : "+v"(mine));      // read each time
    const s16x8* rest = (const s16x8*)so + mine;
    float s[8];                          // keys 4 lg + 0..3, then 16 on
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < KS; ++k) {
#pragma unroll
        for (int i = NQ - 1; i >= 0; --i)
          acc = mma(kf[t][k], i < NR ? qf[k][i % NR] : rest[(k * 2 + i - 1) * 64],
                    acc);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        s[4 * t + r] = k0 + 16 * t + 4 * lg + r > last ? -1.f / 0.f
                                                       : acc[r] * c;
    }
    float mx = fmaxf(s[0], s[1]);
#pragma unroll
    for (int i = 2; i < 8; ++i) mx = fmaxf(mx, s[i]);
    const float mn = fmaxf(m, head_max(mx));
    const float al = __builtin_amdgcn_exp2f(m - mn);
    m = mn;
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      s[i] = __builtin_amdgcn_exp2f(s[i] - mn);
      ps += s[i];
    }
    l = fmaf(l, al, ps);
    s16x8 p[3];
    parts3(s, p);
#pragma unroll
    for (int w = 0; w < VC / 2; ++w)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        u32x4 t;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          t[i] = __builtin_amdgcn_perm(vf[2 * i + 1][w], vf[2 * i][w],
                                       hf ? 0x07060302u : 0x05040100u);
        const s16x8 va = __builtin_bit_cast(s16x8, t);
        f32x4& oe = o[2 * w + hf];
#pragma unroll
        for (int r = 0; r < 4; ++r) oe[r] *= al;
#pragma unroll
        for (int i = 2; i >= 0; --i) oe = mma(va, p[i], oe);
      }
  }
  l = head_sum(l);
  // column VC * (4 lg + r) + e of head l15 is o[e][r]
  constexpr auto stride = wave_floats<D, ROPE>;
  float* sml = so + WAVES * stride(G);
  if (l15 < G) {
    float* dst = so + wid * stride(G) + l15 * D;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int e = 0; e < VC; e += 4)
        *(f32x4*)(dst + VC * (4 * lg + r) + e) =
            f32x4{o[e][r], o[e + 1][r], o[e + 2][r], o[e + 3][r]};
    if (lg == 0) {
      sml[(wid * G + l15) * 2] = m;
      sml[(wid * G + l15) * 2 + 1] = l;
    }
  }
  __syncthreads();
  const bool whole = used == 1;
  for (int i = tid * 4; i < G * D; i += 64 * WAVES * 4) {
    const int g = i / D, d = i - g * D;
    float mm = M_NONE, ll = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) mm = fmaxf(mm, sml[(w * G + g) * 2]);
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float f = __builtin_amdgcn_exp2f(sml[(w * G + g) * 2] - mm);
      const f32x4 t = *(const f32x4*)(so + w * stride(G) + g * D + d);
      ll = fmaf(f, sml[(w * G + g) * 2 + 1], ll);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = fmaf(f, t[e], v[e]);
    }
    const long hq = (long)b * Hq + hkv * G + g;
    if (whole) {
      const float inv = ll > 0.f ? 1.f / ll : 0.f;
      u16 y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = El<u16>::st(v[e] * inv);
      __builtin_memcpy(a.out + hq * D + d, y, sizeof(y));
    } else {
      *(f32x4*)(a.po + (hq * a.splits + split) * D + d) = v;
      if (d == 0)
        *(f32x2*)(a.pml + (hq * a.splits + split) * 2) = f32x2{mm, ll};
    }
  }
}

// out[b,hq] from the splits that have keys; nothing to do where one had all.
// One block per head, 8 (D = 128) or 16 splits side by side. Bound by the latency
// of a launch and its loads: those of the first 16 splits go out with that of the
// position, before it is known how many there are (what lies there otherwise is
// not used).
template <int D>
__global__ void __launch_bounds__(256) k_attn_decode_combine(const DecodeAttn a) {
  constexpr int SIDE = 256 / (D / 4);
  __shared__ f32x4 part[SIDE][D / 4];
  const long hq = blockIdx.x;
  const int b = hq / (a.Hkv * a.G);
  const int tid = threadIdx.x, lane = tid & 63;
  const int side = tid / (D / 4), d = tid % (D / 4);
  const f32x2* ml = (const f32x2*)(a.pml + hq * a.splits * 2);
  const f32x4* po = (const f32x4*)(a.po + hq * a.splits * D) + d;
  constexpr int PRE = 16 / SIDE;
  f32x4 x[PRE];
#pragma unroll
  for (int i = 0; i < PRE; ++i)
    x[i] = po[(long)min(side + i * SIDE, a.splits - 1) * (D / 4)];
  f32x2 t = ml[min(lane, a.splits - 1)];
  const int used = used_splits<SHARE>(a, keys_at(a, b));
  if (used == 1) return;
  if (lane >= used) t = f32x2{M_NONE, 0.f};
  float m = row16_max(t[0]);
  f32x2 sw = swap16(m);
  sw = both_halves(fmaxf(sw[0], sw[1]));
  m = fmaxf(sw[0], sw[1]);
  const float w = __builtin_amdgcn_exp2f(t[0] - m);    // of split ``lane``
  float l = row16_sum(t[1] * w);
  sw = swap16(l);
  sw = both_halves(sw[0] + sw[1]);
  l = sw[0] + sw[1];
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < PRE; ++i) {
    const float f = __shfl(w, side + i * SIDE);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = side + i * SIDE < used ? fmaf(f, x[i][e], v[e]) : v[e];
  }
#pragma unroll 4
  for (int s = side + 16; s < used; s += SIDE) {
    const float f = __builtin_amdgcn_exp2f(ml[s][0] - m);
    const f32x4 y = po[(long)s * (D / 4)];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = fmaf(f, y[e], v[e]);
  }
  part[side][d] = v;
  __syncthreads();
  if (side) return;
#pragma unroll
  for (int i = 1; i < SIDE; ++i)
    if (i < used)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += part[i][d][e];
  const float inv = l > 0.f ? 1.f / l : 0.f;
  u16 y[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = El<u16>::st(v[e] * inv);
  __builtin_memcpy(a.out + hq * D + d * 4, y, sizeof(y));
}

template <int D, int WAVES>
void launch_waves(const DecodeAttn& a, dim3 grid, hipStream_t stream) {
  const int lds = WAVES * (wave_floats<D, false>(a.G) + 2 * a.G) * 4;
  const int roped = WAVES * (wave_floats<D, true>(a.G) + 2 * a.G) * 4;
#define GO(PAGED, ROPE)                                                     \
  allow_lds(k_attn_decode<D, PAGED, ROPE, WAVES>, ROPE ? roped : lds);      \
  hipLaunchKernelGGL((k_attn_decode<D, PAGED, ROPE, WAVES>), grid,          \
                     dim3(64 * WAVES), ROPE ? roped : lds, stream, a)
  if (a.table) {
    if (a.cs) { GO(true, true); } else { GO(true, false); }
  } else {
    if (a.cs) { GO(false, true); } else { GO(false, false); }
  }
#undef GO
}

// Keys up to which a block takes all of a head's, given how many heads of keys there
// are: then nothing is left to combine. Split and combined, or whole, us in a graph:
// 1 sequence of 256 keys and 8 heads of 64 6.7, 6.2; of 320 6.6, 6.8; 8 of 576 9.0,
// 8.0, of 1024 9.7, 11.0; 20 of 600 in pages 12.7, 9.5; 32 of 2048 34.0, 29.3. Heads
// of 128, 8 sequences of 320 9.2, 8.8, of 448 9.5, 10.1; 12 of 512 12.4, 12.5; 20 of
// 1024 21.8, 19.7, of half that 17.0, 11.8. One long sequence among short ones is alone
// on its CUs: 20 of 60 keys, but one of 512 9.5, 9.5, of 640 9.3, 10.6, of 1024 13.3,
// 14.3, of 2048 17.4, 23.6, so that beyond 1024 keys are split. For the same reason
// there are as many splits as were asked for, however many sequences: with no more
// blocks than places, 64 of which one had 8192 keys took 80 us for 41.
inline int whole_keys(int heads, int D) {
  if (heads >= 160) return 1024;
  if (heads < 64) return 256;
  return D == 64 ? 768 : heads < 96 ? 320 : 512;
}

// Returns how many splits there are to sum, if that was left to the caller (``open``).
template <int D>
int launch_decode(DecodeAttn a, int B, bool open, hipStream_t stream) {
  if (a.max_seq > CHUNK * SHARE && a.max_seq <= whole_keys(a.Hkv * B, D)) {
    a.splits = 1;
    launch_waves<D, whole_waves(D)>(a, dim3(a.Hkv, B), stream);
    return 1;
  }
  // Splits that no sequence can have are not launched, and those beyond 16 come
  // last: a block waits for the position to know that it has no keys, and keeps
  // its place meanwhile. 20 sequences of up to 600 keys in pages, 16 splits
  // asked for: 15.9 -> 7.8 us.
  const int all = max(1, min(a.splits, (a.max_seq + CHUNK * SHARE - 1) /
                                           (CHUNK * SHARE)));
  const int side = min(all, 16);
  launch_waves<D, SHARE>(a, dim3(a.Hkv * side, B, (all + side - 1) / side),
                         stream);
  if (all > 1 && !open)
    hipLaunchKernelGGL(k_attn_decode_combine<D>, dim3(B * a.Hkv * a.G),
                       dim3(256), 0, stream, a);
  return all;
}

}  // namespace

// max_seq: rows of a head in a contiguous cache; of a paged one (table not
// null) the positions that a row of the table can name. cs null: q is roped and
// the new token's row is in the cache. Up to 16 query heads a kv head, up to 64
// splits; D is 64 or 128. Nothing is launched for an empty batch.
static int decode(const void* q, void* kc, void* vc, const int* table, float* po,
                  float* pml, void* out, const int* pos, int B, int Hq, int Hkv,
                  int D, int max_seq, int bs_log, int W, int splits, float scale,
                  long q_bs, const void* kin, const void* vin, const float* cs,
                  long kv_bs, bool open, hipStream_t stream) {
  if (B <= 0 || Hkv <= 0) return 1;
  const DecodeAttn a{(const u16*)q, (u16*)kc,         (u16*)vc,
                     table,         po,               pml,
                     (u16*)out,     pos,              (const u16*)kin,
                     (const u16*)vin, cs,             Hq / Hkv,
                     Hkv,           max_seq,          bs_log,
                     W,             splits,           scale,
                     q_bs,          kv_bs};
  if (D == 128) return launch_decode<128>(a, B, open, stream);
  if (D == 64) return launch_decode<64>(a, B, open, stream);
  return 1;
}

extern "C" {

void fei_attn_decode(const void* q, void* kc, void* vc, const int* table, float* po,
                     float* pml, void* out, const int* pos, int B, int Hq, int Hkv,
                     int D, int max_seq, int bs_log, int W, int splits, float scale,
                     long q_bs, const void* kin, const void* vin, const float* cs,
                     long kv_bs, hipStream_t stream) {
  decode(q, kc, vc, table, po, pml, out, pos, B, Hq, Hkv, D, max_seq, bs_log, W,
         splits, scale, q_bs, kin, vin, cs, kv_bs, false, stream);
}

void fei_gemv_splits(void* out, const void* x, const void* w, const float* wscale,
                     int N, int K, const float* po, const float* pml,
                     const int* pos, int splits, int left, int room, int keys,
                     int D, hipStream_t stream);
void fei_gemv(void* out, const void* x, const void* gain, const void* w,
              const float* wscale, int M, int N, int K, float eps, int epi,
              float* ssq, hipStream_t stream);

// Decode attention of one sequence and its output product, added to res [1, N]: w [N, Hq
// D], wscale null or the scales of fp8 rows. Where the splits are few the product sums
// them (gemv.hip), and out is not written. The rest as above.
void fei_attn_decode_product(const void* q, void* kc, void* vc, const int* table,
                             float* po, float* pml, void* out, const int* pos,
                             int Hq, int Hkv, int D, int max_seq, int bs_log, int W,
                             int splits, float scale, long q_bs, const void* kin,
                             const void* vin, const float* cs, long kv_bs,
                             void* res, const void* w, const float* wscale, int N,
                             hipStream_t stream) {
  // of few long rows k_gemv has its waves share them
  const int K = Hq * D, most = K <= 2048 ? 16 : K <= 4096 && N > 2048 ? 5 : 0;
  const bool open = min(splits, (max_seq + CHUNK * SHARE - 1) / (CHUNK * SHARE)) <=
                    most;
  const int left = decode(q, kc, vc, table, po, pml, out, pos, 1, Hq, Hkv, D,
                          max_seq, bs_log, W, splits, scale, q_bs, kin, vin, cs,
                          kv_bs, open, stream);
  if (open && left > 1)
    return fei_gemv_splits(res, out, w, wscale, N, K, po, pml, pos, splits, left,
                           max_seq, CHUNK * SHARE, D, stream);
  constexpr int GEMV_RES = 1;
  fei_gemv(res, out, nullptr, w, wscale, 1, N, K, 0.f, GEMV_RES, nullptr, stream);
}

}  // extern "C"
