// Causal (or bidirectional) GQA attention of prompt rows over contiguous
// caches, gfx950. Semantics: fei_amd/ops/reference.py::attn_prefill - q
// [B,S,Hq,D] (roped), caches [B,Hkv,max_seq,D] already hold the roped K and V
// for positions [0, pos0+S); q token s attends cache [0, pos0+s] (causal) or
// [0, kv_len) (bidirectional, the encoder's).
//
// A row is a (token, query head) pair of one kv head, token-major, so that all
// heads of a group share the tiles of K and V. A block takes 128 rows, a wave
// 32 of them, over tiles of 64 keys that direct loads bring to LDS one tile
// ahead. Scores are computed transposed (K times Q^T, 32x32x16): a lane has 32
// scores of ONE row, so that the softmax needs a single exchange between lanes,
// and its weights are, as they lie, the second operand of V^T times P^T, whose
// sums again belong to the lane's row. K and V lie in LDS as in memory but for
// a permutation of a row's places by the row, which spreads the fragment reads over
// the banks; V is turned by the transposing LDS read. The products with the values
// stand between the exponentials of the next 16 keys, one for two or four.
//
// What bounds it: per 64 keys a wave has 32 matrix instructions (1024 cycles
// at D = 128) and 900 of softmax, and the two waves of a SIMD overlap little of them:
// a tile takes 2400. Counters (2 x 2048 tokens): matrix units 36 % of the time, vector
// units 36, LDS 18 (36 before its reads were free of bank conflicts, which by itself
// gained nothing). Two groups of waves that take turns, in step, at products and
// softmax and share the keys of a block's rows were no faster (2048 tokens 50.5 us,
// heads of 64, 6 x 1001, 58). Against all products behind all exponentials and a
// lane's addresses made anew for each tile: 2048 tokens, 32/8 heads of 128, 55 -> 51
// us, over 2048 more 116 -> 107; 6 x 1001, heads of 64, 43 -> 40; 64 x 256, 12 heads,
// not causal 28 -> 26. Measured in a
// model's layers against a wave of 16 queries of one head with the values turned
// on the way into LDS: 2048 tokens, 32/8 heads of 128: 282 -> 63 us (545 TFLOP/s
// of the causal half); 6 x 1001 tokens, heads of 64: 235 -> 49; 64 x 256, 12 heads
// of 64, not causal: 59 -> 32; 75 tokens over 1875 keys: 139 -> 20 with splits and
// their combine (24 blocks without).
#include "fei_mma.h"

namespace {

typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

constexpr int MAX_SPLITS = 16;
constexpr int ROWS = 128;              // rows per block
constexpr int KEYS = 64;               // keys per tile
constexpr float M_NONE = -3.0e38f;     // maximum of a row without keys
constexpr float DONE = -1.f;           // sum of a row that one split finished

struct Prefill {
  const u16 *q, *kc, *vc;
  u16* out;
  float *po, *pml;                     // partial results of splits
  const int *pos0, *kv_len, *starts;   // starts: the first row of each text, PACKED
  int B, S, G, Hkv, heads, tiles, max_seq, causal, splits;
  int share;                           // keys for the rows of a batch row: cut_keys
  float scale;
  long q_ts;
  long kv_b, kv_h, kv_t;               // strides of the caches
};

// Keys that the rows up to r_hi of batch row b see.
__device__ __forceinline__ int keys_of(const Prefill& a, int b, int r_hi) {
  const int n = a.causal ? a.pos0[b] + r_hi / a.G + 1 : a.kv_len[b];
  return min(n, a.max_seq);
}

// Whether the keys of a batch row are cut into splits: where its last row sees more than
// few (asked of one block of rows by itself, those of few keys would have them all and be
// the last: 500 tokens over 1800 keys 58 us for 39). How many are few is what the results
// of splits and the combine cost, which grow with the rows that are cut: 3 tiles, and a
// key for 14 rows of the batch rows that are cut. In one and cut, us, over room for 8192
// keys, 32 heads of 128, 8 of keys: 150 tokens over 300 keys 19.0, 19.3, over 600 23.9,
// 21.1; 300 over 600 27.1, 31.1; 500 over 600 31.0, 33.8, over 1000 38.0, 36.1; 4 x 75
// over 600 24.0, 28.8, over 1800 44.5, 41.7, where three of the four begin 42.5, 33.0.
constexpr int FEW = 3 * KEYS;
__device__ __forceinline__ bool cut_keys(const Prefill& a, int b) {
  const int last = a.S * a.G - 1, n = keys_of(a, b, last);
  if (n <= FEW + a.share || a.B == 1) return n > FEW + a.share;
  int cut = 0;                           // batch rows that would be, by themselves
  for (int i = 0; i < a.B; i += 64) {
    const int at = i + (threadIdx.x & 63);
    cut += __popcll(__ballot(at < a.B && keys_of(a, min(at, a.B - 1), last) >
                                             FEW + a.share));
  }
  return n > FEW + cut * a.share;
}
// Tiles of a split of n keys.
__device__ __forceinline__ int split_tiles(const Prefill& a, int n) {
  return max(((n + KEYS - 1) / KEYS + a.splits - 1) / a.splits, 3);
}

// By what the 16-byte places of a row of K or V in LDS are turned round, so that the
// fragment reads take all 64 banks: 16 lanes read a place of 16 rows of K, 32 lanes
// two of 32 bytes of 4 rows of V; a row fills the banks (D = 128) or half of them.
template <int D>
__device__ __forceinline__ int key_turn(int row) {
  return D == 128 ? row & 15 : row >> 1 & 7;
}
template <int D>
__device__ __forceinline__ int value_turn(int row) {
  return D == 128 ? (row & 3) * 4 : (row & 2) * 2;
}

// Tile of the j-th block of a kv head. Causal tiles cost as much as they have
// keys before them. Where all blocks fit on the chip at once (two per CU), the
// second half takes the light ones upwards, so that a CU's pair costs the same
// everywhere; otherwise the heavy ones go first.
__device__ __forceinline__ int tile_of(const Prefill& a, int j) {
  const int half = (a.tiles + 1) / 2;
  if (a.causal && a.heads * a.tiles <= 512 && j >= half) return j - half;
  return a.tiles - 1 - j;
}

// PACKED: a row of the batch has kv_len[b] <= S tokens, whose queries, keys, values and
// results are rows starts[b] and on; of those that it has not nothing is touched.
template <int D, bool SPLIT, bool PACKED = false>
__global__ void __launch_bounds__(256, 2) k_attn_prefill(const Prefill a) {
  constexpr int KS = D / 16;           // steps of a score product
  constexpr int DT = D / 32;           // tiles of 32 value columns
  constexpr int LPR = D / 8;           // 16-byte places of a cache row
  constexpr int RPI = 64 / LPR;        // rows of a load of 64 lanes
  constexpr int LOADS = KEYS / RPI / 4;    // a wave's, of K and of V each
  __shared__ __align__(16) u16 buf[2][2][KEYS * D];
  const int head = blockIdx.x % a.heads, j = blockIdx.x / a.heads;
  const int b = head / a.Hkv, hkv = head - b * a.Hkv;
  // where nothing is cut the first splits come first, so that each has a CU by itself,
  // and the others leave at once (4 x 150 rows over 1950 keys 56 us -> 38); else those of
  // a tile, so that two on a CU are of unlike tiles (75 over 4000 31.8 -> 30.1)
  const bool cut = SPLIT && cut_keys(a, b);
  const int split = !SPLIT ? 0 : cut ? j % a.splits : j / a.tiles;
  if (SPLIT && !cut && split) return;
  const int tile = tile_of(a, cut ? j / a.splits : j);
  const int R = (PACKED ? keys_of(a, b, 0) : a.S) * a.G, row0 = tile * ROWS;
  if (PACKED && row0 >= R) return;
  const long tok0 = PACKED ? a.starts[b] : (long)b * a.S;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l31 = lane & 31, h = lane >> 5;
  const int n = keys_of(a, b, min(row0 + ROWS, R) - 1);
  const int r = row0 + wid * 32 + l31;
  const int s = min(r, R - 1) / a.G, g = min(r, R - 1) - s * a.G;
  const long prow = ((long)head * R + r) * a.splits + split;
  int t0 = 0, t1 = (n + KEYS - 1) / KEYS;
  if (cut) {
    const int per = split_tiles(a, n);
    t0 = split * per;
    t1 = min(t1, t0 + per);
    if (t0 >= t1 && split) {           // no keys: the sums are never read
      if (h == 0 && r < R) *(f32x2*)(a.pml + prow * 2) = f32x2{M_NONE, 0.f};
      return;
    }
  }

  // last key that the lane's row sees; first tile that needs a mask; keys past
  // the wave's last row are skipped
  const int lim = a.causal ? min(a.pos0[b] + s, n - 1) : n - 1;
  const int r_first = min(row0 + wid * 32, R - 1);
  const int r_last = min(row0 + wid * 32 + 31, R - 1);
  const int lim_lo = a.causal ? min(a.pos0[b] + r_first / a.G, n - 1) : n - 1;
  const int lim_hi = a.causal ? min(a.pos0[b] + r_last / a.G, n - 1) : n - 1;

  // a negative scale turns the queries round, a zero one clears them, so that
  // the largest score stays the largest after scaling
  const float c = a.scale == 0.f ? 1.f : fabsf(a.scale) * El<u16>::base;
  const u32 flip = a.scale < 0.f ? 0x80008000u : 0u;
  const u32 keep = a.scale == 0.f ? 0u : 0xffffffffu;
  s16x8 fq[KS];
  {
    const u16* qp = a.q + (tok0 + s) * a.q_ts +
                    (long)(hkv * a.G + g) * D + 8 * h;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      u32x4 v = *(const u32x4*)(qp + k * 16);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (v[e] ^ flip) & keep;
      fq[k] = __builtin_bit_cast(s16x8, v);
    }
  }

  const long kv0 = (PACKED ? tok0 * a.kv_t : b * a.kv_b) + hkv * a.kv_h;
  const u16 *kb = a.kc + kv0, *vb = a.vc + kv0;
  const u32 lds =
      (u32)(uintptr_t)(__attribute__((address_space(3))) u16*)&buf[0][0][0];
  // what a lane loads of a tile, in bytes from its first row: the wave's LOADS times
  // RPI rows, of V behind that of K. A tile that ends past the keys reads its last
  // one again.
  u32 at[2][LOADS];
  const int lrow = wid * LOADS * RPI + lane / LPR, place = lane % LPR;
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = lrow + i * RPI;
    at[0][i] = row * (u32)a.kv_t * 2 + (place ^ key_turn<D>(row)) * 16;
    at[1][i] = row * (u32)a.kv_t * 2 + (place ^ value_turn<D>(row)) * 16;
  }
  const bool near = a.kv_t < 1 << 24;      // such offsets have 32 bits
  auto load = [&](int t, auto which) __attribute__((always_inline)) {
    constexpr int V = decltype(which)::value;
    const u16* base = V ? vb : kb;
    const u32 to = lds + (((t - t0) & 1) * 2 + V) * KEYS * D * 2 +
                   wid * LOADS * 1024;
    if (near && t * KEYS + KEYS <= n) {
      base += (long)t * KEYS * a.kv_t;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) load_lds_from(base, at[V][i], to + i * 1024);
    } else {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        const int row = lrow + i * RPI;
        const int c = place ^ (V ? value_turn<D>(row) : key_turn<D>(row));
        load_lds(base + (long)min(t * KEYS + row, n - 1) * a.kv_t + c * 8,
                 to + i * 1024);
      }
    }
  };

  float m = M_NONE, l = 0.f;
  f32x16 o[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[i][e] = 0.f;

  // Step k of a score product of tile t, 32 keys of it.
  auto key = [&](int t, int k, int i) __attribute__((always_inline)) {
    return ld8(buf[(t - t0) & 1][0] + (i * 32 + l31) * D +
               (((k * 2 + h) ^ key_turn<D>(l31)) << 3));
  };
  // 32 columns of 16 keys, 4 values of a column at a time in the order of the keys
  // that the lane's weights have: 16 i + 4 h + 0..3, then + 8
  const int vr = 4 * h + ((lane & 15) >> 2), vc0 = (lane >> 4) & 1;
  auto value = [&](int t, int i, int dt) __attribute__((always_inline)) {
    const u16* vp = buf[(t - t0) & 1][1] + (i * 16 + vr) * D +
                    (((dt * 4 + vc0 * 2) ^ value_turn<D>(vr)) << 3) +
                    (lane & 3) * 4;
    return turn8(vp, vp + 8 * D);
  };
  if (t0 < t1) {
    load(t0, First{});
    load(t0, Second{});
  }
  for (int t = t0; t < t1; ++t) {
    // the tile is there, and all waves are done with the other buffer
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (t + 1 < t1) {
      load(t + 1, First{});
      load(t + 1, Second{});
    }
    if (t * KEYS > lim_hi) continue;
    f32x16 sc[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) sc[i][e] = 0.f;
    s16x8 vf[DT];
    if constexpr (D == 128) {
      // fragments 8 products ahead; heads of 64 would lose the fourth wave of a SIMD
      // by the registers (6 x 1001 tokens 40.4 -> 41.8 us; of 128 73.3 -> 70.2)
      constexpr int AHEAD = 8;
      s16x8 kf[AHEAD];
#pragma unroll
      for (int x = 0; x < AHEAD; ++x) kf[x] = key(t, x / 2, x % 2);
#pragma unroll
      for (int x = 0; x < 2 * KS; ++x) {
        sc[x % 2] = mma32(kf[x % AHEAD], fq[x / 2], sc[x % 2]);
        if (x + AHEAD < 2 * KS)
          kf[x % AHEAD] = key(t, (x + AHEAD) / 2, (x + AHEAD) % 2);
        else if (x + DT >= 2 * KS)
          vf[x + DT - 2 * KS] = value(t, 0, x + DT - 2 * KS);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int i = 0; i < 2; ++i) sc[i] = mma32(key(t, k, i), fq[k], sc[i]);
#pragma unroll
      for (int j = 0; j < DT; ++j) vf[j] = value(t, 0, j);
    }
    // register e of sc[i] is key t * 64 + i * 32 + 8 (e / 4) + 4 h + e % 4
    if (t * KEYS + KEYS - 1 > lim_lo) {
      const int d = lim - t * KEYS - 4 * h;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (i * 32 + 8 * (e / 4) + e % 4 > d) sc[i][e] = -1.f / 0.f;
    }
    float mx = fmaxf(sc[0][0], sc[1][0]);
#pragma unroll
    for (int e = 1; e < 16; ++e) mx = fmaxf(fmaxf(mx, sc[0][e]), sc[1][e]);
    const f32x2 two = both_halves(mx);
    mx = fmaxf(two[0], two[1]) * c;
    // the maximum may lag behind by 2^8: weights and sums are float32 with
    // room for that, and most tiles leave the sums as they are
    if (__any(mx > m + 8.f)) {
      const float mn = fmaxf(m, mx);
      const float al = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      l *= al;
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[i][e] *= al;
    }
    // weights of 16 keys at a time; between them, the products with the 16 before
    s16x8 fp;
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float x[8];
      u32x4 w;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        if (i && u % (8 / DT) == 0) {
          const int j = u / (8 / DT);
          o[j] = mma32(vf[j], fp, o[j]);
          vf[j] = value(t, i, j);
        }
        x[u] = __builtin_amdgcn_exp2f(fmaf(sc[i >> 1][(i & 1) * 8 + u], c, -m));
        if (u & 1) {
          ps += x[u - 1] + x[u];
          w[u >> 1] = __builtin_bit_cast(
              u32, __builtin_convertvector(f32x2{x[u - 1], x[u]}, bf16x2));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      fp = __builtin_bit_cast(s16x8, w);
      if (i & 1) {
        l += ps;
        ps = 0.f;
      }
    }
#pragma unroll
    for (int j = 0; j < DT; ++j) o[j] = mma32(vf[j], fp, o[j]);
  }

  const f32x2 lt = both_halves(l);
  l = lt[0] + lt[1];
  if (r >= R) return;
  // column dt * 32 + 8 i + 4 h + 0..3 in registers 4 i .. of o[dt]
  if (SPLIT) {
    if (cut && split_tiles(a, n) * KEYS < n) {   // there are other splits
      float* po = a.po + prow * D + 4 * h;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          *(f32x4*)(po + dt * 32 + 8 * i) =
              f32x4{o[dt][4 * i], o[dt][4 * i + 1], o[dt][4 * i + 2],
                    o[dt][4 * i + 3]};
      if (h == 0) *(f32x2*)(a.pml + prow * 2) = f32x2{m, l};
      return;
    }
    if (h == 0) *(f32x2*)(a.pml + prow * 2) = f32x2{M_NONE, DONE};
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  u16* op = a.out + ((tok0 + s) * a.Hkv * a.G + hkv * a.G + g) * D + 4 * h;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u16 v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = El<u16>::st(o[dt][4 * i + e] * inv);
      __builtin_memcpy(op + dt * 32 + 8 * i, v, sizeof(v));
    }
}

// Sums of the splits of a row; one wave per row, rows that one split finished
// are left alone. All splits are asked for at once: 75 rows of 32 heads of 128, 16
// splits: 9.3 -> 6.2 us.
template <int D>
__global__ void __launch_bounds__(256)
k_attn_prefill_combine(const Prefill a) {
  const int R = a.S * a.G, lane = threadIdx.x & 63;
  const long id = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (id >= (long)a.heads * R) return;
  const int head = id / R, r = id - (long)head * R;
  const int b = head / a.Hkv, hkv = head - b * a.Hkv;
  // a lane has the maximum and the sum of a split
  const float* ml = a.pml + id * a.splits * 2;
  float m = M_NONE, l = 0.f;
  if (lane < a.splits) {
    m = ml[2 * lane];
    l = ml[2 * lane + 1];
  }
  // known sooner than the sums are here
  if (keys_of(a, b, R - 1) <= FEW + a.share) return;
  if (__builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(
          __builtin_bit_cast(int, l))) == DONE)
    return;
  const u64 used = __ballot(lane == 0 || l != 0.f || m != M_NONE);
  float top = m;
#pragma unroll
  for (int i = 1; i < MAX_SPLITS; i *= 2) top = fmaxf(top, __shfl_xor(top, i));
  const float w = __builtin_amdgcn_exp2f(m - top);
  l *= w;
#pragma unroll
  for (int i = 1; i < MAX_SPLITS; i *= 2) l += __shfl_xor(l, i);
  l = __shfl(l, 0);
  const int n = 64 - __builtin_clzll(used);
  float o[D / 64];
#pragma unroll
  for (int e = 0; e < D / 64; ++e) o[e] = 0.f;
  const float* po = a.po + id * a.splits * D + lane * (D / 64);
#pragma unroll 4
  for (int i = 0; i < n; ++i) {
    const float wi = __shfl(w, i);
    const bool has = used >> i & 1;        // others left nothing behind
#pragma unroll
    for (int e = 0; e < D / 64; ++e) {
      const float v = po[i * D + e];
      o[e] = fmaf(wi, has ? v : 0.f, o[e]);
    }
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  const int s = r / a.G, g = r - s * a.G;
  u16* op = a.out + (((long)b * a.S + s) * a.Hkv * a.G + hkv * a.G + g) * D +
            lane * (D / 64);
#pragma unroll
  for (int e = 0; e < D / 64; ++e) op[e] = El<u16>::st(o[e] * inv);
}

template <int D>
void launch_prefill(const Prefill& a, hipStream_t stream) {
  const dim3 grid((unsigned)a.heads * a.tiles * a.splits);
  if (a.splits > 1) {
    hipLaunchKernelGGL((k_attn_prefill<D, true>), grid, dim3(256), 0, stream,
                       a);
    const long rows = (long)a.heads * a.S * a.G;
    hipLaunchKernelGGL(k_attn_prefill_combine<D>, dim3((rows + 3) / 4),
                       dim3(256), 0, stream, a);
  } else {
    hipLaunchKernelGGL((k_attn_prefill<D, false>), grid, dim3(256), 0, stream,
                       a);
  }
}

}  // namespace

extern "C" {

// Strides of both caches by batch row, head and position; rows of D values,
// 16-byte aligned. po [B * Hkv, S * G, splits, D] and pml [.., splits, 2] float32,
// where splits > 1; at most 16.
void fei_attn_prefill(const void* q, const void* k_cache, const void* v_cache,
                      void* out, const int* pos0, const int* kv_len, int B,
                      int S, int Hq, int Hkv, int D, int max_seq, float scale,
                      int causal, long q_ts, int splits, float* po, float* pml,
                      long kv_b, long kv_h, long kv_t, hipStream_t stream) {
  const int G = Hq / Hkv, tiles = (S * G + ROWS - 1) / ROWS;
  const Prefill a{(const u16*)q, (const u16*)k_cache, (const u16*)v_cache,
                  (u16*)out,     po,     pml,  pos0,  kv_len, nullptr,
                  B,             S,      G,    Hkv,
                  B * Hkv,       tiles,  max_seq, causal, splits,
                  Hkv * S * G / 14,
                  scale,         q_ts,   kv_b, kv_h,  kv_t};
  if (D == 128) launch_prefill<128>(a, stream);
  else if (D == 64) launch_prefill<64>(a, stream);
}

// Attention of B texts of kv_len[b] of at most S tokens among themselves, whose rows lie
// one behind another from row starts[b] on: q, k and v a row of 3 H D values, out of H D.
// D is 64 or 128; all on 16 bytes. kv_len is taken at S where it is more.
void fei_attn_packed(const void* qkv, void* out, const int* kv_len,
                     const int* starts, int B, int S, int H, int D, float scale,
                     hipStream_t stream) {
  const int HD = H * D, tiles = (S + ROWS - 1) / ROWS;
  const u16* p = (const u16*)qkv;
  const Prefill a{p, p + HD, p + 2 * HD, (u16*)out, nullptr, nullptr, kv_len,
                  kv_len, starts, B, S, 1, H, B * H, tiles, S, 0, 1, 0, scale,
                  3L * HD, 0, D, 3L * HD};
  const dim3 grid((unsigned)a.heads * tiles);
  if (D == 128)
    hipLaunchKernelGGL((k_attn_prefill<128, false, true>), grid, dim3(256), 0,
                       stream, a);
  else
    hipLaunchKernelGGL((k_attn_prefill<64, false, true>), grid, dim3(256), 0,
                       stream, a);
}

// ---------------------------------------------------------------------------
// MFMA layout probe: C[16x16] = A[16x32] @ B[32x16] with the fragment maps
// above, all matrices row-major bf16 in global memory. Lets the GPU test
// falsify the assumed lane mappings with asymmetric inputs (guide §3).
// ---------------------------------------------------------------------------
__global__ void k_mfma_probe(const u16* __restrict__ A,
                             const u16* __restrict__ Bm,
                             float* __restrict__ C) {
  const int lane = threadIdx.x & 63;
  const int l15 = lane & 15;
  const int lg = lane >> 4;
  s16x8 a, b;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    a[j] = (short)A[l15 * 32 + 8 * lg + j];
    b[j] = (short)Bm[(8 * lg + j) * 16 + l15];
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
#pragma unroll
  for (int r = 0; r < 4; ++r) C[(4 * lg + r) * 16 + l15] = acc[r];
}

void fei_mfma_probe(const void* A, const void* B, float* C,
                    hipStream_t stream) {
  hipLaunchKernelGGL(k_mfma_probe, dim3(1), dim3(64), 0, stream,
                     (const u16*)A, (const u16*)B, C);
}

}  // extern "C"
