// All layers of an encoder over up to 128 rows, and the texts' means, in one launch (gfx950).
//
// A chain of launches over so few rows is 5 a layer, each of 4 to 8 us for products that
// take 1: a launch, its first loads, its last blocks. Here 256 blocks of one a CU stay, and
// hand results on as fei_chain.h says. A layer has five phases, whose items are of 16 rows:
//   QKV   LayerNorm of what OUT left; 16 T columns of queries, keys and values
//   ATT   a wave has the queries of a head
//   MID   16 columns of the output product, of many rows 32 of them
//   INNER LayerNorm; 16 T columns of the GELU product
//   OUT   16 columns of the outer product, as MID
// Blocks of QKV and INNER make the norms for themselves, and keep the residual in registers.
// Eight waves share K; weights, biases and gains are asked for before the input is there,
// OUT's weights, 96 KB, two phases ahead to LDS. What ATT, MID and OUT read is handed on in
// the order of matrix fragments, 1 KB of 32 columns and 16 rows, so that a wave's loads are
// whole lines. Who reads much asks, past the L2, for one dword of each item first; when they
// are there, it reads through the L2, and what it finds to be NONE all the same again past it.
//
// Bound by the seams, 1.5 to 1.8 us each from one phase's end to what the next has read, and
// by the norms, which take 2.4 us of 16 rows: two rows a wave, whose instructions are 4 cycles
// each. Whole encoders, 12 layers of 768, us, the chain's (native) first: 8 rows 307 -> 224;
// 24 371 -> 236; 40 418 -> 276; 64 485 -> 281, 8 texts of 8 486 -> 297; 80 556 -> 361; 128 567
// -> 440, and each further tile of 16 rows takes 25 more, where the chain takes 3. What goes
// into a norm is handed on in float32: in bfloat16, as the chain's up to 64 rows, 24 took 234,
// and embeddings were over ten seeds 0.391 % from float64, 0.341 now, the chain's 0.378; of
// 100 rows, where the chain keeps float32 too, 0.292, 0.253, 0.260. Loads of what is handed on
// for the lanes that have a row alone took 24 rows 250. Items of all rows, so that
// a block made the norm of 64, took 376 for 24 and 527 for 64 rows; weights of OUT in
// registers, asked for behind INNER, 4 us a layer more where blocks have items of both;
// attention made by each block of MID for itself 440 and 614; biases and gains asked for
// behind the wait 1.5 us a phase. All that reads asking past the L2 at once, without flags
// first (as ATT and MID do): the same; all waves looking at the flags 234 -> 249.
//
// Forward progress: see fei_chain.h. By ticket an item waits only for items of smaller
// tickets, norms and residual come from memory, and any number of blocks comes to the end: of
// 24 rows with 255 blocks 269 us for 236, of 128 467 for 443. Two side by side, of 24 rows,
// take 239 each, as chains 216: every CU is kept to the end.
// Waits end after LIMIT looks all the same; nothing but a fault of this file would make
// them, and the embeddings are NaN then.
#include "fei_attn.h"
#include "fei_chain.h"
#include "fei_epilogue.h"

namespace {

constexpr int NW = 8, THREADS = NW * 64;
constexpr int BLOCKS = 256;
constexpr int MOST = 32;                 // layers
constexpr int ROWS = 128;
constexpr int D = 64;                    // of a head
// a lane's groups of 4 columns of C; a wave's steps of 32 of C and H D, and of 64 of I
constexpr int NC = 3, NEAR = 3, FAR = 6;
constexpr float M_NONE = -3.0e38f;

enum { QKV, ATT, MID, INNER, OUT, LAST, POOL };
constexpr int PHASES = 5;                // of a layer; behind the last one the last norm, and means

struct Layer {                           // as in fei_encoder_layers
  const u16 *wqkv, *bqkv, *wo, *bo, *gain1, *shift1, *wi, *bi, *wo2, *bo2, *gain2, *shift2;
};

struct Encoder {
  Layer layer[MOST];
  const u16* h;                          // [M, C], normed embeddings
  float* out;                            // [B, C]
  const int* lens;
  u32 *buf, *state;
  int layers, B, S, M, tiles, H, C, I;   // tiles of 16 rows
  // dwords of a layer's room, and to what is handed on in it: queries and keys as fragments;
  // values as rows; ATT's results as fragments, MID's as rows of float32, INNER's as fragments,
  // OUT's as rows of float32; by ticket normed rows. Behind the last layer's LAST's rows
  int stride, v, att, mid, inner, o2, keep1, keep2;
  float eps, c;
};

// The arguments, read where they are used: what follows from them would be kept over all
// phases and spilled.
typedef const __attribute__((address_space(4))) Encoder Args;
__device__ __forceinline__ Args& args() {
  Args* p = (Args*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *p;
}
// The same of the thread's place, from which addresses follow.
__device__ __forceinline__ int here() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

struct Lds { u32 dead, ticket; float red[NW]; };

__device__ __forceinline__ bool lost(Lds* s) { return __builtin_amdgcn_readfirstlane(raised(&s->dead)); }

typedef __attribute__((ext_vector_type(2))) u32 u32x2;

__device__ __forceinline__ bool there(u32x2 v) { return v[0] != NONE && v[1] != NONE; }
__device__ __forceinline__ bool there(u32x4 v) {
  return v[0] != NONE && v[1] != NONE && v[2] != NONE && v[3] != NONE;
}
__device__ __forceinline__ u32x2 past2(const u32* p) {
  return __builtin_bit_cast(u32x2, ld_sc((const u64*)p));
}
__device__ __forceinline__ u32x4 past4(const u32* p) {
  const u32x2 a = past2(p), b = past2(p + 2);
  return u32x4{a[0], a[1], b[0], b[1]};
}
__device__ __forceinline__ u32x2 past(const u32* p, u32x2) { return past2(p); }
__device__ __forceinline__ u32x4 past(const u32* p, u32x4) { return past4(p); }

// Two dwords handed on.
__device__ __forceinline__ void give(u32* p, u32 a, u32 b) {
  const u32x2 v = {a == NONE ? NONE - 1 : a, b == NONE ? NONE - 1 : b};
  __hip_atomic_store((u64*)p, __builtin_bit_cast(u64, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// N values, dwords off(i) from base, of which need(i) are handed on: all asked for at once,
// through the L2 (LATER: past it), and until they are there past it. MADE: by another
// launch, so there.
enum { THROUGH, LATER, MADE };
enum { BF16, GELU, F32 };                // what a product's sums become: bfloat16, that of GELU, float32
template <int N, typename V, typename Off, typename Need>
__device__ __forceinline__ void take(V (&v)[N], const u32* base, Off off, Need need, Lds* s, int how = THROUGH) {
  auto at = [&](int i) { return (const u32*)((const char*)base + (u32)(off(i) * 4)); };
#pragma unroll
  for (int i = 0; i < N; ++i) {
    v[i] = V{};
    if (need(i)) v[i] = how == LATER ? past(at(i), V{}) : *(const V*)at(i);
  }
  for (int n = 0; ; ++n) {
    bool ok = true;
#pragma unroll
    for (int i = 0; i < N; ++i) ok &= there(v[i]);
    if (how == MADE || __all(ok)) break;
    if (n > LIMIT || lost(s)) { raise(&s->dead); break; }
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (need(i)) v[i] = past(at(i), V{});
  }
}

// A wave waits for n items, up to 64 K, each told by the dword flag(i) from base.
template <int K, typename Flag>
__device__ __forceinline__ void wait(int n, const u32* base, Flag flag, Lds* s, int lane) {
  for (int k = 0; ; ++k) {
    bool ok = true;
#pragma unroll
    for (int i = 0; i < K; ++i) ok &= ld_sc(base + (u32)flag(min(i * 64 + lane, n - 1))) != NONE;
    if (__all(ok)) break;
    if (k > LIMIT || lost(s)) { raise(&s->dead); break; }
  }
}

// Dwords to a place in a product's input as fragments: columns 4 c on of a row of K. In LDS
// the rows' places are permuted, so that lanes along c spread over the banks.
__device__ __forceinline__ int at_frag(int row, int c, int K) {
  return (row >> 4) * 8 * K + ((c >> 1) * 16 + (row & 15)) * 4 + (c & 1) * 2;
}
__device__ __forceinline__ int at_lds(int row, int c) { return ((c >> 1) * 16 + ((row ^ (c >> 1)) & 15)) * 4 + (c & 1) * 2; }

// A wave's steps of 32 of K, which step i is, and whether it is one: those behind the last
// read it again and count 0, so that there are no branches.
struct Part {
  int lo, n;
  __device__ __forceinline__ int at(int i) const { return lo + min(i, max(n - 1, 0)); }
  __device__ __forceinline__ s16x8 only(int i, s16x8 f) const { return i < n ? f : s16x8{0, 0, 0, 0, 0, 0, 0, 0}; }
};
__device__ __forceinline__ Part part(int K, int w) {
  const int steps = K / 32, per = (steps + NW - 1) / NW, lo = min(w * per, steps);
  return Part{min(lo, steps - 1), min(steps, lo + per) - lo};
}

// A wave's fragments of 16 rows of W.
template <int N>
__device__ __forceinline__ void weights(s16x8 (&f)[N], const u16* W, int tile, int K, Part p, int lane) {
  const u16* at = W + (long)(tile * 16 + (lane & 15)) * K + (lane >> 4) * 8;
#pragma unroll
  for (int i = 0; i < N; ++i) f[i] = ld8(at + p.at(i) * 32);
}

// The bias of a lane's columns.
__device__ __forceinline__ u32x2 bias(const u16* b, int tile, int lane) {
  return *(const u32x2*)(b + tile * 16 + (lane >> 4) * 4);
}

// Sums the waves' shares of tiles j0 .. j1 of columns, of which a wave hands on one: lane's 4
// (lane / 16) on of row lane % 16, to to(j, row, column / 4 of the tile), null if there is none.
template <int T, int AS, typename To>
__device__ __forceinline__ void hand_tiles(int j0, int j1, const u32x2 (&b)[T], const f32x4* red, To to, int lane, int w) {
#pragma unroll
  for (int j = 0; j < T; ++j)
    if (j >= j0 && j <= j1 && w == j - j0) {
      const f32x4* p = red + w * NW * 64 + lane;
      f32x4 v = p[0];
#pragma unroll
      for (int k = 1; k < NW; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += p[k * 64][e];
      const float x[4] = {v[0] + lo(b[j][0]), v[1] + hi(b[j][0]), v[2] + lo(b[j][1]), v[3] + hi(b[j][1])};
      u32* at = to(j, lane & 15, lane >> 4);
      if (!at) return;
      if (AS == F32) {
        give(at, __builtin_bit_cast(u32, x[0]), __builtin_bit_cast(u32, x[1]));
        give(at + 2, __builtin_bit_cast(u32, x[2]), __builtin_bit_cast(u32, x[3]));
      } else if (AS == GELU) {
        give(at, pack(gelu_erf(x[0]), gelu_erf(x[1])), pack(gelu_erf(x[2]), gelu_erf(x[3])));
      } else {
        give(at, pack(x[0], x[1]), pack(x[2], x[3]));
      }
    }
}

// All T of them, in room for PASS at a time.
constexpr int PASS = 3;
template <int T, int AS, typename To>
__device__ __forceinline__ void hand_on(const f32x4 (&acc)[T], const u32x2 (&b)[T], f32x4* red, To to, int tid) {
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
  for (int j = 0; j < T; ++j) {
    if (j && j % PASS == 0) sync_lds();    // it has been read
    red[(j % PASS * NW + w) * 64 + lane] = acc[j];
    if (j % PASS < PASS - 1 && j < T - 1) continue;
    sync_lds();
    hand_tiles<T, AS>(j - j % PASS, j, b, red, to, lane, w);
  }
}

// xs = LayerNorm of 16 rows of x (float32) + res from row0 on, which becomes the new residual. A wave
// has rows w and w + 8, its lanes columns 4 lane on and every 256 further. gv, sv: their
// gains and shifts. Not normed: the first layer's rows, as they are. from: by ticket where
// the residual is; keep: where rows tile and every tiles-th of the new one go to.
__device__ __forceinline__ void norm(Lds* s, const u32* x, bool normed, const u32x2 (&gv)[NC], const u32x2 (&sv)[NC],
                                     u32x2 (&res)[2 * NC], u32* xs, const u32* from, u32* keep, int row0, int tile,
                                     int tiles, int tid) {
  Args& a = args();
  const int M = a.M, C = a.C, n4 = C / 4, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto place = [&](int i) { return (row0 + w + NW * (i / NC)) * (C / 2) + 2 * (lane + 64 * (i % NC)); };
  // the next one that there is: loads of all lanes cost less than to leave some out
  auto near = [&](int i) { return min(row0 + w + NW * (i / NC), M - 1) * (C / 2) + 2 * min(lane + 64 * (i % NC), n4 - 1); };
  auto need = [&](int i) { return row0 + w + NW * (i / NC) < M && lane + 64 * (i % NC) < n4; };
  const u32* h = (const u32*)a.h;
  if (from) take(res, from, place, need, s, from == h ? MADE : THROUGH);
  u32x2 v[2 * NC];
  f32x4 y[2 * NC];
  if (normed) {
    u32x4 z[2 * NC];
    take(z, x, [&](int i) { return 2 * near(i); }, [&](int) { return true; }, s);
#pragma unroll
    for (int i = 0; i < 2 * NC; ++i) y[i] = need(i) ? __builtin_bit_cast(f32x4, z[i]) : f32x4{0.f, 0.f, 0.f, 0.f};
  } else {
    take(v, x, place, need, s, MADE);
#pragma unroll
    for (int i = 0; i < 2 * NC; ++i) y[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  if (normed) {
    float f[2][NC][4], sum[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float t = 0.f;                       // lanes without columns have 0
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        const f32x4 z = y[i * NC + k];
        const u32x2 r = res[i * NC + k];
        f[i][k][0] = z[0] + lo(r[0]);
        f[i][k][1] = z[1] + hi(r[0]);
        f[i][k][2] = z[2] + lo(r[1]);
        f[i][k][3] = z[3] + hi(r[1]);
        t += (f[i][k][0] + f[i][k][1]) + (f[i][k][2] + f[i][k][3]);
      }
      sum[i] = t;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) sum[i] = wave_sum(sum[i]);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float mean = sum[i] / (float)C;
      float t = 0.f;
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        float q = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          f[i][k][e] -= mean;
          q = fmaf(f[i][k][e], f[i][k][e], q);
        }
        t += lane + 64 * k < n4 ? q : 0.f;
      }
      sum[i] = t;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) sum[i] = wave_sum(sum[i]);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float inv = rsqrtf(sum[i] / (float)C + a.eps);
#pragma unroll
      for (int k = 0; k < NC; ++k)
#pragma unroll
        for (int e = 0; e < 2; ++e)
          v[i * NC + k][e] = pack(fmaf(f[i][k][2 * e] * inv, lo(gv[k][e]), lo(sv[k][e])),
                                 fmaf(f[i][k][2 * e + 1] * inv, hi(gv[k][e]), hi(sv[k][e])));
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = w + NW * i;
    const bool kept = keep && (tiles == 1 || r % tiles == tile);
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const bool here = need(i * NC + k);
      const u32x2 y = here ? v[i * NC + k] : u32x2{0, 0};    // of no row, and of no column
      res[i * NC + k] = y;
      if (lane + 64 * k < n4) *(u32x2*)(xs + at_lds(r, lane + 64 * k)) = y;
      if (kept && here) give(keep + place(i * NC + k), y[0], y[1]);
    }
  }
}

// Attention of 16 queries: of tile u % tiles of head u / tiles. All keys of the text at once,
// KT tiles, their scores transposed, so that a lane has four keys a tile of one query, and as
// they lie they are the second operand of V^T times P^T.
template <int KT>
__device__ __forceinline__ void attend(Lds* s, u32* at, int u, int lane) {
  Args& a = args();
  constexpr int KC = (KT + 1) / 2;       // 32 keys at a time
  const int l15 = lane & 15, lg = lane >> 4, S = a.S, H = a.H, HD = H * D;
  const int tiles = (S + 15) / 16, p = u / tiles, t = u - p * tiles;
  const int b = p / H, head = p - b * H, first = b * S;
  const int n = min(max(a.lens[b], 0), S);
  // keys, then queries as fragments, 8 bytes at a time; values: columns 4 l15 on of 8 keys.
  // All at once, but of more keys than there are registers for
  constexpr int NF = 2 * KT + 2, NV = 8 * KC, NOW = 2 * NF + (KT > 4 ? 0 : NV);
  auto off = [&](int i) {
    if (i < 2 * NF) {
      const int j = i / 2, row = first + min(16 * (j < 2 * KT ? j / 2 : t) + l15, S - 1);
      return at_frag(row, (j < 2 * KT ? H * 16 : 0) + head * 16 + (j & 1) * 8 + lg * 2, 2 * HD) + (i & 1) * 2;
    }
    const int j = i - 2 * NF, key = j / 8 * 32 + (j & 4) * 4 + 4 * lg + (j & 3);
    return a.v + (first + min(key, S - 1)) * (HD / 2) + head * (D / 2) + 2 * l15;
  };
  auto need = [&](int i) { return i < 2 * NF ? i / 2 >= 2 * KT || i / 4 < tiles : (i - 2 * NF) / 8 * 32 < S; };
  u32x2 g[NOW];
  // few read it: asked for past the L2 at once, without flags first (24 rows 234.5 -> 232, 64
  // 286 -> 280)
  take(g, at, off, need, s, LATER);
  s16x8 f[NF];
#pragma unroll
  for (int i = 0; i < NF; ++i) f[i] = __builtin_bit_cast(s16x8, u32x4{g[2 * i][0], g[2 * i][1], g[2 * i + 1][0], g[2 * i + 1][1]});
  float sc[2 * KC][4];
  float m = -1.f / 0.f;
#pragma unroll
  for (int j = 0; j < 2 * KC; ++j) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (j < KT)
#pragma unroll
      for (int k = 0; k < 2; ++k) acc = mma(f[2 * min(j, KT - 1) + k], f[2 * KT + k], acc);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      sc[j][r] = 16 * j + 4 * lg + r < n ? acc[r] : -1.f / 0.f;
      m = fmaxf(m, sc[j][r]);
    }
  }
  m = fmaxf(head_max(m) * a.c, M_NONE);
  u32x2 v[NV];
  if constexpr (NOW > 2 * NF) {
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = g[2 * NF + i];
  } else {
    take(v, at, [&](int i) { return off(2 * NF + i); }, [&](int i) { return need(2 * NF + i); }, s, LATER);
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {           // what lies past the keys counts 0
    const int key = i / 8 * 32 + (i & 4) * 4 + 4 * lg + (i & 3);
    if (key >= n) v[i] = u32x2{0, 0};
  }
  float ls = 0.f;
  f32x4 o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < KC; ++q) {
    s16x8 pr;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float x = __builtin_amdgcn_exp2f(fmaf(sc[2 * q + i / 4][i & 3], a.c, -m));
      ls += x;
      pr[i] = (short)El<u16>::st(x);
    }
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        u32x4 va;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          va[i] = __builtin_amdgcn_perm(v[8 * q + 2 * i + 1][d], v[8 * q + 2 * i][d],
                                        hf ? 0x07060302u : 0x05040100u);
        o[2 * d + hf] = mma(__builtin_bit_cast(s16x8, va), pr, o[2 * d + hf]);
      }
  }
  ls = head_sum(ls);
  const float inv = ls > 0.f || ls != ls ? 1.f / ls : 0.f;
  if (16 * t + l15 < S)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      give(at + a.att + at_frag(first + 16 * t + l15, head * 16 + 4 * lg + r, HD),
           pack(o[0][r] * inv, o[1][r] * inv), pack(o[2][r] * inv, o[3][r] * inv));
}

// OUT's weights: 16 rows of W in LDS, a wave's steps of 64 of K, whose 16-byte places are
// permuted by the row, so that the fragment reads spread over the banks.
struct Far { int lo, n; };
__device__ __forceinline__ Far far_part(int K, int w) {
  const int steps = K / 64, per = (steps + NW - 1) / NW, lo = min(w * per, steps);
  return Far{lo, min(steps, lo + per) - lo};
}
__device__ __forceinline__ void fetch_far(const u16* W, int tile, int K, u16* ws, int tid) {
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r8 = lane >> 3;
  const Far p = far_part(K, w);
  const u16* src = W + (long)(tile * 16 + r8) * K + p.lo * 64 + ((lane & 7) ^ r8) * 8;
  const u32 to = (u32)(uintptr_t)(__attribute__((address_space(3))) u16*)ws + w * FAR * 2048;
  for (int i = 0; i < p.n; ++i) {
    load_lds(src + i * 64, to + i * 2048);
    load_lds(src + (long)8 * K + i * 64, to + i * 2048 + 1024);
  }
}

// Mean of a text's normed rows, to length 1.
__device__ __forceinline__ void pool(Lds* s, const u32* rows, int b, int tid) {
  Args& a = args();
  const int n = min(max(a.lens[b], 0), a.S), C = a.C;
  const bool mine = tid < C / 4;
  float v[4] = {0.f, 0.f, 0.f, 0.f}, sq = 0.f;
  for (int i0 = 0; i0 < n; i0 += 8) {
    u32x2 x[8];
    take(x, rows, [&](int i) { return (b * a.S + i0 + i) * (C / 2) + 2 * tid; },
         [&](int i) { return mine && i0 + i < n; }, s, LATER);
#pragma unroll
    for (int i = 0; i < 8; ++i) {          // 0 behind the last
      v[0] += lo(x[i][0]);
      v[1] += hi(x[i][0]);
      v[2] += lo(x[i][1]);
      v[3] += hi(x[i][1]);
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] /= (float)max(n, 1);
    sq = fmaf(v[e], v[e], sq);
  }
  const float len = sqrtf(block_reduce_sum(sq, s->red));
  const float by = len < 1e-12f ? 1e-12f : len;   // NaN stays
  if (mine) *(f32x4*)(a.out + (long)b * C + tid * 4) = f32x4{v[0] / by, v[1] / by, v[2] / by, v[3] / by};
}

template <int T>
__global__ void __launch_bounds__(THREADS, 1) k_encoder_one(const Encoder) {
  // a text's tiles of keys; tiles of rows of MID's and OUT's items, whose weights they share
  constexpr int KT = T < 3 ? T : T < 4 ? 4 : 8, RP = T < 5 ? 1 : 2;
  extern __shared__ __align__(16) char lds[];
  __shared__ Lds s;
  f32x4* red = (f32x4*)lds;
  u16* far = (u16*)(lds + min(T, PASS) * NW * 1024);
  u32* xs = (u32*)(lds + min(T, PASS) * NW * 1024 + NW * FAR * 2048);
  u32* state = args().state;
  if (threadIdx.x == 0) {
    s.dead = 0;
    s.ticket = arrive(state, BLOCKS);
  }
  __syncthreads();
  const u32 rank = __builtin_amdgcn_readfirstlane(s.ticket);
  const bool fixed = rank != NONE;
  u32x2 res[2 * NC];
#pragma unroll
  for (int i = 0; i < 2 * NC; ++i) res[i] = u32x2{0, 0};
  int ly = 0, kind = QKV, item = 0;
  for (;;) {
    Args& a = args();
    const int tid = here(), lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int C = a.C, I = a.I, HD = a.H * D, layers = a.layers, MT = a.tiles;
    // items of the phases: of QKV and INNER of one tile of rows, so that a block's residual
    // is; MID's and OUT's from the last block on
    const int gq = (3 * HD / 16 + T - 1) / T, gi = (I / 16 + T - 1) / T, nm = C / 16;
    const int nq = gq * MT, ni = gi * MT, no = nm * ((MT + RP - 1) / RP);
    const int units = a.B * a.H * ((a.S + 15) / 16), na = min(units, BLOCKS);
    if (!fixed) {
      __syncthreads();
      if (tid == 0) s.ticket = count(a.state + TICKET);
      __syncthreads();
      int t = __builtin_amdgcn_readfirstlane(s.ticket);
      const int all = nq + na + no + ni + no;
      ly = t / all;
      t -= ly * all;
      if (ly >= layers) {
        t += (ly - layers) * all;
        ly = layers;
        kind = LAST;
        if (t >= MT) {
          kind = POOL;
          t -= MT;
          if (t >= a.B) break;
        }
      } else if (t < nq) {
        kind = QKV;
      } else if ((t -= nq) < na) {
        kind = ATT;
      } else if ((t -= na) < no) {
        kind = MID;
      } else if ((t -= no) < ni) {
        kind = INNER;
      } else {
        t -= ni;
        kind = OUT;
      }
      item = t;
    } else {
      item = kind == MID || kind == OUT ? BLOCKS - 1 - rank : rank;
    }
    u32* at = a.buf + (long)ly * a.stride;
    if (kind == QKV || kind == INNER || kind == LAST) {
      if (!fixed || item < (kind == LAST ? MT : max(nq, ni))) {
        const bool second = kind == INNER;
        const int rt = item % MT, group = item / MT, groups = kind == LAST ? 1 : second ? gi : gq;
        const bool mine = kind != LAST && group < groups, normed = second || ly;
        const int last = (second ? I : 3 * HD) / 16 - 1;
        const Part p = part(C, w);
        s16x8 f[T][NEAR];
        u32x2 b[T], gv[NC], sv[NC];
        if (mine) {
#pragma unroll
          for (int j = 0; j < T; ++j) {
            const int tile = min(group * T + j, last);
            weights(f[j], second ? a.layer[ly].wi : a.layer[ly].wqkv, tile, C, p, lane);
            b[j] = bias(second ? a.layer[ly].bi : a.layer[ly].bqkv, tile, lane);
          }
        }
        if (normed) {
          const u16 *gain = second ? a.layer[ly].gain1 : a.layer[ly - 1].gain2,
                    *shift = second ? a.layer[ly].shift1 : a.layer[ly - 1].shift2;
#pragma unroll
          for (int k = 0; k < NC; ++k) {
            gv[k] = ((const u32x2*)gain)[min(lane + 64 * k, C / 4 - 1)];
            sv[k] = ((const u32x2*)shift)[min(lane + 64 * k, C / 4 - 1)];
          }
        }
        const u32 *x = (const u32*)a.h, *from = nullptr;
        u32* keep = kind == LAST ? at : nullptr;
        if (second) {
          x = at + a.mid;
          if (!fixed) {
            from = ly ? at + a.keep2 : (const u32*)a.h;
            keep = at + a.keep1;
          }
        } else if (ly) {
          const u32* before = at - a.stride;           // the layer before
          x = before + a.o2;
          if (!fixed) {
            from = before + a.keep1;
            if (kind != LAST) keep = at + a.keep2;
          }
        }
        if (normed) {
          if (w == 0) wait<1>(nm, x, [&](int i) { return (rt * 16 + 15) * C + i * 16 + 15; }, &s, lane);
          sync_lds();
        }
        norm(&s, x, normed, gv, sv, res, xs, from, keep, rt * 16, group, groups, tid);
        sync_lds();
        if (lost(&s)) break;
        if (mine) {
          f32x4 acc[T];
#pragma unroll
          for (int j = 0; j < T; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int i = 0; i < NEAR; ++i) {
            const int g = p.at(i) * 4 + (lane >> 4);
            const s16x8 y = p.only(i, ld8((const u16*)(xs + (g * 16 + ((lane ^ g) & 15)) * 4)));
#pragma unroll
            for (int j = 0; j < T; ++j) acc[j] = mma(f[j][i], y, acc[j]);
          }
          if (second) {
            hand_on<T, GELU>(acc, b, red, [&](int j, int row, int c4) {
              const int tile = group * T + j;
              return tile > last ? nullptr : at + a.inner + at_frag(rt * 16 + row, tile * 4 + c4, I);
            }, tid);
          } else {
            hand_on<T, BF16>(acc, b, red, [&](int j, int row, int c4) {
              const int tile = group * T + j, c = tile * 16 - 2 * HD, r = rt * 16 + row;
              return tile > last ? nullptr : at + (c < 0 ? at_frag(r, tile * 4 + c4, 2 * HD) : a.v + r * (HD / 2) + c / 2 + 2 * c4);
            }, tid);
          }
        }
      }
    } else if (kind == ATT) {
      const int out = BLOCKS - 1 - (int)rank;
      if (fixed && out < no) fetch_far(a.layer[ly].wo2, out % nm, I, far, tid);
      const int u = item + BLOCKS * w;
      if (item < na && u < units) attend<KT>(&s, at, u, lane);
      sync_lds();
      if (lost(&s)) break;
    } else if (kind == POOL) {
      if (item < a.B) pool(&s, at, item, tid);
      if (lost(&s)) break;
    } else if (item < no) {
      const int rp = item / nm, tile = item - rp * nm;
      const bool mid = kind == MID;
      u32x2 b[RP];
      f32x4 acc[RP];
#pragma unroll
      for (int r = 0; r < RP; ++r) {
        b[r] = bias(mid ? a.layer[ly].bo : a.layer[ly].bo2, tile, lane);
        acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      if (mid) {
        const Part p = part(HD, w);
        s16x8 f[NEAR];
        weights(f, a.layer[ly].wo, tile, HD, p, lane);
        u32x4 x[RP * NEAR];
        // the last row stands in for those behind it, which nobody writes
        take(x, at + a.att, [&](int i) {
          const int rt = min(rp * RP + i / NEAR, MT - 1);
          return rt * 8 * HD + p.at(i % NEAR) * 256 + (lane & 48) * 4 + min(lane & 15, a.M - 1 - rt * 16) * 4;
        }, [&](int) { return true; }, &s, LATER);
#pragma unroll
        for (int i = 0; i < RP * NEAR; ++i)
          acc[i / NEAR] = mma(f[i % NEAR], p.only(i % NEAR, __builtin_bit_cast(s16x8, x[i])), acc[i / NEAR]);
      } else {
        const Far p = far_part(I, w);
        if (!fixed) fetch_far(a.layer[ly].wo2, tile, I, far, tid);
        if (p.n) {
          const u16* ws = far + w * FAR * 1024;
#pragma unroll
          for (int r = 0; r < RP; ++r) {
            const int rt = rp * RP + r;
            if (rt >= MT) break;
            const u32* from = at + a.inner + rt * 8 * I;
            wait<1>(4 * p.n, from, [&](int i) { return at_frag(15, (4 * p.lo + i) * 4 + 3, I) + 1; }, &s, lane);
            u32x4 x[2 * FAR];
            take(x, from, [&](int i) { return (2 * p.lo + min(i, 2 * p.n - 1)) * 256 + lane * 4; }, [&](int) { return true; }, &s);
            // the weights too: they were asked for before what has come
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
            for (int i = 0; i < 2 * FAR; ++i)
              if (i < 2 * p.n)
                acc[r] = mma(ld8(ws + i / 2 * 1024 + (lane & 15) * 64 + (((i & 1) * 4 + (lane >> 4)) ^ (lane & 7)) * 8),
                             __builtin_bit_cast(s16x8, x[i]), acc[r]);
          }
        }
      }
      hand_on<RP, F32>(acc, b, red, [&](int j, int r, int c4) {
        const int rt = rp * RP + j;
        return rt < MT ? at + (mid ? a.mid : a.o2) + (rt * 16 + r) * C + tile * 16 + 4 * c4 : nullptr;
      }, tid);
      if (lost(&s)) break;
    }
    if (fixed) {
      if (kind == POOL) break;
      ++kind;
      if (kind == PHASES) {
        kind = QKV;
        if (++ly == layers) kind = LAST;
      }
      // red and xs have been read
      sync_lds();
    }
  }
  Args& a = args();
  if (lost(&s))
    for (int i = threadIdx.x; i < a.B * a.C; i += THREADS) a.out[i] = __builtin_nanf("");
}

// Empties what blocks hand to each other, and the launch's state.
__global__ void __launch_bounds__(256) k_encoder_one_begin(u32* ws, long dwords) {
  const long i0 = blockIdx.x * 256 + threadIdx.x, n = gridDim.x * 256;
  for (long i = i0 * 4; i < dwords; i += n * 4) *(u32x4*)(ws + i) = u32x4{NONE, NONE, NONE, NONE};
  if (i0 < STATE) ws[dwords + i0] = 0;
}

inline int tiles_of(int M) { return (M + 15) / 16; }

inline long room_of(Encoder& a) {
  const int R = a.tiles * 16, HD = a.H * D;
  int o = 0;
  auto room = [&](int n) { const int at = o; o += n; return at; };
  room(R * HD);
  a.v = room(R * HD / 2);
  a.att = room(R * HD / 2);
  a.mid = room(R * a.C);
  a.inner = room(R * a.I / 2);
  a.o2 = room(R * a.C);
  a.keep1 = room(R * a.C / 2);
  a.keep2 = room(R * a.C / 2);
  a.stride = o;
  return (long)o * a.layers + R * a.C / 2;
}

// T: the fewest tiles of columns an item with which INNER, of up to 192, has no more items
// than blocks
inline int per_item(int tiles) { return tiles < 3 ? tiles : tiles < 5 ? 3 : tiles < 8 ? tiles - 1 : 6; }
// more than half of a CU's: one block each
inline int lds_of(const Encoder& a) {
  const int T = per_item(a.tiles);
  return (T < PASS ? T : PASS) * NW * 1024 + NW * FAR * 2048 + 32 * a.C;
}

}  // namespace

// blocks: of the launch, 256, fewer to have items taken by ticket.
struct EncoderShape { int layers, B, S, H, C, I, blocks; float eps, scale; };

namespace {
inline Encoder encoder_of(const EncoderShape& p) {
  Encoder a{};
  a.layers = p.layers; a.B = p.B; a.S = p.S; a.M = p.B * p.S; a.H = p.H; a.C = p.C; a.I = p.I;
  a.tiles = tiles_of(a.M);
  a.eps = p.eps;
  a.c = p.scale * El<u16>::base;
  return a;
}
}  // namespace

extern "C" {

// Bytes of room that it takes, 0 where it cannot run it. Heads of 64.
long fei_encoder_one_room(const EncoderShape* p) {
  // more blocks than items would write in front of the buffers
  if (p->blocks < 1 || p->blocks > BLOCKS || p->layers <= 0 || p->layers > MOST || p->B <= 0 || p->S <= 0 || p->B > ROWS || p->S > ROWS || p->B * p->S > ROWS ||
      p->H <= 0 || p->H > 12 || p->C <= 0 || p->C > 768 || p->I <= 0 || p->I > 3072 || p->C % 64 || p->I % 64)
    return 0;
  // so that there are no more items of a phase than blocks
  Encoder a = encoder_of(*p);
  return (room_of(a) + STATE) * 4;
}

// ptrs: 12 a layer, as in fei_encoder_layers; h [B * S, C] normed embeddings; out [B, C]
// float32; ws: fei_encoder_one_room bytes. All on 16 bytes.
void fei_encoder_one(const void* const* ptrs, const EncoderShape* p, const void* h, void* out, void* ws,
                     const int* lens, hipStream_t stream) {
  Encoder a = encoder_of(*p);
  const long dwords = room_of(a);
  for (int i = 0; i < p->layers; ++i) a.layer[i] = *(const Layer*)(ptrs + 12 * i);
  a.h = (const u16*)h;
  a.out = (float*)out;
  a.lens = lens;
  a.buf = (u32*)ws;
  a.state = a.buf + dwords;
  hipLaunchKernelGGL(k_encoder_one_begin, dim3(256), dim3(256), 0, stream, a.buf, dwords);
  const int bytes = lds_of(a);
  auto go = [&](auto kernel) {
    allow_lds(kernel, bytes);
    hipLaunchKernelGGL(kernel, dim3(p->blocks), dim3(THREADS), bytes, stream, a);
  };
  switch (per_item(a.tiles)) {
    case 1: return go(k_encoder_one<1>);
    case 2: return go(k_encoder_one<2>);
    case 3: return go(k_encoder_one<3>);
    case 4: return go(k_encoder_one<4>);
    case 5: return go(k_encoder_one<5>);
    default: return go(k_encoder_one<6>);
  }
}

}  // extern "C"
