// A decoding step of one sequence on a Llama-style decoder, all layers and the vocabulary's
// product in one launch (gfx950).
//
// A chain of launches loses 3 us and more at each of its 5 seams a layer: the last blocks
// run out, a launch, its first loads. Here 256 blocks of one a CU stay, and hand their
// results on in memory: a block has a fixed 256th of each product's rows (QKV, WO, GU,
// DOWN, HEAD), of the attention's keys (ATT) and of the sums of their splits (SUM).
//
// Handing on. All room is filled with NONE first; a result is one dword of two bfloat16 or
// a float32, written once past the L2 (agent scope), and never NONE (a NaN of that pattern
// becomes another). Who needs it reads until it is no longer NONE: no counters, no fences,
// and nothing is in flight that an order would matter for. One wave of a block asks, past
// the L2, for one dword of each of the 256 items; when they are there, the block's other
// waves read the input through the L2, which 32 CUs share, and what they find to be NONE
// all the same again past it. 256 blocks handing 8 dwords each to all, and nothing else,
// us a phase: so 1.5, all asking for all past the L2 1.9 to 2.1, flags behind a wait for
// the stores 4.0, counters 4.9.
//
// The other 8 waves multiply: a step is 2 rows of w times 2 loads of 16 bytes a lane, two
// steps are in flight a wave and are asked for before the input is there. A CU's loads come
// back in order, whoever asked, so the serving wave has none of its own, asks only when the
// weights should have come (1.35 us), and goes before the others, whose next loads its
// results would wait behind. Of the three steps below, us, all as it is 604, 2664, 1706; three
// steps in flight 600, 2588, 1715, half of two 633, 2772, 1763; asking at once 624, 2712, 1733,
// after 0.8 us 612, 2664, 1722, after 1.9 619, 2642, 1710; nobody before others 617, 2655, 1793.
//
// Forward progress. Blocks count themselves at the start. If all 256 are there within 100
// looks, all of them are on the chip, and each keeps its item of every phase. If not,
// whatever holds the other CUs, items are taken by ticket, in the order of the phases: an
// item waits only for items of smaller tickets, which blocks that run have taken, so that
// any number of blocks, one too, comes to the end. Nothing is asked for ahead then: with 255
// blocks the three take 858, 3785 and 2447. Waits end after LIMIT looks all the same; nothing
// but a fault of this file would make them, and the logits are NaN then. The launch keeps
// every CU to its end, so that two steps side by side are slower than as chains, whose
// launches run in between one another's: two of the first case 598 each and 468, of the
// second 2626 and 2322.
//
// Bound by HBM while products run (27 to 30 KB a us and CU, 7 TB/s) and by the seams, 2 to
// 3 us each; the eight XCDs get 5 % more or less of it, and all wait for the last. Whole
// steps by a graph, which is played again, with the embedding, us, the chain's first: 16
// layers of 2048, 300 keys 646 -> 604; 32 of 4096, 512 keys 2883 -> 2664; fp8 weights, 3400
// keys 1996 -> 1706 (each time other keys, from HBM: 2034 -> 1762). Four layers of 2048 and
// 3400 keys 172 -> 156, 32000 205 -> 186, 131000 349 -> 330, of 4096 365 -> 341, 445 -> 419,
// 723 -> 710: of so many keys a wave has no loads ahead of the 32 it works on. Which
// steps are taken: ops.llama_one_pays.
#include "fei_attn.h"
#include "fei_chain.h"

namespace {

constexpr int NW = 8;                    // waves of a block that multiply
constexpr int THREADS = (NW + 1) * 64;   // and one that serves them
constexpr int U = 2, DEPTH = 2;          // loads of a row a step; steps in flight a wave
constexpr int BLOCKS = 256;              // items of a phase
constexpr int MOST = 32;                 // layers of a launch
constexpr int CHUNK = 32;                // keys of a wave at a time
constexpr float M_NONE = -3.0e38f;       // maximum of no keys

enum { QKV, WO, GU, DOWN, HEAD, ATT, SUM };
constexpr int PHASES = 6;                // of a layer

struct Layer {
  const void* w[4];
  const float* s[4];                     // scales of fp8 rows
  const u16* gain[2];                    // of QKV's and GU's norm
  u16 *kc, *vc;
};

// A product: P pairs of rows of w (of SwiGLU a gate's and an up's), K columns in steps
// of which parts have ``per``, 1 << kp parts. Dwords from a layer's room to its input,
// to what tells that it is there, to what is added, to the results and to the sums of
// their squares.
struct Shape { int P, N, K, steps, kp, per, src, poll, res, dst, sum; };

struct One {
  Layer layer[MOST + 1];                 // behind the last one the head, as its QKV
  u32* logits;
  const int* pos;
  const float* cs;
  u32 *buf, *state;
  Shape shape[5];
  int layers, head, Hq, Hkv, room, slog, red, stride, part, ml, att, qkv;
  float eps, scale;
};

// The arguments, read where they are used: kept in registers over all phases they would
// be spilled.
typedef const __attribute__((address_space(4))) One Args;
__device__ __forceinline__ Args& args() {
  Args* p = (Args*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *p;
}

// The same of what follows from the thread's place.
__device__ __forceinline__ int here() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// Where an item's sum of squares lies. All blocks ask for all of them at a time: 16 to a
// memory channel's 256 bytes, not 64.
constexpr int SUMS = BLOCKS * 4;
__host__ __device__ __forceinline__ int sum_at(int item) { return (item >> 4) * 64 + (item & 15); }

// Of an item of a product, and a wave's share of it: first unit, its first step, steps in
// all, first pair.
struct Item { int p0, np, kp, per, steps, K, N, src, poll, res, dst, sum; };
struct Share { int u0, k0, left, pair; };

struct Lds {
  u32 dead, late, ticket;
  float inv;
  float cs[128];
  Item item[5];
  Share share[5][NW];
  u64 layer[2][12];                      // pointers of the layer at work and of the next
  u32 go;                                // steps a product's waves may ask for; ALL: its input is there
};
constexpr u32 ALL = 255;

__device__ __forceinline__ float as_float(u32 v) { return __builtin_bit_cast(float, v); }
__device__ __forceinline__ u32 as_u32(float v) { return __builtin_bit_cast(u32, v); }



template <typename T> __device__ __forceinline__ T same(T v) {     // in all lanes
  static_assert(sizeof(T) % 4 == 0, "");
  u32 w[sizeof(T) / 4];
  __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
  for (int i = 0; i < (int)sizeof(T) / 4; ++i) w[i] = __builtin_amdgcn_readfirstlane(w[i]);
  __builtin_memcpy(&v, w, sizeof(T));
  return v;
}

// Threads 0 .. 5 * NW - 1 work out the block's items.
__device__ __forceinline__ void divide(Lds* s, int item, int tid) {
  Args& a = args();
  const int kind = tid / NW, wave = tid % NW;
  if (kind >= 5) return;
  const auto& g = a.shape[kind];
  // of SwiGLU two results are a dword
  const int two = kind == GU, half = g.P >> two;
  const int p0 = (item * half >> 8) << two, np = ((item + 1) * half >> 8 << two) - p0;
  const int units = np << g.kp, mask = (1 << g.kp) - 1;
  const int u0 = wave * units / NW, u1 = (wave + 1) * units / NW;
  const int k0 = (u0 & mask) * g.per;
  s->share[kind][wave] = Share{
      u0, k0, ((u1 >> g.kp) - (u0 >> g.kp)) * g.steps + (u1 & mask) * g.per - k0,
      p0 + (u0 >> g.kp)};
  if (wave == 0)
    s->item[kind] = Item{p0, np, g.kp, g.per, g.steps, g.K, g.N, g.src, g.poll,
                         g.res + p0, g.dst + (p0 >> two), g.sum + sum_at(item)};
}
// Lanes 0 .. 11 fetch a layer's pointers.
__device__ __forceinline__ void fetch_layer(Lds* s, int ly, int lane) {
  if (lane < 12) s->layer[ly & 1][lane] = ((const u64*)&args().layer[ly])[lane];
}

// The weights of a job on their way through registers. The units of a wave lie behind one
// another, so that its steps run on from part to part and from pair to pair.
template <bool FP8>
struct Stream {
  static constexpr int E = FP8 ? 16 : 8, EL = FP8 ? 1 : 2, STEP = U * 64 * E;
  const int lane, steps, bytes, per;
  const Share sh;
  const long pair, second;               // bytes from a pair to the next, to its second row
  char* w;
  int k, left;                           // next step to fetch, and how many
  u32x4 buf[DEPTH][U][2];

  __device__ __forceinline__ Stream(const Item& t, const Share& h, const void* base, bool gu, int l)
      : lane(l), steps(t.steps), bytes(t.K * EL), per(t.per), sh(h), pair((long)bytes << !gu),
        second((long)bytes * (gu ? t.N : 1)), w((char*)base + h.pair * pair), k(h.k0), left(h.left) {}
  // Always as many loads, so that the compiler knows which are on the way; those past a
  // row's end, or behind the last step, read nothing.
  __device__ __forceinline__ void fetch(u32x4 (&d)[U][2]) {
    const int n = left > 0 ? bytes : 0, at = k * (STEP * EL) + lane * 16;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      d[u][0] = __builtin_amdgcn_raw_buffer_load_b128(
          __builtin_amdgcn_make_buffer_rsrc(w, 0, n, 0x00020000), at + u * 1024, 0, 2);
      d[u][1] = __builtin_amdgcn_raw_buffer_load_b128(
          __builtin_amdgcn_make_buffer_rsrc(w + second, 0, n, 0x00020000), at + u * 1024, 0, 2);
    }
    --left;
    if (++k == steps) {
      k = 0;
      w += pair;
    }
  }
  // Sums of the units with xs, to red.
  __device__ __forceinline__ void run(const u16* xs, float* red) {
    float acc0 = 0.f, acc1 = 0.f;
    int todo = sh.left, c = sh.k0, part = min(per, steps - c);
    float* to = red + sh.u0 * 2;
    // no way out between the steps: where ways meet, the compiler would wait for all
    // that any of them has asked for
    while (todo > 0) {
#pragma unroll
      for (int i = 0; i < DEPTH; ++i) {
        if (todo > 0) {
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const u16* xp = xs + c * STEP + (u * 64 + lane) * E;
            if (FP8) {
              const s16x8 x0 = ld8(xp), x1 = ld8(xp + 8);
              auto dot = [&](const u32x4& d) {
                float sum = 0.f;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                  const f32x2 c0 = __builtin_amdgcn_cvt_pk_f32_fp8(d[q], false);
                  const f32x2 c1 = __builtin_amdgcn_cvt_pk_f32_fp8(d[q], true);
                  const s16x8 y = q < 2 ? x0 : x1;
                  sum = fmaf(c0[0], bf2f((u16)y[q % 2 * 4]), sum);
                  sum = fmaf(c0[1], bf2f((u16)y[q % 2 * 4 + 1]), sum);
                  sum = fmaf(c1[0], bf2f((u16)y[q % 2 * 4 + 2]), sum);
                  sum = fmaf(c1[1], bf2f((u16)y[q % 2 * 4 + 3]), sum);
                }
                return sum;
              };
              acc0 += dot(buf[i][u][0]);
              acc1 += dot(buf[i][u][1]);
            } else {
              const s16x8 x = ld8(xp);
              acc0 += dot8_bf16(x, __builtin_bit_cast(s16x8, buf[i][u][0]));
              acc1 += dot8_bf16(x, __builtin_bit_cast(s16x8, buf[i][u][1]));
            }
          }
          ++c;
          --todo;
          if (--part == 0) {
            acc0 = wave_sum(acc0);
            acc1 = wave_sum(acc1);
            if (lane == 0) *(f32x2*)to = f32x2{acc0, acc1};
            acc0 = acc1 = 0.f;
            to += 2;
            if (c == steps) c = 0;
            part = min(per, steps - c);
          }
        }
        // behind the use, into the same registers
        asm volatile("" : "+v"(acc0), "+v"(acc1) :: "memory");
        fetch(buf[i]);
      }
    }
  }
};

typedef __attribute__((ext_vector_type(2))) u32 u32x2;

// A product's input, in xs.
template <bool FP8>
__device__ __forceinline__ void input(const u32* src, const u16* gain, int K, int steps, bool norm,
                                      Lds* s, u16* xs, u32x2 gv, int tid) {
  const int n4 = K / 4, STEP = U * 64 * (FP8 ? 16 : 8);
  const float inv = norm ? s->inv : 1.f;
  constexpr int NB = 8192 / (NW * 64 * 4);
  for (int c0 = 0; c0 < n4; c0 += NW * 64 * NB) {
    u32x2 v[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k)
      if (c0 + k * NW * 64 < n4) v[k] = ((const u32x2*)src)[min(c0 + k * NW * 64 + tid, n4 - 1)];
    for (int i = 0; ; ++i) {
      bool ok = true;
#pragma unroll
      for (int k = 0; k < NB; ++k)
        if (c0 + k * NW * 64 < n4) ok &= v[k][0] != NONE && v[k][1] != NONE;
      if (ok) break;
      if (i > LIMIT) { raise(&s->late); break; }
#pragma unroll
      for (int k = 0; k < NB; ++k)
        if (c0 + k * NW * 64 < n4)
          v[k] = __builtin_bit_cast(u32x2, ld_sc((const u64*)src + min(c0 + k * NW * 64 + tid, n4 - 1)));
    }
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int c = c0 + k * NW * 64 + tid;
      if (c < n4) {
        if (norm) {
          if (c != tid) gv = ((const u32x2*)gain)[c];
#pragma unroll
          for (int i = 0; i < 2; ++i)
            v[k][i] = (u32)El<u16>::st(lo(v[k][i]) * inv * lo(gv[i])) |
                      (u32)El<u16>::st(hi(v[k][i]) * inv * hi(gv[i])) << 16;
        }
        ((u32x2*)xs)[c] = v[k];
      }
    }
  }
  // a step's end behind the last column
  for (int c = n4 + tid; c < steps * STEP / 4; c += NW * 64) ((u32x2*)xs)[c] = u32x2{0, 0};
}

// What the wave that writes the results adds and scales them with.
struct Extra { u32 res; f32x2 s0, s1; };
template <bool FP8>
__device__ __forceinline__ Extra extra(const Item& t, int kind, const u32* res, const float* sc, int lane) {
  Extra x = {0, {1.f, 1.f}, {1.f, 1.f}};
  if ((kind == WO || kind == DOWN) && lane < t.np) {
    x.res = res[lane];
    for (int i = 0; x.res == NONE && i < LIMIT; ++i) x.res = ld_sc(res + lane);
  }
  if (FP8 && kind != HEAD) {
    const bool gu = kind == GU;
    const int q = 2 * min(lane, (gu ? t.np / 2 : t.np) - 1) + (gu ? t.p0 : 2 * t.p0);
    x.s0 = f32x2{sc[q], sc[q + 1]};
    if (gu) x.s1 = f32x2{sc[t.N + q], sc[t.N + q + 1]};
  }
  return x;
}

// Sums the parts of an item and hands its results on: one wave.
template <bool FP8>
__device__ __forceinline__ void output(const Item& t, int kind, u32* at, const float* sc,
                                       const float* red, Extra x, int lane) {
  auto sum = [&](int q) {
    f32x2 v = *(const f32x2*)(red + (q << t.kp) * 2);
    for (int i = 1; i < 1 << t.kp; ++i) {
      const f32x2 r = *(const f32x2*)(red + ((q << t.kp) + i) * 2);
      v[0] += r[0];
      v[1] += r[1];
    }
    return v;
  };
  if (kind == GU) {
    for (int q = lane; q < t.np / 2; q += 64) {
      f32x2 u = sum(2 * q), v = sum(2 * q + 1);
      if (FP8) {
        if (q != lane) {
          const float* c = sc + t.p0 + 2 * q;
          x.s0 = f32x2{c[0], c[1]};
          x.s1 = f32x2{c[t.N], c[t.N + 1]};
        }
        u = f32x2{u[0] * x.s0[0], u[1] * x.s1[0]};
        v = f32x2{v[0] * x.s0[1], v[1] * x.s1[1]};
      }
      st_sc(at + t.dst + q, pack(u[0] / (1.f + __expf(-u[0])) * u[1], v[0] / (1.f + __expf(-v[0])) * v[1]));
    }
    return;
  }
  float ssq = 0.f;
  for (int q = lane; q < t.np; q += 64) {
    f32x2 v = sum(q);
    if (FP8) {
      if (q != lane || kind == HEAD) {
        const float* c = sc + 2 * (t.p0 + q);
        x.s0 = f32x2{c[0], c[1]};
      }
      v = f32x2{v[0] * x.s0[0], v[1] * x.s0[1]};
    }
    if (kind == WO || kind == DOWN) {
      v[0] += lo(x.res);
      v[1] += hi(x.res);
    }
    const u32 o = pack(v[0], v[1]);
    if (kind == HEAD) {
      args().logits[t.p0 + q] = o;
    } else {
      st_sc(at + t.dst + q, o);
      ssq = fmaf(lo(o), lo(o), ssq);
      ssq = fmaf(hi(o), hi(o), ssq);
    }
  }
  if (kind == WO || kind == DOWN) {
    ssq = wave_sum(ssq);
    if (lane == 0) st_sc(at + t.sum, as_u32(ssq));
  }
}

// Sums the splits of the keys for an item of the columns: one wave. A lane has two
// columns of some of the splits.
template <int D>
__device__ __forceinline__ void sum_splits(Lds* s, int ly, int item) {
  Args& a = args();
  const int lane = here() & 63;
  const int P = a.Hq * D / 2, p0 = item * P >> 8, np = ((item + 1) * P >> 8) - p0;
  const int keys = min(*a.pos + 1, a.room), used = min(1 << a.slog, (keys + CHUNK - 1) / CHUNK);
  u32* at = a.buf + (long)ly * a.stride;
  const int dl = 31 - __builtin_clz(2 * np - 1), side = 64 >> dl;   // np up to 32
  const int d = lane & ((1 << dl) - 1), col = 2 * (p0 + min(d, np - 1)), hq = col / D;
  const u32 *mp = at + a.ml + hq * (2 << a.slog),
            *vp = at + a.part + hq * (D << a.slog) + (col & (D - 1));
  float m = M_NONE, ll = 0.f, t0 = 0.f, t1 = 0.f;
  for (int b = lane >> dl; b < used; b += 4 * side) {
    u32x2 ml[4], v[4];
    for (int i = 0; ; ++i) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int sp = min(b + k * side, used - 1);
        ml[k] = __builtin_bit_cast(u32x2, ld_sc((const u64*)(mp + sp * 2)));
        v[k] = __builtin_bit_cast(u32x2, ld_sc((const u64*)(vp + sp * D)));
      }
      bool ok = true;
#pragma unroll
      for (int k = 0; k < 4; ++k) ok &= ml[k][0] != NONE && ml[k][1] != NONE && v[k][0] != NONE && v[k][1] != NONE;
      if (__all(ok)) break;
      if (i > LIMIT || raised(&s->late)) { raise(&s->late); break; }
    }
    float mn = m;
#pragma unroll
    for (int k = 0; k < 4; ++k) mn = fmaxf(mn, as_float(ml[k][0]));
    const float al = __builtin_amdgcn_exp2f(m - mn);
    m = mn;
    ll *= al;
    t0 *= al;
    t1 *= al;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (b + k * side < used) {
        const float f = __builtin_amdgcn_exp2f(as_float(ml[k][0]) - m);
        ll = fmaf(f, as_float(ml[k][1]), ll);
        t0 = fmaf(f, as_float(v[k][0]), t0);
        t1 = fmaf(f, as_float(v[k][1]), t1);
      }
  }
  for (int o = 1 << dl; o < 64; o <<= 1) {
    const float mo = __shfl_xor(m, o), mn = fmaxf(m, mo);
    const float x = __builtin_amdgcn_exp2f(m - mn), y = __builtin_amdgcn_exp2f(mo - mn);
    ll = ll * x + __shfl_xor(ll, o) * y;
    t0 = t0 * x + __shfl_xor(t0, o) * y;
    t1 = t1 * x + __shfl_xor(t1, o) * y;
    m = mn;
  }
  const float r = ll > 0.f ? 1.f / ll : 0.f;
  if (lane < np) st_sc(at + a.att + p0 + lane, pack(t0 * r, t1 * r));
}

template <int D>
__device__ __forceinline__ void attend(Lds* s, char* lds, int ly, int item) {
  Args& a = args();
  constexpr int KS = D / 32, VC = D / 16;
  typedef __attribute__((ext_vector_type(VC / 2))) u32 vrow;
  const int tid = here(), lane = tid & 63, l15 = lane & 15, lg = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hk = item >> a.slog, split = item & ((1 << a.slog) - 1);
  if (hk >= a.Hkv) return;
  const int n = min(*a.pos + 1, a.room), last = n - 1;
  const int chunks = (n + CHUNK - 1) / CHUNK, used = min(1 << a.slog, chunks);
  if (split >= used) return;
  u16 *kc0 = (u16*)same(s->layer[ly & 1][10]), *vc0 = (u16*)same(s->layer[ly & 1][11]);
  const char *kc = (const char*)(kc0 + (long)hk * a.room * D);
  const char *vc = (const char*)(vc0 + (long)hk * a.room * D);
  const int G = a.Hq / a.Hkv;
  u32* at = a.buf + (long)ly * a.stride;
  s16x8* qp = (s16x8*)lds;                               // [KS][3][64]
  u16* fresh = (u16*)(qp + KS * 3 * 64);                 // [2][D]
  float* so = (float*)(fresh + 2 * D);                   // [NW][G][D], then m and l
  float* sml = so + NW * G * D;
  s16x8 kf[2][KS];
  vrow vf[8];
  int ch = split + used * w;
  auto load_k = [&](int k0) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const u32 kp = min(k0 + 16 * t + l15, last) * (D * 2) + 16 * lg;
#pragma unroll
      for (int k = 0; k < KS; ++k) kf[t][k] = *(const s16x8*)(kc + (kp + k * 64));
    }
  };
  auto load_v = [&](int k0) {
#pragma unroll
    for (int r = 0; r < 8; ++r)
      vf[r] = *(const vrow*)(vc + (u32)(min(k0 + (r & 4) * 4 + 4 * lg + (r & 3), last) * (D * 2) + 2 * VC * l15));
  };
  // the serving wave and the last one, which has the fewest keys, make the queries and the
  // new row ready
  const bool maker = w >= NW - 1;
  if (!maker) {
    if (ch < chunks) {
      load_k(ch * CHUNK);
      load_v(ch * CHUNK);
    }
    sync_lds();
  } else if (w == NW) {
    const u64* q = (const u64*)(at + a.qkv + (hk * G + min(l15, G - 1)) * (D / 2) + 4 * lg);
    u32x2 v[KS][2];
    for (int i = 0; ; ++i) {
#pragma unroll
      for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int e = 0; e < 2; ++e) v[k][e] = __builtin_bit_cast(u32x2, ld_sc(q + k * 8 + e));
      bool ok = true;
#pragma unroll
      for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int e = 0; e < 2; ++e) ok &= v[k][e][0] != NONE && v[k][e][1] != NONE;
      if (__all(ok)) break;
      if (i > LIMIT || raised(&s->late)) { raise(&s->late); break; }
    }
    float x[KS][8];
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[k][2 * e] = lo(v[k][e / 2][e % 2]);
        x[k][2 * e + 1] = hi(v[k][e / 2][e % 2]);
      }
#pragma unroll
    for (int k = 0; k < KS / 2; ++k)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const f32x2 t = *(const f32x2*)(s->cs + (k * 32 + 8 * lg + e) * 2);
        const float u = x[k][e], v = x[k + KS / 2][e];
        x[k][e] = u * t[0] - v * t[1];
        x[k + KS / 2][e] = v * t[0] + u * t[1];
      }
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      s16x8 p[3];
      parts3(x[k], p);
#pragma unroll
      for (int i = 0; i < 3; ++i) qp[(k * 3 + i) * 64 + lane] = p[i];
    }
    sync_lds();
  } else {
    // dimensions 2 i and 2 i + 1 of both halves
    const int i = lane & (D / 4 - 1);
    const u32* kr = at + a.qkv + (a.Hq + hk) * (D / 2) + i;
    const u32* vr = kr + a.Hkv * (D / 2);
    u32 v[4];
    for (int k = 0; ; ++k) {
      v[0] = ld_sc(kr);
      v[1] = ld_sc(kr + D / 4);
      v[2] = ld_sc(vr);
      v[3] = ld_sc(vr + D / 4);
      if (__all(v[0] != NONE && v[1] != NONE && v[2] != NONE && v[3] != NONE)) break;
      if (k > LIMIT || raised(&s->late)) { raise(&s->late); break; }
    }
    const f32x4 t = *(const f32x4*)(s->cs + 4 * i);
    const u32 k0 = (u32)El<u16>::st(lo(v[0]) * t[0] - lo(v[1]) * t[1]) |
                   (u32)El<u16>::st(hi(v[0]) * t[2] - hi(v[1]) * t[3]) << 16;
    const u32 k1 = (u32)El<u16>::st(lo(v[1]) * t[0] + lo(v[0]) * t[1]) |
                   (u32)El<u16>::st(hi(v[1]) * t[2] + hi(v[0]) * t[3]) << 16;
    u32* fr = (u32*)fresh + i;
    fr[0] = k0;
    fr[D / 4] = k1;
    fr[D / 2] = v[2];
    fr[D / 2 + D / 4] = v[3];
    sync_lds();
    if ((chunks - 1) % used == split) {
      const long row = ((long)hk * a.room + last) * (D / 2) + i;
      ((u32*)kc0)[row] = k0;
      ((u32*)kc0)[row + D / 4] = k1;
      ((u32*)vc0)[row] = v[2];
      ((u32*)vc0)[row + D / 4] = v[3];
    }
  }
  const bool mine_too = w < NW && ch < chunks;
  if (maker && mine_too) {
    load_k(ch * CHUNK);
    load_v(ch * CHUNK);
  }
  const int waves = min(NW, (chunks - split + used - 1) / used);   // that have keys
  if (mine_too) {
    const float c = a.scale * El<u16>::base;
    float m = M_NONE, ls = 0.f;
    f32x4 o[VC];
#pragma unroll
    for (int e = 0; e < VC; ++e) o[e] = f32x4{0.f, 0.f, 0.f, 0.f};
    int mine = lane;
    for (;;) {
      const int k0 = ch * CHUNK;
      if (ch == chunks - 1) {              // the new token's row is in LDS
#pragma unroll
        for (int t = 0; t < 2; ++t)
          if (k0 + 16 * t + l15 == last)
#pragma unroll
            for (int k = 0; k < KS; ++k) kf[t][k] = ld8(fresh + 8 * lg + k * 32);
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const int key = k0 + (r & 4) * 4 + 4 * lg + (r & 3);
          if (key == last) vf[r] = *(const vrow*)(fresh + D + VC * l15);
          if (key > last)                  // what lies past the keys counts 0
#pragma unroll
            for (int e = 0; e < VC / 2; ++e) vf[r][e] = 0;
        }
      }
      float sv[8];
      f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        asm volatile("" : "+v"(mine));     // read each time, and not all at once
#pragma unroll
        for (int i = 2; i >= 0; --i) {
          const s16x8 q = qp[(k * 3 + i) * 64 + mine];
          acc[0] = mma(kf[0][k], q, acc[0]);
          acc[1] = mma(kf[1][k], q, acc[1]);
        }
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          sv[4 * t + r] = k0 + 16 * t + 4 * lg + r > last ? -1.f / 0.f : acc[t][r] * c;
      float mx = fmaxf(sv[0], sv[1]);
#pragma unroll
      for (int i = 2; i < 8; ++i) mx = fmaxf(mx, sv[i]);
      const float mn = fmaxf(m, head_max(mx));
      const float al = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      float ps = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        sv[i] = __builtin_amdgcn_exp2f(sv[i] - mn);
        ps += sv[i];
      }
      ls = fmaf(ls, al, ps);
      s16x8 p[3];
      parts3(sv, p);
#pragma unroll
      for (int q = 0; q < VC / 2; ++q)
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
          u32x4 t;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            t[i] = __builtin_amdgcn_perm(vf[2 * i + 1][q], vf[2 * i][q],
                                         hf ? 0x07060302u : 0x05040100u);
          const s16x8 va = __builtin_bit_cast(s16x8, t);
          f32x4& oe = o[2 * q + hf];
#pragma unroll
          for (int r = 0; r < 4; ++r) oe[r] *= al;
#pragma unroll
          for (int i = 2; i >= 0; --i) oe = mma(va, p[i], oe);
        }
      ch += used * NW;
      if (ch >= chunks) break;
      load_k(ch * CHUNK);
      load_v(ch * CHUNK);
    }
    ls = head_sum(ls);
    if (l15 < G) {
      float* dst = so + (w * G + l15) * D;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int e = 0; e < VC; e += 4)
          *(f32x4*)(dst + VC * (4 * lg + r) + e) =
              f32x4{o[e][r], o[e + 1][r], o[e + 2][r], o[e + 3][r]};
      if (lg == 0) {
        sml[(w * G + l15) * 2] = m;
        sml[(w * G + l15) * 2 + 1] = ls;
      }
    }
  }
  sync_lds();
  for (int i = tid * 4; w < NW && i < G * D; i += 64 * NW * 4) {
    const int g = i / D, d = i - g * D;
    float mm = M_NONE, ll = 0.f;
    for (int q = 0; q < waves; ++q) mm = fmaxf(mm, sml[(q * G + g) * 2]);
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    for (int q = 0; q < waves; ++q) {
      const float f = __builtin_amdgcn_exp2f(sml[(q * G + g) * 2] - mm);
      const f32x4 t = *(const f32x4*)(so + (q * G + g) * D + d);
      ll = fmaf(f, sml[(q * G + g) * 2 + 1], ll);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = fmaf(f, t[e], v[e]);
    }
    const int hs = ((hk * G + g) << a.slog) + split;
    u32x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = as_u32(v[e]) == NONE ? NONE - 1 : as_u32(v[e]);
    __builtin_amdgcn_raw_buffer_store_b128(
        y, __builtin_amdgcn_make_buffer_rsrc(at + a.part, 0, (a.Hq * D << a.slog) * 4, 0x00020000),
        (hs * D + d) * 4, 0, 16);
    if (d == 0) {
      st_sc(at + a.ml + hs * 2, __builtin_bit_cast(u32, mm));
      st_sc(at + a.ml + hs * 2 + 1, __builtin_bit_cast(u32, ll));
    }
  }
}

template <bool FP8, int D>
__global__ void __launch_bounds__(THREADS, 1) k_decode_one(const One) {
  Args& a = args();
  extern __shared__ __align__(16) char lds[];
  __shared__ Lds s;
  const int tid = threadIdx.x;
  // the serving wave's few instructions are what other blocks wait for
  if (__builtin_amdgcn_readfirstlane(tid >> 6) == NW) __builtin_amdgcn_s_setprio(3);
  u32* state = a.state;
  if (tid == 0) {
    s.dead = s.late = s.go = 0;
    s.ticket = arrive(state, BLOCKS);
  }
  const int last = min(*a.pos + 1, a.room) - 1;
  if (tid < D) s.cs[tid] = a.cs[(long)max(last, 0) * D + tid];
  __syncthreads();
  const u32 rank = __builtin_amdgcn_readfirstlane(s.ticket);
  const bool fixed = rank != NONE;
  float* red = (float*)lds;
  u16* xs = (u16*)(lds + a.red);
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int layers = a.layers, head = a.head;
  int item = rank, ly = 0, kind = QKV;
  u32 turn = 0;                          // of products
  if (fixed) {
    divide(&s, item, tid);
    if (w == NW) fetch_layer(&s, 0, lane);
    __syncthreads();
  }
  for (;;) {
    if (!fixed) {
      __syncthreads();
      if (tid == 0) s.ticket = count(state + TICKET);
      __syncthreads();
      const u32 t = __builtin_amdgcn_readfirstlane(s.ticket);
      const int n = t / BLOCKS;
      if (n >= layers * PHASES + head) break;
      item = t % BLOCKS;
      ly = n / PHASES;
      const int order = n - ly * PHASES;             // QKV, ATT, SUM, WO, GU, DOWN
      kind = ly == layers ? HEAD : order == 0 ? QKV : order < 3 ? ATT + order - 1 : order - 2;
      divide(&s, item, tid);
      if (w == NW) fetch_layer(&s, ly, lane);
      __syncthreads();
    }
    if (kind == ATT) attend<D>(&s, lds + a.red, ly, item);
    const u32 base = turn << 8;
    if (fixed ? kind == ATT : kind == SUM) {
      if (w == NW) sum_splits<D>(&s, ly, item);
      kind = fixed ? WO : SUM;
    }
    if (kind == ATT || kind == SUM) continue;
    ++turn;
    const bool norm = kind != WO && kind != DOWN;
    const Item t = same(s.item[kind]);
    u32* at = args().buf + (long)ly * args().stride;
    if (w == NW) {
      const float* sc = (const float*)same(s.layer[ly & 1][4 + (kind & 3)]);
      // what tells that the input is there: sums of squares, or the last dword of what
      // each item writes
      const u32* flag = at + t.poll;
      int off[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = k * 64 + lane;
        off[k] = norm ? sum_at(i) : ((i + 1) * (t.K / 2) >> 8) - 1;
      }
      if (raised(&s.late)) raise(&s.dead);
      u32 v[4];
      if (kind == WO)
        __hip_atomic_store(&s.go, base | 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __builtin_amdgcn_s_sleep(50);
      for (int i = 0; ; ++i) {
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = ld_sc(flag + off[k]);
        if (__all(v[0] != NONE && v[1] != NONE && v[2] != NONE && v[3] != NONE)) break;
        if (i > LIMIT || raised(&s.dead)) { raise(&s.dead); break; }
      }
      if (norm) {
        const float ss = wave_sum((as_float(v[0]) + as_float(v[1])) + (as_float(v[2]) + as_float(v[3])));
        if (lane == 0) s.inv = rsqrtf(ss / (float)t.K + args().eps);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __hip_atomic_store(&s.go, base | ALL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      sync_lds();
      const Extra x = extra<FP8>(t, kind, at + t.res, sc, lane);
      if (fixed && kind == QKV) fetch_layer(&s, ly + 1, lane);
      sync_lds();
      if (__builtin_amdgcn_readfirstlane(raised(&s.dead))) break;
      output<FP8>(t, kind, at, sc, red, x, lane);
    } else {
      const u16* gain = (const u16*)same(s.layer[ly & 1][8 + ((kind & 3) >> 1)]);
      Stream<FP8> f(t, same(s.share[kind][w]), (const void*)same(s.layer[ly & 1][kind & 3]), kind == GU, lane);
      u32x2 gv = {0, 0};
      if (norm) gv = ((const u32x2*)gain)[min(tid, t.K / 4 - 1)];
      u32 g;
      if (kind == WO)                    // the splits' sums first
        do {
          g = __builtin_amdgcn_readfirstlane(raised(&s.go)) - base;
        } while (g > ALL || g == 0);
#pragma unroll
      for (int i = 0; i < DEPTH; ++i) f.fetch(f.buf[i]);
      do {
        g = __builtin_amdgcn_readfirstlane(raised(&s.go)) - base;
      } while (g != ALL);
      asm volatile("" ::: "memory");
      input<FP8>(at + t.src, gain, t.K, t.steps, norm, &s, xs, gv, tid);
      sync_lds();
      f.run(xs, red);
      sync_lds();
      if (__builtin_amdgcn_readfirstlane(raised(&s.dead))) break;
    }
    if (fixed) {
      if (kind == HEAD) break;
      if (kind == DOWN && ++ly == layers) {
        if (!head) break;
        kind = HEAD;
      } else {
        kind = kind == QKV ? ATT : (kind + 1) & 3;
      }
    }
  }
  if (raised(&s.dead) && args().logits)
    for (int i = tid; i < args().shape[HEAD].P; i += THREADS) args().logits[i] = 0x7fc07fc0u;
}

// Empties what the blocks hand to each other and all launches' state, and puts the first
// residual there.
__global__ void __launch_bounds__(256)
k_decode_one_begin(u32* ws, long dwords, int stat, const u32* x, int C, int sums) {
  const long i0 = blockIdx.x * 256 + threadIdx.x, n = gridDim.x * 256;
  // the first residual and its sums are not
  for (long i = sums + SUMS + i0 * 4; i < dwords - stat; i += n * 4)
    *(u32x4*)(ws + i) = u32x4{NONE, NONE, NONE, NONE};
  if (i0 < stat) ws[dwords - stat + i0] = 0;
  if (blockIdx.x != gridDim.x - 1) return;
  const int t = threadIdx.x, P = C / 2;
  float ss = 0.f;
#pragma unroll 4
  for (int i = t; i < P; i += 256) {
    const u32 v = x[i];
    ws[i] = v == NONE ? NONE - 1 : v;
    ss = fmaf(lo(v), lo(v), ss);
    ss = fmaf(hi(v), hi(v), ss);
  }
  const u32 z = as_u32(ss);
  ws[sums + sum_at(t)] = z == NONE ? NONE - 1 : z;
}

}  // namespace

// vocab: rows of the head. blocks: of a launch, 256, fewer to have items taken by ticket.
struct OneShape { int layers, C, I, Hq, Hkv, D, room, vocab, fp8, blocks; float eps, scale; };

namespace {

inline Shape shape_of(int pairs, int N, int K, bool fp8, int src, int poll, int res, int dst, int sum) {
  const int step = U * (fp8 ? 1024 : 512);
  Shape s{pairs, N, K, (K + step - 1) / step, 0, 0, src, poll, res, dst, sum};
  // as many parts of K as make the waves' shares even
  const int np = (pairs + BLOCKS - 1) / BLOCKS;
  for (int kp = 0, best = 1 << 30; kp <= 4 && 1 << kp <= s.steps; ++kp) {
    const int per = (s.steps + (1 << kp) - 1) >> kp, most = ((np << kp) + NW - 1) / NW * per;
    if (((1 << kp) - 1) * per < s.steps && most < best) best = most, s.kp = kp, s.per = per;
  }
  return s;
}

// What launches share, and the dwords of room.
inline One plan(const OneShape& p, long& dwords, int& bytes) {
  One a{};
  a.Hq = p.Hq; a.Hkv = p.Hkv; a.room = p.room;
  a.eps = p.eps; a.scale = p.scale;
  const int HD = p.Hq * p.D, W = (p.Hq + 2 * p.Hkv) * p.D, G = p.Hq / p.Hkv;
  while (p.Hkv << (a.slog + 1) <= BLOCKS) ++a.slog;
  int o = 0;
  auto room = [&](int n) { const int at = o; o += (n + 3) / 4 * 4; return at; };
  const int h = room(p.C / 2), hs = room(SUMS);
  a.qkv = room(W / 2);
  const int h1 = room(p.C / 2), s1 = room(SUMS), act = room(p.I / 2);
  a.att = room(HD / 2);
  a.part = room(HD << a.slog);
  a.ml = room(p.Hq * 2 << a.slog);
  a.stride = o;
  a.shape[QKV] = shape_of(W / 2, W, p.C, p.fp8, h, hs, h, a.qkv, hs);
  a.shape[WO] = shape_of(p.C / 2, p.C, HD, p.fp8, a.att, a.att, h, h1, s1);
  a.shape[GU] = shape_of(p.I, p.I, p.C, p.fp8, h1, s1, h1, act, s1);
  // to the next layer's room
  a.shape[DOWN] = shape_of(p.C / 2, p.C, p.I, p.fp8, act, act, h1, o + h, o + hs);
  a.shape[HEAD] = shape_of(p.vocab / 2, p.vocab, p.C, p.fp8, h, hs, h, h, hs);
  dwords = (long)o * p.layers + hs + SUMS + (p.layers + MOST - 1) / MOST * STATE;
  const int step = U * (p.fp8 ? 1024 : 512), widest = max(max(p.C, p.I), HD);
  int units = 0;
  for (const Shape& g : a.shape) units = max(units, ((g.P + 2 * BLOCKS - 1) / BLOCKS + 1) << g.kp);
  a.red = (units * 8 + 15) / 16 * 16;
  const int xs = (widest + step - 1) / step * step * 2;
  const int att = p.D / 32 * 3 * 1024 + 2 * p.D * 2 + NW * G * (p.D + 2) * 4;
  // more than half of a CU's: one block each
  bytes = max(a.red + max(xs, att), 84 * 1024);
  return a;
}

template <bool FP8, int D>
void launch(const One& a, int blocks, int bytes, hipStream_t stream) {
  allow_lds(k_decode_one<FP8, D>, bytes);
  hipLaunchKernelGGL((k_decode_one<FP8, D>), dim3(blocks), dim3(THREADS), bytes, stream, a);
}

}  // namespace

extern "C" {

// Bytes of room that a step takes, 0 if this cannot run it.
long fei_decode_one_room(const OneShape* p) {
  const int HD = p->Hq * p->D, e = p->fp8 ? 16 : 8;
  // more blocks than items would take rows past the products' ends
  if (p->blocks < 1 || p->blocks > BLOCKS || p->layers <= 0 || p->Hkv <= 0 || p->Hkv > BLOCKS || p->Hq % p->Hkv || p->Hq / p->Hkv > 16 ||
      (p->D != 64 && p->D != 128) || p->C % e || p->I % e || HD % e || p->vocab % 2 ||
      // each item has rows, and what one wave writes of them it has registers for
      p->C < 512 || p->I < 512 || HD < 512 || p->vocab < 512 || p->C > 16384 || HD > 16384 ||
      p->I > 1 << 20 || p->vocab > 1 << 22 || p->room <= 0 || (long)p->room * p->D * 2 >= 1l << 31)
    return 0;
  long dwords;
  int bytes;
  plan(*p, dwords, bytes);
  return bytes <= 152 * 1024 ? dwords * 4 : 0;
}

// ptrs: of each layer w of QKV, output, gates and up, down; their rows' scales (fp8, else
// null); gains of both norms; caches of k and v [Hkv, room, D]. Then w and scales of the
// head and the gain in front of it. x [C], logits [vocab] bfloat16; ws: fei_decode_one_room
// bytes on 16. At pos[0] keys and values are written. cs: see attn_decode.hip.
void fei_decode_one(const void* const* ptrs, const OneShape* p, const void* x, void* logits,
                    void* ws, const int* pos, const float* cs, hipStream_t stream) {
  long dwords;
  int bytes;
  One a = plan(*p, dwords, bytes);
  const int launches = (p->layers + MOST - 1) / MOST;
  u32 *buf = (u32*)ws, *state = buf + dwords - launches * STATE;
  a.pos = pos;
  a.cs = cs;
  hipLaunchKernelGGL(k_decode_one_begin, dim3(256), dim3(256), 0, stream, buf, dwords, launches * STATE,
                     (const u32*)x, p->C, a.shape[QKV].poll);
  for (int i = 0; i < launches; ++i) {
    const int done = i * MOST;
    a.buf = buf + (long)done * a.stride;
    a.state = state + i * STATE;
    a.layers = min(MOST, p->layers - done);
    for (int k = 0; k < a.layers; ++k) a.layer[k] = *(const Layer*)(ptrs + 12 * (done + k));
    a.head = i == launches - 1;
    if (a.head) {
      const void* const* t = ptrs + 12 * p->layers;
      Layer& l = a.layer[a.layers];
      l.w[0] = t[0];
      l.s[0] = (const float*)t[1];
      l.gain[0] = (const u16*)t[2];
      a.logits = (u32*)logits;
    }
    if (p->D == 128) {
      if (p->fp8) launch<true, 128>(a, p->blocks, bytes, stream);
      else launch<false, 128>(a, p->blocks, bytes, stream);
    } else {
      if (p->fp8) launch<true, 64>(a, p->blocks, bytes, stream);
      else launch<false, 64>(a, p->blocks, bytes, stream);
    }
  }
}

}  // extern "C"
