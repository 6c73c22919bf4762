// Products of hundreds of rows and more with a weight matrix (gfx950):
// out[M, N] = x[M, K] @ W[N, K]^T in bfloat16 with float32 sums, where what follows
// the product is done on its sums, or K is cut so that all CUs have a tile.
#include <algorithm>
#include <type_traits>

#include "fei_epilogue.h"
#include "fei_mma.h"

namespace {

enum {
  TILE_BF16 = 0,
  TILE_SWIGLU = 1,     // W has N rows of gates, then N of up
  TILE_GELU = 2,       // with a bias per column
  TILE_RELU2 = 3,
  TILE_PARTS = 4,      // float32 sums of a part of K, [parts][M][N]
  TILE_BIAS = 5,       // a bias per column alone
};

__device__ __forceinline__ int uniform(int v) {
  return __builtin_amdgcn_readfirstlane(v);
}

struct TileArgs {
  void* out;
  const u16* x;
  const u16* w;
  const u16* bias;
  const int* rows;     // k_tile_counted: how many of the M rows there are
  long os, xs;         // rows of out and x are this far apart
  int M, N, K, nx, parts;
};

template <int N>
using Int = std::integral_constant<int, N>;

// A tile's columns of out, and of W a half of them for gates where there are gates.
template <int WM, int XI, int WI, int EPI>
struct Shape {
  static constexpr int rows = 32 * WM * XI, width = 32 * (8 / WM) * WI;
  static constexpr int columns = EPI == TILE_SWIGLU ? width / 2 : width;
};

// A block's part of the work: of its XCD's tiles from id ``first`` on, each in MC * NC
// pieces, ``count`` in all.
struct Share {
  int first, count;
};

// A block: 8 waves, two on a SIMD, that share tiles of 32 WM XI rows of x and
// 32 WN WI rows of W (SWIGLU: half of them gates, the others the same of up),
// WN = 8 / WM, 64 steps of K at a time. Both operands come in halves; a wave has
// XI x WI fragments of each of the four quarters. Waves 0-3 are one
// barrier ahead of waves 4-7, so that of the two waves on a SIMD one multiplies
// while the other reads fragments and sends loads. A step is two such turns:
//   first half of x, both of W -> its two quarters of the tile
//   second half of x           -> the other two
// Each group loads its half of x and W, straight to LDS, two steps ahead of the
// products, in two buffers: what a turn has read is free when the turn's barrier
// is past (reads are waited for in front of it), and is filled again in the next.
// Loads are waited for a turn before they are read, by their number, so that
// those of a step and more stay in flight. The stream of loads runs on
// into the block's next tile, and results are written while the other group
// multiplies: a tile's first loads and last stores cost little then.
//
// The 16-byte places of a row in LDS are permuted by the row, in the address that
// a lane loads from, so that the reads of 16 rows spread over the banks. Row
// i of a fragment of W is row 4 WI (i / 4) + 4 j + i % 4 of the wave's, j the
// fragment, so that a lane has 4 WI consecutive columns of a row of out.
//
// Blocks of an XCD take consecutive tiles, eight of rows times all of columns, rows
// first: its L2 holds what they share. XCDs start at different steps of K, or
// all would read the same columns of W, rows of which lie a power of two apart,
// from the same memory channels.
//
// Bound by the matrix units: 2310 cycles a step of 256 x 256 x 64, of which they
// need 2048, at the 1.7 to 2.1 GHz that the card keeps under this load; four turns
// of one quarter took 2510, and more where both groups ran the same branching code.
// Against the library, us: 2 x 14336 x 4096 of 2048 rows with SwiGLU 348 (360 + 33
// for the pass of its own); 3072 x 768 of 16384 with bias and GELU 104 to
// 109 (68.5 + 52); 4096 x 14336 of 2048 in two parts 170 (204); 8192^3 706 (700).
//
// B: the Shape in which tiles are counted.
template <typename B, int WM, int XI, int WI, int EPI>
__device__ __forceinline__ void run_tiles(const TileArgs& g, const Share share,
                                          u16* const buf, int M, int nm) {
  typedef Shape<WM, XI, WI, EPI> P;
  constexpr int WN = 8 / WM;
  constexpr int HA = 16 * WM * XI, HB = 16 * WN * WI;   // rows of a half
  constexpr int TM = 2 * HA, TN = 2 * HB;
  constexpr int PA = HA / 32, PB = HB / 32;             // loads of a wave
  constexpr bool PAIR = EPI == TILE_SWIGLU;
  constexpr bool BIAS = EPI == TILE_GELU || EPI == TILE_BIAS;
  constexpr int STAGE = (TM + TN) * 64;
  constexpr int MC = B::rows / P::rows, NC = B::columns / P::columns;
  u16* const lbias = buf + 2 * STAGE;                   // [4 tiles][512]
  const int N = g.N, K = g.K, parts = g.parts;
  const int total = g.nx * nm;
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, slots = gridDim.x >> 3;
  const int lim = share.count;
  if (slot >= lim) return;
  const int all = K / 64;
  const bool spread = (long)M * K <= 2 << 20;
  struct Tile { int m0, n0, part, first, steps, turn; };
  auto locate = [&](int i) __attribute__((always_inline)) {
    Tile t;
    int id = share.first + i / (MC * NC);
    t.part = uniform(id / total);
    id -= t.part * total;
    const int g0 = uniform(id / (8 * g.nx)) * 8, gm = min(8, nm - g0);
    const int gr = id - g0 * g.nx, c = uniform(gr / gm);
    t.n0 = c * B::columns + i % NC * P::columns;
    t.m0 = (g0 + gr - c * gm) * B::rows + i / NC % MC * P::rows;
    t.first = uniform((int)((u32)(t.part * all) / (u32)parts));
    t.steps = uniform((int)((u32)((t.part + 1) * all) / (u32)parts)) - t.first;
    t.turn = uniform((u32)(xcd * t.steps / 8 + (spread ? 3 * c : 0)) % (u32)t.steps);
    return t;
  };
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = uniform(tid >> 6), grp = wid >> 2, w4 = wid & 3;
  const int wm = WM == 4 ? w4 : grp, wn = WM == 4 ? grp : w4;
  const u32 lds = (u32)(uintptr_t)(__attribute__((address_space(3))) u16*)buf;

  // the wave's stream of loads: its pieces of 8 rows of its group's halves
  Tile ld = locate(slot);
  int li = slot, lk = 0, ltile = 0;
  bool live = true;                        // there are steps left to load
  u32 ls = 0;                              // buffer, in bytes
  u32 oa[PA], ob[PB];
  const u16 *pa, *pb;
  auto aim = [&]() __attribute__((always_inline)) {
    // a lane's share is made anew for each tile: kept, it would not fit
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int r8 = ln >> 3, c8 = ln & 7;
    const int ma = ld.m0 + grp * HA, last_a = max(M - 1 - ma, 0);
    pa = g.x + min(ma, M - 1) * g.xs + ld.first * 64;
#pragma unroll
    for (int i = 0; i < PA; ++i)
      oa[i] = (u32)min((w4 * PA + i) * 8 + r8, last_a) * (u32)(g.xs * 2) +
              (c8 ^ r8) * 16;
    const int nb = PAIR ? ld.n0 : ld.n0 + grp * HB, last_b = max(N - 1 - nb, 0);
    pb = g.w + ((long)min(nb, N - 1) + (PAIR && grp ? N : 0)) * K +
         ld.first * 64;
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      const int r = (w4 * PB + i) * 8 + r8;
      const int f = (r & 3) | ((r % (16 * WI) / (4 * WI)) & 1) << 2;
      ob[i] = (u32)min(r, last_b) * (u32)(K * 2) + (c8 ^ f) * 16;
    }
    if (BIAS && wid == 0)
      load_lds_from(g.bias, (u32)min(ld.n0 + (ln & 31) * 8, N - 8) * 2,
                    lds + 4 * STAGE + (ltile & 3) * 1024);
  };
  aim();
  auto column = [&]() __attribute__((always_inline)) {
    const int t = lk + ld.turn;
    return (t < ld.steps ? t : t - ld.steps) * 64;
  };
  auto load_a = [&]() __attribute__((always_inline)) {
    if (!live) return;
    const u16* p = pa + column();
    const u32 d = lds + ls + (grp * HA + w4 * PA * 8) * 128;
#pragma unroll
    for (int i = 0; i < PA; ++i) load_lds_from(p, oa[i], d + i * 1024);
  };
  auto load_b = [&]() __attribute__((always_inline)) {
    if (!live) return;
    const u16* p = pb + column();
    const u32 d = lds + ls + (TM + grp * HB + w4 * PB * 8) * 128;
#pragma unroll
    for (int i = 0; i < PB; ++i) load_lds_from(p, ob[i], d + i * 1024);
  };
  auto advance = [&]() __attribute__((always_inline)) {
    ls ^= STAGE * 2;
    if (__builtin_expect(lk + 1 < ld.steps, 1)) {
      ++lk;
    } else if (li + slots < lim) {
      li += slots;
      ++ltile;
      ld = locate(li);
      lk = 0;
      aim();
    } else {
      live = false;
    }
  };

  s16x8 fa[XI][2], fb[2][WI][2];
  const int l15 = lane & 15, lg = lane >> 4;
  const int pl0 = (lg ^ (l15 & 7)) * 8, pl1 = ((4 + lg) ^ (l15 & 7)) * 8;
  const int xa = (wm * 16 * XI + l15) * 64;
  const int wa = (TM + wn * 16 * WI + 4 * WI * (l15 >> 2) + (l15 & 3)) * 64;
  int cs = 0;                              // buffer of the products
  auto read_a = [&](int h) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const u16* p = buf + cs + xa + (h * HA + i * 16) * 64;
      fa[i][0] = ld8(p + pl0);
      fa[i][1] = ld8(p + pl1);
    }
  };
  auto read_b = [&](int h) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < WI; ++j) {
      const u16* p = buf + cs + wa + (h * HB + 4 * j) * 64;
      fb[h][j][0] = ld8(p + pl0);
      fb[h][j][1] = ld8(p + pl1);
    }
  };
  f32x4 acc[2][2][XI][WI];
  auto clear = [&](auto ha, auto hb) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XI; ++i)
#pragma unroll
      for (int j = 0; j < WI; ++j)
        acc[ha.value][hb.value][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  clear(First{}, First{});
  clear(First{}, Second{});
  clear(Second{}, First{});
  clear(Second{}, Second{});
  auto barrier = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // until all but a step's loads, the last sent, have arrived; behind the end all
  // but those of a half of x where ``half``
  auto wait = [&](auto half) __attribute__((always_inline)) {
    if (__builtin_expect(live, 1))
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PA + PB) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(half.value * PA) : "memory");
  };
  auto product = [&](auto ha) __attribute__((always_inline)) {
    constexpr int a = decltype(ha)::value;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    barrier();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int i = 0; i < XI; ++i)
#pragma unroll
          for (int j = 0; j < WI; ++j)
            acc[a][b][i][j] = mma(fb[b][j][kk], fa[i][kk], acc[a][b][i][j]);
    __builtin_amdgcn_s_setprio(0);
    barrier();
  };
  // results of a quarter of the tile (SWIGLU: of a half's gates and ups)
  auto store = [&](auto ha, auto hb, const Tile& t, int tile)
                   __attribute__((always_inline)) {
    constexpr int a = decltype(ha)::value, b = decltype(hb)::value, V = 4 * WI;
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int nr = b * HB + wn * 16 * WI + V * (ln >> 4), n = t.n0 + nr;
    u16 add[V];
    if (BIAS)
#pragma unroll
      for (int j = 0; j < WI; ++j)
        __builtin_memcpy(add + 4 * j, lbias + (tile & 3) * 512 + nr + 4 * j, 8);
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int m = t.m0 + a * HA + wm * 16 * XI + i * 16 + (ln & 15);
      if (m < M && n < N) {
        if (EPI == TILE_PARTS) {
          float* p = (float*)g.out + ((long)t.part * g.M + m) * N + n;
#pragma unroll
          for (int j = 0; j < WI; ++j)
            if (n + 4 * j < N) *(f32x4*)(p + 4 * j) = acc[a][b][i][j];
        } else {
          u16 v[V];
#pragma unroll
          for (int j = 0; j < WI; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              float y = acc[a][b][i][j][e];
              if (PAIR) y = swiglu(y, acc[a][1][i][j][e]);
              if (BIAS) y += bf2f(add[j * 4 + e]);
              if (EPI == TILE_GELU) y = gelu_erf(y);
              if (EPI == TILE_RELU2) y = relu2(y);
              v[j * 4 + e] = El<u16>::st(y);
            }
          u16* p = (u16*)g.out + m * g.os + n;
          constexpr int W = WI % 2 ? 4 : 8;             // of a store; N % 8 == 0
#pragma unroll
          for (int c = 0; c < V; c += W)
            if (n + c < N)
              __builtin_memcpy(__builtin_assume_aligned(p + c, 2 * W), v + c,
                               2 * W);
        }
      }
      __builtin_amdgcn_sched_barrier(0);   // a row at a time: registers
    }
    clear(ha, hb);
    if (PAIR) clear(ha, Second{});
  };

  int ct = 0;
  auto step = [&](const Tile& t, auto lastc, auto gc)
                  __attribute__((always_inline)) {
    constexpr bool last = decltype(lastc)::value, late = decltype(gc)::value;
    read_a(0);
    read_b(0);
    read_b(1);
    if (late) {
      load_a();
      wait(First{});                       // this step's second half of x
      advance();
    }
    product(First{});
    read_a(1);
    if (!late) load_a();
    load_b();
    wait(gc);                              // all else of the next step
    if (!late) advance();
    if (last) {
      store(First{}, First{}, t, ct);
      if (!PAIR) store(First{}, Second{}, t, ct);
    }
    product(Second{});
    if (last) {
      store(Second{}, First{}, t, ct);
      if (!PAIR) store(Second{}, Second{}, t, ct);
    }
    cs ^= STAGE;
  };
  // one loop a group, so that neither branches on it
  auto run = [&](auto gc) __attribute__((always_inline)) {
    for (int i = slot; i < lim; i += slots, ++ct) {
      const Tile t = locate(i);
      for (int k = 0; k < t.steps - 1; ++k) step(t, First{}, gc);
      step(t, Second{}, gc);
    }
  };
  if (grp == 0) {
    load_a();
    load_b();
    advance();
    load_a();
    load_b();
    wait(First{});
    advance();
    barrier();
    run(First{});
    barrier();
  } else {
    load_b();
    load_a();
    advance();
    load_b();
    wait(Second{});
    barrier();
    barrier();
    run(Second{});
  }
}

// MC * NC = 2: where an XCD's CUs have a last round of tiles for half of them or less, its
// tiles are cut, rows or columns, so that all CUs have one. A kernel of its own: where
// nothing is cut the other is faster by 1 to 2 us of 35 to 300. Us, uncut and cut: 2 x
// 6144 x 2048 with SwiGLU, 1301 rows 70, 66; 2304 x 768 with bias and GELU, 10336 rows
// 61, 56; 3072 x 768, 6144 rows 48, 46; 2 x 14336 x 4096, 2048 rows, 3 1/2 rounds 362,
// 361 by itself, 9 less in a model's layers: with CUs idle the others keep a higher clock,
// so that a long round gains little.
template <int WM, int XI, int WI, int EPI, int MC, int NC>
__global__ void __launch_bounds__(512, 2) k_tile(TileArgs g) {
  typedef Shape<WM, XI, WI, EPI> B;
  extern __shared__ __align__(16) u16 buf[];
  const int M = g.M, nm = (M + B::rows - 1) / B::rows;
  const int tiles = g.nx * nm * g.parts, per = (tiles + 7) / 8;
  const int xcd = blockIdx.x & 7, slots = gridDim.x >> 3;
  const int lim = min(per, tiles - xcd * per);          // tiles of the XCD
  const int rest = MC * NC > 1 && lim > 0 ? uniform(lim % slots) : 0;
  const int cut = rest * MC * NC <= slots ? rest : 0;
  run_tiles<B, WM, XI, WI, EPI>(g, Share{xcd * per, lim - cut}, buf, M, nm);
  if (MC * NC > 1 && cut) {
    // what is in LDS has been read
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    run_tiles<B, WM, XI / MC, WI / NC, EPI>(
        g, Share{xcd * per + lim - cut, cut * MC * NC}, buf, M, nm);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

template <int WM, int XI, int WI, int EPI, int MC = 1, int NC = 1>
void launch(TileArgs g, hipStream_t stream) {
  typedef Shape<WM, XI, WI, EPI> B;
  constexpr int lds = 2 * (B::rows + B::width) * 128 + 4096;
  g.nx = (g.N + B::columns - 1) / B::columns;
  const long nm = (g.M + B::rows - 1) / B::rows;
  const long per = (nm * g.nx * g.parts + 7) / 8;       // tiles of an XCD
  const int slots = (int)std::min(32L, per);            // a block a CU
  auto go = [&](auto kernel) {
    allow_lds(kernel, lds);
    hipLaunchKernelGGL(kernel, dim3(8 * slots), dim3(512), lds, stream, g);
  };
  const int rest = (int)(per % slots);
  if (MC * NC > 1 && rest && rest * MC * NC <= slots)
    go(k_tile<WM, XI, WI, EPI, MC, NC>);
  else
    go(k_tile<WM, XI, WI, EPI, 1, 1>);
}

// The same of as many rows as the device finds, in the tiles that suit them: by the time
// of a round of each, us of a step of 64 of K with one tile on the chip, what comes on
// top with one on every CU (TILES of ops/tiles.py), and of a round. 12 layers of 768, texts of 64 to 256 tokens,
// 10336 rows of 16384: 2304 x 768 in tiles of 256 x 256, which suit 16384, 45.6 us, of 192
// x 256 36.2; 768 x 768 21.5 and, of 128 x 256, 16.3; 768 x 3072 56.3, 46.2; 3072 x 768
// with GELU 63, 72 of either other. Rests are not cut: with 12 steps of K that gains less
// than to start anew costs. Blocks without a tile leave at once.
template <int EPI>
__global__ void __launch_bounds__(512, 2) k_tile_counted(const TileArgs all) {
  extern __shared__ __align__(16) u16 buf[];
  TileArgs g = all;
  const int M = uniform(min(*g.rows, g.M));
  const float steps = (float)(g.K / 64 / g.parts);
  // us of GELU on 256 x 256 sums
  const float act = EPI == TILE_GELU ? 14.f : 0.f;
  auto tiles = [&](int rows, int width) {
    return (M + rows - 1) / rows * ((g.N + width - 1) / width) * g.parts;
  };
  auto time = [&](int rows, int width, float alone, float full) {
    const int n = tiles(rows, width);
    const float round = steps * alone + 3.f + act * (float)(rows * width) / 65536.f;
    return (float)((n + 255) / 256) * round + steps * full * (float)n / 256.f;
  };
  const float t0 = time(256, 256, 1.f, 0.46f), t1 = time(256, 192, 0.875f, 0.36f);
  const float t2 = time(192, 256, 0.82f, 0.34f), t3 = time(128, 256, 0.73f, 0.13f);
  auto run = [&](auto wm, auto xi, auto wi) __attribute__((always_inline)) {
    typedef Shape<decltype(wm)::value, decltype(xi)::value, decltype(wi)::value, EPI> B;
    g.nx = (g.N + B::columns - 1) / B::columns;
    const int nm = (M + B::rows - 1) / B::rows;
    const int per = (g.nx * nm * g.parts + 7) / 8, xcd = blockIdx.x & 7;
    run_tiles<B, decltype(wm)::value, decltype(xi)::value, decltype(wi)::value, EPI>(
        g, Share{xcd * per, min(per, g.nx * nm * g.parts - xcd * per)}, buf, M, nm);
  };
  const float best = fminf(fminf(t0, t1), fminf(t2, t3));
  switch (uniform(best == t0 ? 0 : best == t1 ? 1 : best == t2 ? 2 : 3)) {
    case 0: run(Int<2>{}, Int<4>{}, Int<2>{}); break;
    case 1: run(Int<4>{}, Int<2>{}, Int<3>{}); break;
    case 2: run(Int<2>{}, Int<3>{}, Int<2>{}); break;
    default: run(Int<2>{}, Int<2>{}, Int<2>{});
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

template <int EPI>
void launch_counted(const TileArgs& g, hipStream_t stream) {
  constexpr int lds = 2 * 512 * 128 + 4096;
  allow_lds(k_tile_counted<EPI>, lds);
  hipLaunchKernelGGL(k_tile_counted<EPI>, dim3(256), dim3(512), lds, stream, g);
}

template <int EPI>
void by_size(int rows, int width, const TileArgs& g, hipStream_t stream) {
  if (rows == 192) launch<2, 3, 2, EPI, 1, 2>(g, stream);
  else if (rows == 128) launch<2, 2, 2, EPI>(g, stream);
  else if (width == 256) launch<2, 4, 2, EPI, 2, 1>(g, stream);
  else if (width == 192) launch<4, 2, 3, EPI, 2, 1>(g, stream);
  else launch<4, 2, 2, EPI>(g, stream);
}

}  // namespace

extern "C" {

// Rows of x (xs apart) and w on 16 bytes and less than 2^24 values apart, K % 64 == 0
// and at least 64 a part, N % 8 == 0; rows of out (os apart) on 16 bytes, as the bias. A tile has rows x width
// rows of x and w: 256 x 256, 192 or 128, 192 x 256, 128 x 256. epi: see above; parts
// are 1 but for TILE_PARTS.
void fei_tile(void* out, long os, const void* x, long xs, const void* w,
              const void* bias, int M, int N, int K, int epi, int rows,
              int width, int parts, hipStream_t stream) {
  const TileArgs g = {out, (const u16*)x, (const u16*)w, (const u16*)bias, nullptr,
                      os, xs, M, N, K, 0, parts};
  switch (epi) {
    case TILE_BF16: return by_size<TILE_BF16>(rows, width, g, stream);
    case TILE_SWIGLU: return by_size<TILE_SWIGLU>(rows, width, g, stream);
    case TILE_GELU: return by_size<TILE_GELU>(rows, width, g, stream);
    case TILE_RELU2: return by_size<TILE_RELU2>(rows, width, g, stream);
    case TILE_PARTS: return by_size<TILE_PARTS>(rows, width, g, stream);
  }
}

// The same of as many of the M rows as the device finds at ``count``, in tiles that it
// chooses: with a bias, and GELU of that, or (TILE_PARTS) float32 [parts, M, N].
void fei_tile_counted(void* out, long os, const void* x, long xs, const void* w,
                      const void* bias, int M, int N, int K, int epi, int parts,
                      const int* count, hipStream_t stream) {
  const TileArgs g = {out, (const u16*)x, (const u16*)w, (const u16*)bias, count,
                      os, xs, M, N, K, 0, parts};
  switch (epi) {
    case TILE_BIAS: return launch_counted<TILE_BIAS>(g, stream);
    case TILE_GELU: return launch_counted<TILE_GELU>(g, stream);
    case TILE_PARTS: return launch_counted<TILE_PARTS>(g, stream);
  }
}

}  // extern "C"
