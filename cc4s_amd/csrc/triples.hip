// The (T) correction.  The connected triples amplitude of a hole triple
// i <= j <= k, the six-fold symmetrised W_abcijk
// (PerturbativeTriplesReference.cxx:106-116), comes as three parts that the
// first kernel forms:
//   W_abc = Y_i[a;b,c] + Y_j[b;a,c] + Y_k[c;a,b],
//   Y_i[a;b,c] = sum_d V_bcdk T_adij + V_cbdj T_adik
//              - sum_l T_bcjl conj(V_kila) + T_cbkl conj(V_jila)
// (Y_j and Y_k with the holes and particles exchanged likewise).  The energy
// kernel adds them up, and the disconnected part, the spin-adapted combination
// and the denominator (:118-163):
//   S_x   = W_x + T1_{x1 i} V_{x2 x3 j k} + T1_{x2 j} V_{x1 x3 i k} + T1_{x3 k} V_{x1 x2 i j}
//   Z     = 4/3 S_abc - 2 S_acb + 2/3 S_bca
//   E    += Re(W_abc Z) / (e_i + e_j + e_k - e_a - e_b - e_c).
// W and S are unchanged by a simultaneous permutation of the (a,i), (b,j),
// (c,k) pairs, so the six orderings of a hole triple contribute together
//   Re(W_abc Zs) / D,  Zs = 8 S_abc - 4 (S_bac + S_cba + S_acb) + 2 (S_bca + S_cab)
// (the sum of Z over the six orderings, written at the ordering i <= j <= k);
// i <= j <= k runs once, weighted 1 for distinct holes, 1/2 for two equal,
// 1/6 for three equal.  Bandwidth-bound: each element of S is formed once,
// in LDS, and read there at its six orderings.  Each block keeps its running
// sum across launches in `acc[block]` (one stream: a fixed order), so the
// energy is reproducible.  Blocks of 512 threads, as many as are resident at
// once (the grid is one wave of blocks: a second, partial wave would leave
// most CUs idle while it runs).
#include "triples.hpp"

#include <algorithm>
#include <type_traits>

namespace cc4s_amd {

namespace {

constexpr int kBlock = 512;
constexpr int kComplexBlocks = 512;

using dbl4 = double __attribute__((ext_vector_type(4)));

// hole triple number n: tetrahedral(k) + triangular(j) + i, i <= j <= k
__device__ __forceinline__ void hole_triple(int64_t n, int64_t (&h)[3]) {
  h[2] = h[1] = 0;
  while ((h[2] + 1) * (h[2] + 2) * (h[2] + 3) / 6 <= n) ++h[2];
  n -= h[2] * (h[2] + 1) * (h[2] + 2) / 6;
  while ((h[1] + 1) * (h[1] + 2) / 2 <= n) ++h[1];
  h[0] = n - h[1] * (h[1] + 1) / 2;
}

template <bool CPLX>
struct TS;
template <>
struct TS<false> {
  using T = double;
  __device__ static T mul(T a, T b) { return a * b; }
  __device__ static double re_mul(T a, T b) { return a * b; }
  __device__ static T add_scaled(T a, double y, T b) { return a + y * b; }
  __device__ static T plus(T a, T b) { return a + b; }
};
template <>
struct TS<true> {
  using T = double2;
  __device__ static T mul(T a, T b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
  }
  __device__ static double re_mul(T a, T b) { return a.x * b.x - a.y * b.y; }
  __device__ static T add_scaled(T a, double y, T b) {
    return make_double2(a.x + y * b.x, a.y + y * b.y);
  }
  __device__ static T plus(T a, T b) { return make_double2(a.x + b.x, a.y + b.y); }
};

// Y_y1[x1; x2, x3] of the hole triples t0 ... and of their parts part0 ..., one
// after the other.  As a product it has M = (x2, x3), N = x1 and K in four
// segments, d twice and l twice; every address is affine in m, n and k, so there
// are no tables, and with H in T's order only bases, a stride and K differ between
// the segments.  Bound by the matrix pipe where 2 Nv is long against the
// prologue and the epilogue, and next by the traffic of Y: each of the three parts
// is written once and read once by the energy kernel (as six contractions into one
// W it was written six times and read five times between), in one launch for all
// hole triples (330 launches, most too small for the chip).  M is walked in blocks
// of 8 x 8 (x2, x3): V_x2x3 and V_x3x2 are then both read in whole 128-byte lines.
// 128 rows by BN = 96 or 64 columns, whichever leaves fewer columns of padding
// (Nv = 96 on tiles of 64 would multiply 1.33 times as much); eight waves of 32 x
// BN / 2, in stages of 16 k that are loaded two stages ahead, in parts between the
// MFMAs.  Measured with the energy at complex No=10, Nv=96: 28.2 -> 18.3 ms.
struct ProductArgs {
  const void *V, *T, *H;  // V[x2,x3,d,k], T[a,b,i,j], H[a,l,j,i] = -conj(V_ijla)
  void *Y;
  int64_t No, Nv, t0;  // first hole triple
  int tiles;           // of all the parts and triples
  int parts, part0;    // parts per triple, the first of them
  bool add;            // one part: Y += in W's order [a, b, c]
};

typedef double dbl2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void store_stream(double *p, double x) {
  __builtin_nontemporal_store(x, p);
}
__device__ __forceinline__ void store_stream(double2 *p, double2 x) {
  __builtin_nontemporal_store(dbl2{x.x, x.y}, reinterpret_cast<dbl2 *>(p));
}

template <bool CPLX, int BN>
__global__ __launch_bounds__(512, CPLX ? 2 : 4) void triples_product_kernel(ProductArgs p) {
  using T = typename TS<CPLX>::T;
  constexpr int NT = 512, BM = 128, BK = 16, MB = 2, NB = BN / 32;
  constexpr int EA = BM * BK / NT, EB = BN * BK / NT, PARTS = BK / 4 - 1;
  constexpr int PAD = CPLX ? 1 : 18;  // as in the contraction engine
  static_assert(BN % 32 == 0 && BN * BK % NT == 0, "whole subtiles and elements");
  __shared__ T As[2][BK][BM + PAD];
  __shared__ T Bs[2][BK][BN + PAD];
  const int t = threadIdx.x;
  const int64_t v = p.Nv, o = p.No;
  const int64_t v2 = v * v;
  // a run of consecutive tiles per workgroup; consecutive workgroups are dealt to
  // the 8 XCDs in turn, so that an XCD's runs follow each other and share V or T
  // in its L2
  const int grid = gridDim.x, place = (blockIdx.x & 7) * (grid >> 3) + (blockIdx.x >> 3);
  const int first = static_cast<int>(static_cast<int64_t>(p.tiles) * place / grid);
  const int last = static_cast<int>(static_cast<int64_t>(p.tiles) * (place + 1) / grid);
  if (first == last) return;
  const int nb = static_cast<int>((v + 7) / 8);  // blocks of 8 along x2 and x3
  const int tilesM = (nb * nb + 1) / 2, tilesN = static_cast<int>((v + BN - 1) / BN);
  struct Tile {
    int batch, part, n0;
    int x2, x3, d2, d3;  // of its first block of (x2, x3), and to its second
    int two;             // whether there is a second (else the first again)
    int64_t y1, y2, y3;
  };
  auto locate = [&](int g) {
    Tile c;
    c.batch = g / (tilesM * tilesN);
    g -= c.batch * (tilesM * tilesN);
    const int tm = g / tilesN, triple = c.batch / p.parts;
    c.n0 = (g - tm * tilesN) * BN;
    c.part = p.part0 + c.batch - triple * p.parts;
    c.two = 2 * tm + 1 < nb * nb;
    const int q = c.two ? 2 * tm + 1 : 2 * tm, r2 = 2 * tm / nb, r3 = q / nb;
    c.x3 = r2 * 8;
    c.x2 = (2 * tm - r2 * nb) * 8;
    c.d3 = r3 * 8 - c.x3;
    c.d2 = (q - r3 * nb) * 8 - c.x2;
    int64_t h[3];
    hole_triple(p.t0 + triple, h);
    c.y1 = c.part == 0 ? h[0] : c.part == 1 ? h[1] : h[2];
    c.y2 = c.part == 0 ? h[1] : h[0];
    c.y3 = c.part == 2 ? h[1] : h[2];
    return c;
  };
  // what this thread loads of the tile in the load pipeline, in bytes: the row of
  // (x2, x3), what (x3, x2) adds to it, the columns; past the edge the last are read
  constexpr int ES = sizeof(T);
  uint32_t row23, drow, nB[EB];
  int64_t y1, y2, y3;
  auto load_from = [&](const Tile &c) {
    const bool k = t & 64;
    const int x2 = min(c.x2 + (k ? c.d2 : 0) + (t & 7), static_cast<int>(v) - 1),
              x3 = min(c.x3 + (k ? c.d3 : 0) + ((t >> 3) & 7), static_cast<int>(v) - 1);
    row23 = static_cast<uint32_t>(x2 + v * x3) * ES;
    drow = static_cast<uint32_t>(x3 + v * x2) * ES - row23;
    y1 = c.y1;
    y2 = c.y2;
    y3 = c.y3;
#pragma unroll
    for (int i = 0; i < EB; ++i)
      nB[i] = static_cast<uint32_t>(min(c.n0 + (t + NT * i) % BN, static_cast<int>(v) - 1)) * ES;
  };
  const int kA = __builtin_amdgcn_readfirstlane(t / BM);  // k of element i: kA + 4 i
  int kB[EB];
#pragma unroll
  for (int i = 0; i < EB; ++i) kB[i] = (t + NT * i) / BN;
  const int stD = static_cast<int>((v + BK - 1) / BK), stL = static_cast<int>((o + BK - 1) / BK);
  const int nstages = 2 * (stD + stL);
  // segment 0 to 3 of stage s and its first k: V T, V~ T, T H, T~ H (~: x2, x3
  // exchanged).  Sums of conditions and masks, here and below: choices would
  // become branches, at whose ends the compiler waits for every LDS operation
  auto segment = [&](int s, int &d1, int &d2, int &d3) {
    d1 = s >= stD;
    d2 = s >= 2 * stD;
    d3 = s >= 2 * stD + stL;
    return (s - stD * (d1 + d2) - stL * d3) * BK;
  };
  // the stage being loaded
  const char *A, *B;  // of its first k
  int64_t sA;         // A's bytes per k; B's are v elements
  int left;           // k to the end of the segment
  uint32_t rowA;
  const char *A0 = static_cast<const char *>(p.V), *B0 = static_cast<const char *>(p.T);
  const int64_t toHoleA = static_cast<const char *>(p.T) - A0,
                toHoleB = static_cast<const char *>(p.H) - B0;
  auto begin_load = [&](int s) {
    int d1, d2, d3;
    const int64_t kb = segment(s, d1, d2, d3);
    const int64_t hole = -static_cast<int64_t>(d2), other = -static_cast<int64_t>(d1 ^ d3);
    const int64_t dy = (y2 - y3) & other, K = v + ((o - v) & hole);
    sA = ES * (v2 + ((v2 * o - v2) & hole));
    A = A0 + (toHoleA & hole) + ES * v2 * (y3 + dy) * (v + ((1 - v) & hole)) + kb * sA;
    B = B0 + (toHoleB & hole) + ES * v * (K * (y1 + o * (y2 - dy)) + kb);
    left = static_cast<int>(K - kb);
    rowA = row23 + (drow & -static_cast<uint32_t>((d1 + d2 + d3) & 1));
  };
  T ra[EA], rb[EB];
  auto lo = [](int q) { return q * (EA + EB) / PARTS; };
  // a part of it to registers; past a segment's K valid elements are read
  auto load_part = [&](auto part_c) {
    constexpr int part_ = decltype(part_c)::value;
#pragma unroll
    for (int i = 0; i < EA; ++i)
      if (i >= lo(part_) && i < lo(part_ + 1))
        ra[i] = *reinterpret_cast<const T *>(A + min(kA + 4 * i, left - 1) * sA + rowA);
#pragma unroll
    for (int i = 0; i < EB; ++i)
      if (EA + i >= lo(part_) && EA + i < lo(part_ + 1))
        rb[i] = *reinterpret_cast<const T *>(
            B + (nB[i] + static_cast<uint32_t>(min(kB[i], left - 1)) *
                             static_cast<uint32_t>(v * ES)));
  };
  // a part of stage s to LDS, zero past K
  auto store_part = [&](int s, int buf, auto part_c) {
    constexpr int part_ = decltype(part_c)::value;
    int d1, d2, d3;
    const int kb = segment(s, d1, d2, d3);
    const int within = static_cast<int>(v + ((o - v) & -static_cast<int64_t>(d2))) - kb;
#pragma unroll
    for (int i = 0; i < EA; ++i)
      if (i >= lo(part_) && i < lo(part_ + 1))
        As[buf][kA + 4 * i][t % BM] = kA + 4 * i < within ? ra[i] : T{};
#pragma unroll
    for (int i = 0; i < EB; ++i)
      if (EA + i >= lo(part_) && EA + i < lo(part_ + 1))
        Bs[buf][kB[i]][(t + NT * i) % BN] = kB[i] < within ? rb[i] : T{};
  };

  const int lane = t & 63, w = t >> 6, wm = w >> 1, wn = w & 1;
  // three products per complex one: re re, im im, (re + im)(re + im)
  dbl4 acc[CPLX ? 3 : 1][MB][NB];
  T fa[2][MB], fb[2][NB];
  auto load_frag = [&](int buf, int kq, auto q_c) {
    constexpr int q = decltype(q_c)::value;
    const int kr = kq * 4 + (lane >> 4);
#pragma unroll
    for (int i = 0; i < MB; ++i) fa[q][i] = As[buf][kr][wm * 32 + i * 16 + (lane & 15)];
#pragma unroll
    for (int j = 0; j < NB; ++j) fb[q][j] = Bs[buf][kr][wn * (BN / 2) + j * 16 + (lane & 15)];
  };
  auto multiply = [&](auto q_c) {
    constexpr int q = decltype(q_c)::value;
    auto mma = [&](dbl4(&c)[MB][NB], auto of) {
      double x[MB], y[NB];
#pragma unroll
      for (int i = 0; i < MB; ++i) x[i] = of(fa[q][i]);
#pragma unroll
      for (int j = 0; j < NB; ++j) y[j] = of(fb[q][j]);
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          c[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i], y[j], c[i][j], 0, 0, 0);
    };
    if constexpr (CPLX) {
      mma(acc[0], [](T z) { return z.x; });
      mma(acc[1], [](T z) { return z.y; });
      mma(acc[2], [](T z) { return z.x + z.y; });
    } else {
      mma(acc[0], [](T z) { return z; });
    }
  };

  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  static_assert(PARTS == 3, "three parts, four k steps");
  Tile cur = locate(first);
  load_from(cur);
  begin_load(0);
  load_part(I0{}), load_part(I1{}), load_part(I2{});
  store_part(0, 0, I0{}), store_part(0, 0, I1{}), store_part(0, 0, I2{});
  begin_load(1);
  load_part(I0{}), load_part(I1{}), load_part(I2{});
  __syncthreads();
  load_frag(0, 0, I0{});
  // multiply LDS buffer s & 1, move stage s + 1 from the registers to the other
  // one and load stage s + 2, a part after each k step but the last; the barrier
  // stands before the last k step, whose fragments are in registers, so that the
  // next stage's first are read under its MFMAs.  The stages of a run's tiles follow
  // each other without a gap: a tile's first two are loaded under the last two of
  // the tile before (one workgroup fits a CU, so nothing else would cover a tile's
  // first loads: complex No=10, Nv=96 19.4 -> 18.3 ms, 0.2 of it by the streaming
  // stores)
  auto wrap = [&](int s) { return s - (nstages & -static_cast<int>(s >= nstages)); };
  auto step = [&](int s, auto par_c, auto kq_c) {
    constexpr int par = decltype(par_c)::value, kq = decltype(kq_c)::value;
    constexpr std::integral_constant<int, kq & 1> q;
    constexpr std::integral_constant<int, (kq + 1) & 1> next;
    if constexpr (kq < PARTS) {
      load_frag(par, kq + 1, next);
    } else {
      __syncthreads();
      load_frag(par ^ 1, 0, next);
    }
    __builtin_amdgcn_sched_barrier(0);
    multiply(q);
    if constexpr (kq < PARTS) {
      store_part(wrap(s + 1), par ^ 1, kq_c);
      if constexpr (kq == 0) begin_load(wrap(s + 2));
      load_part(kq_c);
    }
  };
  auto stage = [&](int s, auto par) {
    step(s, par, I0{}), step(s, par, I1{}), step(s, par, I2{}), step(s, par, I3{});
  };
  for (int g = first; g < last; ++g) {
#pragma unroll
    for (int c = 0; c < (CPLX ? 3 : 1); ++c)
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[c][i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
    Tile next = cur;
    for (int s = 0; s < nstages; s += 2) {  // an even number
      if (s + 2 == nstages) {               // past the last tile its own are loaded
        next = locate(min(g + 1, last - 1));
        load_from(next);
      }
      stage(s, I0{});
      stage(s + 1, I1{});
    }

    // element (x1, x2, x3) of a part of its own, or of W[a, b, c]
    int64_t s1 = 1, s2 = v, s3 = v2;
    T *Y = static_cast<T *>(p.Y) + cur.batch * v2 * v;
    if (p.parts == 1) {
      s1 = cur.part == 0 ? 1 : cur.part == 1 ? v : v2;
      s2 = cur.part == 0 ? v : 1;
      s3 = cur.part == 2 ? v : v2;
    }
    const bool second = wm >= 2;  // the wave's rows lie in one block of 64
    const int b2 = cur.x2 + (second ? cur.d2 : 0), b3 = cur.x3 + (second ? cur.d3 : 0);
    if (!second || cur.two) {
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = wm * 32 + i * 16 + 4 * r + (lane >> 4);
          const int x2 = b2 + (m & 7), x3 = b3 + ((m >> 3) & 7);
          if (x2 >= v || x3 >= v) continue;
          T *out = Y + s2 * x2 + s3 * x3;
#pragma unroll
          for (int j = 0; j < NB; ++j) {
            const int64_t x1 = cur.n0 + wn * (BN / 2) + j * 16 + (lane & 15);
            if (x1 >= v) continue;
            T x;
            if constexpr (CPLX)
              x = make_double2(acc[0][i][j][r] - acc[1][i][j][r],
                               acc[2][i][j][r] - (acc[0][i][j][r] + acc[1][i][j][r]));
            else
              x = acc[0][i][j][r];
            if (p.add) x = TS<CPLX>::plus(out[s1 * x1], x);
            store_stream(out + s1 * x1, x);
          }
        }
    }
    cur = next;
  }
}

// The particle triples are taken in tiles of kTile^3 (a, b, c).  A block
// takes a canonical tile triple tA <= tB <= tC and forms S at the six
// orderings of its three index ranges in LDS, reading W, V and T1 with x1
// fastest (coalesced rows); every distinct permutation of the tile triple is
// then evaluated from those six LDS tiles, so each element of S is formed
// once and every permuted read of it comes from LDS.
constexpr int kTile = 8;
constexpr int kTileElems = kTile * kTile * kTile;

// ordering p = abc, bac, cba, acb, bca, cab: position d of (x1, x2, x3) holds
// particle kOrder[p][d] of (a, b, c); kCoef[p] is its weight in Zs
constexpr int kOrder[6][3] = {{0, 1, 2}, {1, 0, 2}, {2, 1, 0}, {0, 2, 1}, {1, 2, 0}, {2, 0, 1}};
constexpr double kCoef[6] = {8.0, -4.0, -4.0, -4.0, 2.0, 2.0};
// kCompose[s][p] = q with kOrder[q][d] = kOrder[s][kOrder[p][d]]: in the
// output tile whose (a, b, c) ranges are the canonical ranges kOrder[s],
// ordering p reads the LDS tile formed for ordering q
constexpr int kCompose[6][6] = {{0, 1, 2, 3, 4, 5}, {1, 0, 5, 4, 3, 2}, {2, 4, 0, 5, 1, 3},
                                {3, 5, 4, 0, 2, 1}, {4, 2, 3, 1, 5, 0}, {5, 3, 1, 2, 0, 4}};

// f(std::integral_constant<int, 0>{}), ..., <5>: the six orderings with their
// tables as constants
template <typename F>
__device__ __forceinline__ void six(F &&f) {
  f(std::integral_constant<int, 0>{});
  f(std::integral_constant<int, 1>{});
  f(std::integral_constant<int, 2>{});
  f(std::integral_constant<int, 3>{});
  f(std::integral_constant<int, 4>{});
  f(std::integral_constant<int, 5>{});
}

// A thread owns one position t of the tile at all six orderings: it reads W
// there once, keeps it in registers for the energy of the same element, and its
// reads of W, V and T1 are in flight together (two blocks per CU with 128
// registers; three with 80 spill and take 4.1 ms below).  Blocks walk the
// canonical triples only, so they share them evenly.  Measured over (T) at
// No=10, Nv=96: 5.6 -> 2.4 ms, and 3.6 with the sum of three parts, which the
// products used to form.
template <bool CPLX>
__global__ __launch_bounds__(kBlock, 4) void triples_energy_kernel(
    const typename TS<CPLX>::T *__restrict__ W, const typename TS<CPLX>::T *__restrict__ V,
    const typename TS<CPLX>::T *__restrict__ T1, const double *__restrict__ eh,
    const double *__restrict__ ep, int64_t No, int64_t Nv, int64_t t0, int64_t count,
    int parts, double *acc) {
  using S = TS<CPLX>;
  using T = typename S::T;
  // S at the six orderings of the canonical tile triple's index ranges
  __shared__ T tile[6][kTileElems];
  __shared__ double sh[kBlock / 64];
  static_assert(kBlock == kTileElems, "one thread per tile position");
  const int64_t v = Nv, o = No;
  const int64_t nt = (v + kTile - 1) / kTile;
  const int64_t nc = nt * (nt + 1) * (nt + 2) / 6;  // canonical tile triples
  const int64_t ntiles = nc * count;
  // V_pphh[p,q,s,r] at p + v (q + v (s + o r)); T1[a,i] at a + v i
  const int t = threadIdx.x;
  const int l[3] = {t % kTile, (t / kTile) % kTile, t / (kTile * kTile)};
  double sum = 0.0;
  for (int64_t tid = blockIdx.x; tid < ntiles; tid += gridDim.x) {
    const int64_t kl = tid / nc;
    // r = tetrahedral(tC) + triangular(tB) + tA, tA <= tB <= tC
    int64_t r = tid - kl * nc;
    int64_t tC = 0, tB = 0;
    while ((tC + 1) * (tC + 2) * (tC + 3) / 6 <= r) ++tC;
    r -= tC * (tC + 1) * (tC + 2) / 6;
    while ((tB + 1) * (tB + 2) / 2 <= r) ++tB;
    const int64_t tA = r - tB * (tB + 1) / 2;
    const int64_t ti[3] = {tA, tB, tC};
    const int64_t r0[3] = {tA * kTile, tB * kTile, tC * kTile};
    const int64_t v3 = v * v * v, base = v3 * kl * parts;
    int64_t hole[3];
    hole_triple(t0 + kl, hole);
    const int64_t i = hole[0], j = hole[1], k = hole[2];
    const T *Vij = V + v * v * (i + o * j), *Vik = V + v * v * (i + o * k),
            *Vjkk = V + v * v * (j + o * k);
    __syncthreads();  // the previous tile's LDS reads are done
    // S at the ordering (x1, x2, x3) and the holes (i, j, k): W plus the
    // disconnected part; x1 runs fastest, so the V and T1 reads along x1 are
    // coalesced and the others are broadcasts.  Past the edge the last element
    // is read and S left zero
    T w[6];
    six([&](auto pc) {
      constexpr int p = decltype(pc)::value;
      const int64_t y1 = r0[kOrder[p][0]] + l[0], y2 = r0[kOrder[p][1]] + l[1],
                    y3 = r0[kOrder[p][2]] + l[2];
      const bool in = y1 < v && y2 < v && y3 < v;
      const int64_t x1 = min(y1, v - 1), x2 = min(y2, v - 1), x3 = min(y3, v - 1);
      w[p] = W[base + x1 + v * (x2 + v * x3)];
      if (parts == 3)
        w[p] = S::plus(w[p], S::plus(W[base + v3 + x2 + v * (x1 + v * x3)],
                                     W[base + 2 * v3 + x3 + v * (x1 + v * x2)]));
      const T s = S::plus(w[p], S::plus(S::mul(T1[x1 + v * i], Vjkk[x2 + v * x3]),
                                        S::plus(S::mul(T1[x2 + v * j], Vik[x1 + v * x3]),
                                                S::mul(T1[x3 + v * k], Vij[x1 + v * x2]))));
      tile[p][t] = in ? s : T{};
    });
    __syncthreads();
    const double weight = (i == j && j == k) ? 1.0 / 6.0 : (i == j || j == k) ? 0.5 : 1.0;
    const double eo = (eh[i] + eh[j]) + eh[k];
    six([&](auto sc) {
      constexpr int sg = decltype(sc)::value;
      // output tile: (a, b, c) over the canonical ranges kOrder[sg]; a
      // permutation that repeats an earlier tile triple is skipped
      bool repeat = false;
#pragma unroll
      for (int s2 = 0; s2 < sg; ++s2)
        repeat = repeat || (ti[kOrder[s2][0]] == ti[kOrder[sg][0]] &&
                            ti[kOrder[s2][1]] == ti[kOrder[sg][1]] &&
                            ti[kOrder[s2][2]] == ti[kOrder[sg][2]]);
      if (repeat) return;
      const int64_t x[3] = {r0[kOrder[sg][0]] + l[0], r0[kOrder[sg][1]] + l[1],
                            r0[kOrder[sg][2]] + l[2]};
      if (x[0] >= v || x[1] >= v || x[2] >= v) return;
      T zs = T{};
#pragma unroll
      for (int p = 0; p < 6; ++p) {
        const int q0 = kOrder[p][0], q1 = kOrder[p][1], q2 = kOrder[p][2];
        zs = S::add_scaled(zs, kCoef[p],
                           tile[kCompose[sg][p]][l[q0] + kTile * (l[q1] + kTile * l[q2])]);
      }
      const double d = eo - ((ep[x[0]] + ep[x[1]]) + ep[x[2]]);
      sum += weight * S::re_mul(w[sg], zs) / d;
    });
  }
  // wavefront sums, then the wave sums in wave order
  sum = wave_sum(sum);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    double b = sh[0];
    for (int k = 1; k < kBlock / 64; ++k) b += sh[k];
    acc[blockIdx.x] += b;
  }
}

}  // namespace

namespace {
// columns of a tile: whichever leaves fewer columns of padding
int64_t tile_columns(int64_t Nv) {
  return (Nv + 95) / 96 * 96 <= (Nv + 63) / 64 * 64 ? 96 : 64;
}
// tiles of one part of one hole triple
int64_t tiles_of(int64_t Nv) {
  const int64_t nb = (Nv + 7) / 8, BN = tile_columns(Nv);
  return (nb * nb + 1) / 2 * ((Nv + BN - 1) / BN);
}
}  // namespace

int64_t triples_chunk(int64_t Nv, int64_t all, int64_t most, int parts) {
  most = std::max<int64_t>(1, std::min(all, most));
  // between half the most and the most, the number whose last wave of
  // workgroups (one per CU) is fullest
  const int64_t tiles = tiles_of(Nv) * parts;
  auto loss = [&](int64_t n) {
    const int64_t slots = (n * tiles + 255) / 256 * 256;
    return static_cast<double>(slots - n * tiles) / static_cast<double>(slots);
  };
  int64_t best = most;
  if (most < all)
    for (int64_t n = most; n > most / 2 && n > most - 64; --n)
      if (loss(n) < loss(best)) best = n;
  return best;
}

void triples_product(hipStream_t s, Field f, const void *Vppph, const void *T2, const void *H,
                     void *Y, int64_t No, int64_t Nv, int64_t t0, int64_t count, int part) {
  CC4S_ASSERT(No > 0 && Nv > 0 && t0 >= 0 && count > 0 && part < 3 &&
                  t0 + count <= No * (No + 1) * (No + 2) / 6,
              "triples: hole triples out of range");
  const bool wide = tile_columns(Nv) == 96;
  const int64_t parts = part < 0 ? 3 : 1, tiles = tiles_of(Nv) * parts;
  const int64_t per = ((int64_t(1) << 31) - 1) / tiles;  // a launch counts tiles in 32 bits
  CC4S_ASSERT(per > 0 && Nv < 16384, "triples: too many tiles for one launch");
  for (int64_t t = 0; t < count; t += per) {
    const int64_t n = std::min(per, count - t);
    ProductArgs a{Vppph, T2, H,
                  static_cast<char *>(Y) + t * parts * Nv * Nv * Nv * scalar_bytes(f),
                  No, Nv, t0 + t, static_cast<int>(tiles * n), static_cast<int>(parts),
                  std::max(part, 0), part > 0};
    // as many workgroups as are resident at once: one per CU (complex) or two
    auto run = [&](auto kernel, int grid) {
      kernel<<<grid, 512, 0, s>>>(a);
      CC4S_HIP(hipGetLastError());
    };
    if (f == Field::Complex)
      wide ? run(triples_product_kernel<true, 96>, 256) : run(triples_product_kernel<true, 64>, 256);
    else
      wide ? run(triples_product_kernel<false, 96>, 512)
           : run(triples_product_kernel<false, 64>, 512);
  }
}

void triples_energy(hipStream_t s, Field f, const void *W, const void *Vpphh,
                    const void *T1, const double *eps_h, const double *eps_p,
                    int64_t No, int64_t Nv, int64_t t0, int64_t count, int parts, double *acc) {
  CC4S_ASSERT(t0 >= 0 && count > 0 && t0 + count <= No * (No + 1) * (No + 2) / 6,
              "triples: hole triples out of range");
  if (f == Field::Complex)
    triples_energy_kernel<true><<<kComplexBlocks, kBlock, 0, s>>>(
        static_cast<const double2 *>(W), static_cast<const double2 *>(Vpphh),
        static_cast<const double2 *>(T1), eps_h, eps_p, No, Nv, t0, count, parts, acc);
  else
    triples_energy_kernel<false><<<kTriplesBlocks, kBlock, 0, s>>>(
        static_cast<const double *>(W), static_cast<const double *>(Vpphh),
        static_cast<const double *>(T1), eps_h, eps_p, No, Nv, t0, count, parts, acc);
  CC4S_HIP(hipGetLastError());
}

}  // namespace cc4s_amd
