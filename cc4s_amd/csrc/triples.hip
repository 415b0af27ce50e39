// Energy kernel of the (T) correction.  For one hole pair (i, j) and a chunk
// of k, W[a,b,c,k] holds the six-fold symmetrised connected triples
// amplitude W_abcijk (PerturbativeTriplesReference.cxx:106-116, formed by
// contractions on the MFMA engine); this kernel adds the disconnected part,
// the spin-adapted combination and the denominator (:118-163):
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

#include <type_traits>

namespace cc4s_amd {

namespace {

constexpr int kBlock = 512;
constexpr int kComplexBlocks = 512;

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
// canonical triples only, so they share them evenly.  Measured over the 55
// launches of (T) at No=10, Nv=96: 5.6 -> 2.4 ms.
template <bool CPLX>
__global__ __launch_bounds__(kBlock, 4) void triples_energy_kernel(
    const typename TS<CPLX>::T *__restrict__ W, const typename TS<CPLX>::T *__restrict__ V,
    const typename TS<CPLX>::T *__restrict__ T1, const double *__restrict__ eh,
    const double *__restrict__ ep, int64_t No, int64_t Nv, int64_t i, int64_t j,
    int64_t k0, int64_t kc, double *acc) {
  using S = TS<CPLX>;
  using T = typename S::T;
  // S at the six orderings of the canonical tile triple's index ranges
  __shared__ T tile[6][kTileElems];
  __shared__ double sh[kBlock / 64];
  static_assert(kBlock == kTileElems, "one thread per tile position");
  const int64_t v = Nv, o = No;
  const int64_t nt = (v + kTile - 1) / kTile;
  const int64_t nc = nt * (nt + 1) * (nt + 2) / 6;  // canonical tile triples
  const int64_t ntiles = nc * kc;
  // V_pphh[p,q,s,r] at p + v (q + v (s + o r)); T1[a,i] at a + v i
  const T *Vjk = V + v * v * j, *Vij = V + v * v * (i + o * j);
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
    const int64_t base = v * v * v * kl;
    const int64_t k = k0 + kl;
    const T *Vik = V + v * v * (i + o * k), *Vjkk = Vjk + v * v * o * k;
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

void triples_energy(hipStream_t s, Field f, const void *W, const void *Vpphh,
                    const void *T1, const double *eps_h, const double *eps_p,
                    int64_t No, int64_t Nv, int64_t i, int64_t j, int64_t k0,
                    int64_t kc, double *acc) {
  CC4S_ASSERT(i >= 0 && i <= j && j < No && k0 >= j && kc > 0 && k0 + kc <= No,
              "triples: hole indices out of range (needs i <= j <= k)");
  if (f == Field::Complex)
    triples_energy_kernel<true><<<kComplexBlocks, kBlock, 0, s>>>(
        static_cast<const double2 *>(W), static_cast<const double2 *>(Vpphh),
        static_cast<const double2 *>(T1), eps_h, eps_p, No, Nv, i, j, k0, kc, acc);
  else
    triples_energy_kernel<false><<<kTriplesBlocks, kBlock, 0, s>>>(
        static_cast<const double *>(W), static_cast<const double *>(Vpphh),
        static_cast<const double *>(T1), eps_h, eps_p, No, Nv, i, j, k0, kc, acc);
  CC4S_HIP(hipGetLastError());
}

}  // namespace cc4s_amd
