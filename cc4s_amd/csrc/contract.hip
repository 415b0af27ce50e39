// GETT kernels (FP64 MFMA, gfx950) and the contraction planner.
#include "contract.hpp"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <numeric>
#include <sstream>
#include <type_traits>

namespace cc4s_amd {

namespace {

typedef double dbl4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;  // 4 wave64 per workgroup
constexpr int kPad = 16;       // LDS row padding (doubles)

struct KArgs {
  const double *A;
  const double *B;
  double *C;
  double *W;
  const int64_t *rowA, *colA, *rowB, *colB, *rowC, *colC;
  // C = alpha A B + beta D: D is C itself or another tensor of C's indices
  const double *D;
  const int64_t *rowD, *colD;
  double signD;  // -1 conjugates D
  int64_t M, N, K, kChunk;
  double alpha, beta;
  double signA, signB;  // -1 conjugates the operand's imaginary part
  int tilesM, tilesN;
  // tiles [0, fullTiles) run over all of K; the others, the last partial wave of
  // workgroups, are cut into tailSplits parts of tailChunk k each, whose sums go
  // to Wt [part][tile][BM][BN] (fullTiles is the tile count where nothing is cut)
  double *Wt;
  int fullTiles, tailTiles, tailSplits;
  int64_t tailChunk;
};

// C[oc] = alpha x + beta D[od]
__device__ __forceinline__ void store_result(const KArgs &p, double2 x, int64_t oc, int64_t od) {
  double2 out = make_double2(p.alpha * x.x, p.alpha * x.y);
  if (p.beta != 0.0) {
    const double2 old = reinterpret_cast<const double2 *>(p.D)[od];
    out.x += p.beta * old.x;
    out.y += p.beta * (p.signD * old.y);
  }
  reinterpret_cast<double2 *>(p.C)[oc] = out;
}
__device__ __forceinline__ void store_result(const KArgs &p, double x, int64_t oc, int64_t od) {
  double out = p.alpha * x;
  if (p.beta != 0.0) out += p.beta * p.D[od];
  p.C[oc] = out;
}

// index in a contiguous run of `n` items per XCD: workgroups go round the 8 XCDs
__device__ __forceinline__ int xcd_run(int g, int n) {
  const int x = g & 7, q = n >> 3, r = n & 7;
  return x * q + min(x, r) + (g >> 3);
}

// (tm, tn) of tile g: groups of GM tile rows are walked column by column, so that
// concurrently running tiles share A rows and B columns in L2
__device__ __forceinline__ void tile_of(int g, int tilesM, int tilesN, int GM, int &tm,
                                        int &tn) {
  const int per_group = GM * tilesN;
  const int first_m = (g / per_group) * GM;
  const int gsize = min(tilesM - first_m, GM);
  tm = first_m + (g % per_group) % gsize;
  tn = (g % per_group) / gsize;
}

// Complex GETT, first generation: workgroup tile BM x BN, K staged BK at a time
// through LDS; 4 waves in a (BM/WM) x (BN/WN) grid, each owning WM x WN of C as
// 16x16 MFMA blocks.  A is read either along K (AKC: consecutive lanes ->
// consecutive k) or along M; B along K (BKC) or along N.  LDS holds A as [k][m] and
// B as [k][n] (one plane per real/imaginary part), which is exactly the lane order
// of the MFMA operands (lane l reads row l%16 at k = l/16).
template <int BM, int BN, int BK, int WM, int WN, bool AKC, bool BKC>
__global__ __launch_bounds__(kThreads, 2) void gett_kernel(KArgs p) {
  constexpr int NPL = 2;
  constexpr int MB = WM / 16, NB = WN / 16;
  constexpr int WAVES_N = BN / WN;
  static_assert((BM / WM) * (BN / WN) == 4, "four waves per workgroup");
  static_assert(BK % 4 == 0, "BK multiple of the MFMA k");
  constexpr int EA = BM * BK / kThreads;
  constexpr int EB = BN * BK / kThreads;
  static_assert(EA >= 1 && EB >= 1, "tile too small");
  static_assert(AKC ? (kThreads % BK == 0) : (kThreads % BM == 0), "A map");
  static_assert(BKC ? (kThreads % BK == 0) : (kThreads % BN == 0), "B map");
  constexpr int NKA = AKC ? 1 : EA;  // distinct k per thread per stage
  constexpr int NRA = AKC ? EA : 1;  // distinct m per thread
  constexpr int NKB = BKC ? 1 : EB;
  constexpr int NRB = BKC ? EB : 1;

  __shared__ double As[NPL][BK][BM + kPad];
  __shared__ double Bs[NPL][BK][BN + kPad];

  const int t = threadIdx.x;
  // tile index: spread consecutive workgroups (round-robin over the 8 XCDs)
  // back into neighbouring tiles per XCD, then walk groups of 8 M-tiles so
  // that concurrently running tiles share A rows and B columns in L2.
  const int ntiles = p.tilesM * p.tilesN;
  int g = blockIdx.x;
  if ((ntiles & 7) == 0) g = (g & 7) * (ntiles >> 3) + (g >> 3);
  constexpr int GM = 8;
  const int per_group = GM * p.tilesN;
  const int first_m = (g / per_group) * GM;
  const int gsize = min(p.tilesM - first_m, GM);
  const int tm = first_m + (g % per_group) % gsize;
  const int tn = (g % per_group) / gsize;
  const int64_t m0 = static_cast<int64_t>(tm) * BM;
  const int64_t n0 = static_cast<int64_t>(tn) * BN;
  const int64_t kbeg = static_cast<int64_t>(blockIdx.y) * p.kChunk;
  const int64_t kend = min(p.K, kbeg + p.kChunk);
  const int nstages = kend > kbeg ? static_cast<int>((kend - kbeg + BK - 1) / BK) : 0;

  // fixed per-thread rows of A and columns of B
  int64_t aRow[NRA];
  bool aRowOk[NRA];
#pragma unroll
  for (int i = 0; i < NRA; ++i) {
    const int64_t m = m0 + (AKC ? (t / BK + i * (kThreads / BK)) : (t % BM));
    aRowOk[i] = m < p.M;
    aRow[i] = aRowOk[i] ? p.rowA[m] : 0;
  }
  int64_t bCol[NRB];
  bool bColOk[NRB];
#pragma unroll
  for (int i = 0; i < NRB; ++i) {
    const int64_t n = n0 + (BKC ? (t / BK + i * (kThreads / BK)) : (t % BN));
    bColOk[i] = n < p.N;
    bCol[i] = bColOk[i] ? p.colB[n] : 0;
  }
  auto a_k = [&](int i) { return AKC ? (t % BK) : (t / BM + i * (kThreads / BM)); };
  auto b_k = [&](int i) { return BKC ? (t % BK) : (t / BN + i * (kThreads / BN)); };

  // K offsets are prefetched one stage ahead of the data they address
  int64_t aK[NKA], aKn[NKA], bK[NKB], bKn[NKB];
  bool aKok[NKA], aKokn[NKA], bKok[NKB], bKokn[NKB];
  auto load_koff = [&](int s, int64_t *ak, bool *akok, int64_t *bk, bool *bkok) {
    const int64_t kb = kbeg + static_cast<int64_t>(s) * BK;
#pragma unroll
    for (int i = 0; i < NKA; ++i) {
      const int64_t k = kb + a_k(i);
      akok[i] = k < kend;
      ak[i] = akok[i] ? p.colA[k] : 0;
    }
#pragma unroll
    for (int i = 0; i < NKB; ++i) {
      const int64_t k = kb + b_k(i);
      bkok[i] = k < kend;
      bk[i] = bkok[i] ? p.rowB[k] : 0;
    }
  };

  double ra[EA][NPL], rb[EB][NPL];
  auto load_data = [&]() {
#pragma unroll
    for (int i = 0; i < EA; ++i) {
      const int ir = AKC ? i : 0, ik = AKC ? 0 : i;
      const bool ok = aRowOk[ir] && aKok[ik];
      const int64_t off = aRow[ir] + aK[ik];
      double2 v = ok ? *reinterpret_cast<const double2 *>(p.A + 2 * off)
                     : make_double2(0.0, 0.0);
      ra[i][0] = v.x;
      ra[i][1] = v.y * p.signA;
    }
#pragma unroll
    for (int i = 0; i < EB; ++i) {
      const int ir = BKC ? i : 0, ik = BKC ? 0 : i;
      const bool ok = bColOk[ir] && bKok[ik];
      const int64_t off = bCol[ir] + bK[ik];
      double2 v = ok ? *reinterpret_cast<const double2 *>(p.B + 2 * off)
                     : make_double2(0.0, 0.0);
      rb[i][0] = v.x;
      rb[i][1] = v.y * p.signB;
    }
  };
  auto store_lds = [&]() {
#pragma unroll
    for (int i = 0; i < EA; ++i) {
      const int k = a_k(i);
      const int m = AKC ? (t / BK + i * (kThreads / BK)) : (t % BM);
#pragma unroll
      for (int c = 0; c < NPL; ++c) As[c][k][m] = ra[i][c];
    }
#pragma unroll
    for (int i = 0; i < EB; ++i) {
      const int k = b_k(i);
      const int n = BKC ? (t / BK + i * (kThreads / BK)) : (t % BN);
#pragma unroll
      for (int c = 0; c < NPL; ++c) Bs[c][k][n] = rb[i][c];
    }
  };

  const int lane = t & 63;
  const int w = t >> 6;
  const int wm = w / WAVES_N, wn = w % WAVES_N;
  dbl4 accR[MB][NB], accI[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      accR[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
      accI[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
    }

  if (nstages > 0) {
    load_koff(0, aK, aKok, bK, bKok);
    if (nstages > 1) load_koff(1, aKn, aKokn, bKn, bKokn);
    load_data();
    store_lds();
    __syncthreads();
  }
  for (int s = 0; s < nstages; ++s) {
    const bool more = s + 1 < nstages;
    if (more) {
#pragma unroll
      for (int i = 0; i < NKA; ++i) { aK[i] = aKn[i]; aKok[i] = aKokn[i]; }
#pragma unroll
      for (int i = 0; i < NKB; ++i) { bK[i] = bKn[i]; bKok[i] = bKokn[i]; }
      if (s + 2 < nstages) load_koff(s + 2, aKn, aKokn, bKn, bKokn);
      load_data();
    }
#pragma unroll
    for (int kq = 0; kq < BK / 4; ++kq) {
      const int kr = kq * 4 + (lane >> 4);
      double ar[MB], ai[MB], br[NB], bi[NB];
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        ar[i] = As[0][kr][wm * WM + i * 16 + (lane & 15)];
        ai[i] = As[1][kr][wm * WM + i * 16 + (lane & 15)];
      }
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        br[j] = Bs[0][kr][wn * WN + j * 16 + (lane & 15)];
        bi[j] = Bs[1][kr][wn * WN + j * 16 + (lane & 15)];
      }
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[i], br[j], accR[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[i], bi[j], accI[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const double nai = -ai[i];
#pragma unroll
        for (int j = 0; j < NB; ++j)
          accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(nai, bi[j], accR[i][j], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[i], br[j], accI[i][j], 0, 0, 0);
    }
    if (more) {
      __syncthreads();
      store_lds();
      __syncthreads();
    }
  }

  // epilogue: lane l, register r of a 16x16 f64 MFMA block holds row
  // 4*r + l/16, column l%16
  int64_t cCol[NB];
  bool cColOk[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int64_t n = n0 + wn * WN + j * 16 + (lane & 15);
    cColOk[j] = n < p.N;
    cCol[j] = (cColOk[j] && !p.W) ? p.colC[n] : 0;
  }
#pragma unroll
  for (int i = 0; i < MB; ++i) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t m = m0 + wm * WM + i * 16 + 4 * r + (lane >> 4);
      if (m >= p.M) continue;
      const int64_t rc = p.W ? 0 : p.rowC[m];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        if (!cColOk[j]) continue;
        const int64_t n = n0 + wn * WN + j * 16 + (lane & 15);
        const double vr = accR[i][j][r];
        const double vi = accI[i][j][r];
        if (p.W) {
          const int64_t o = (static_cast<int64_t>(blockIdx.y) * p.M + m) * p.N + n;
          reinterpret_cast<double2 *>(p.W)[o] = make_double2(vr, vi);
        } else {
          const int64_t o = rc + cCol[j];
          double2 *c = reinterpret_cast<double2 *>(p.C) + o;
          double2 out = make_double2(p.alpha * vr, p.alpha * vi);
          if (p.beta != 0.0) {
            const double2 old = *c;
            out.x += p.beta * old.x;
            out.y += p.beta * old.y;
          }
          *c = out;
        }
      }
    }
  }
}

// The GETT kernel of both fields: NT/64 waves on a BM x BN tile.  LDS holds two
// K-stages (double buffer), complex elements with (re, im) interleaved, so an
// MFMA operand pair is one 128-bit LDS read and a K-stage needs one barrier.
// Global loads for stage s+2 are issued while stage s is multiplied; their K
// offsets were fetched a stage earlier still.
//
// Bound by the FP64 matrix pipe.  What kept it from that was the vector work
// between the MFMAs, which share their issue: the address of an operand element
// is one add (row pointers and K offsets in registers, no bounds: padded K
// tables, the last row repeated), conjugation is a sign-bit flip and elements
// past K are zeroed in their one stage only, 35 vector instructions per stage
// and wave of 32 x 32 instead of 82; and LDS reads and stores waited for in
// place (fragments one k step ahead, no branch around the stores).  Measured
// before -> after: complex ring (8192^3) 55.2 -> 51.9 ms; real ring (7533^3), which
// ran on a single-buffered kernel with loads under branches, 19.8 -> 15.6 ms.
// With memory instructions spread over a stage and K offsets by lane (below)
// 7533^3 takes 39.5 ms complex (86 TFLOP/s of 8 flops per complex MAC) and 13.1
// real (65).
//
// M3 selects the three-product complex multiply (Gauss/Karatsuba):
//   P1 = ar br, P2 = ai bi, P3 = (ar + ai)(br + bi),
//   re = P1 - P2, im = P3 - P1 - P2,
// three MFMA products per complex MAC instead of four.  Its error bound is
// the four-product one with |ar|+|ai| and |br|+|bi| in place of |a|, |b|.
constexpr int kZThreads = 512;

template <bool CPLX>
using Scalar = std::conditional_t<CPLX, double2, double>;
// elements past the end of an LDS row.  Complex: one shifts consecutive k-rows by
// one 16-byte bank group, so the column-wise stores of K-contiguous operands and
// the row-wise 128-bit operand reads are both conflict-free per 16-lane pass.
// Real: a shift of 18 8-byte banks (of 32) spreads the 16 k-rows of a column-wise
// store over all even banks and leaves two of 32 lanes of a row-wise read in
// conflict.
template <bool CPLX>
constexpr int kRowPad = CPLX ? 1 : 18;

// One workgroup: block `block` of the tiles (and tail parts), part `slice` of K.
// DEEP keeps two stages of global loads in flight (two register sets): the
// loads for stage s+3 are issued while stage s is multiplied.  MINW (below) is
// the launch bound's minimum of waves per SIMD (2 with 256 threads: two
// workgroups share a CU, so one's prologue and epilogue overlap the other's
// multiplies).
template <bool CPLX, int NT, int BM, int BN, int BK, int WM, int WN, bool AKC, bool BKC,
          bool M3, bool DEEP>
__device__ __forceinline__ void gett_tile(
    const KArgs &p, int block, int slice,
    Scalar<CPLX> (&As)[2][BK][BM + kRowPad<CPLX>], Scalar<CPLX> (&Bs)[2][BK][BN + kRowPad<CPLX>]) {
  using T = Scalar<CPLX>;
  static_assert(CPLX || !M3, "complex forms");
  constexpr int MB = WM / 16, NB = WN / 16;
  constexpr int WAVES_N = BN / WN;
  static_assert((BM / WM) * (BN / WN) * 64 == NT, "one wave per WM x WN block");
  static_assert(BK % 8 == 0, "an even number of MFMA k steps per stage");
  constexpr int EA = BM * BK / NT;
  constexpr int EB = BN * BK / NT;
  static_assert(EA >= 1 && EB >= 1, "tile too small");
  static_assert(AKC ? (NT % BK == 0) : (NT % BM == 0), "A map");
  static_assert(BKC ? (NT % BK == 0) : (NT % BN == 0), "B map");
  constexpr int NKA = AKC ? 1 : EA;
  constexpr int NRA = AKC ? EA : 1;
  constexpr int NKB = BKC ? 1 : EB;
  constexpr int NRB = BKC ? EB : 1;
  const int t = threadIdx.x;
  int g = block;
  int64_t kbeg = static_cast<int64_t>(slice) * p.kChunk, klen = p.kChunk;
  const bool tail = g >= p.fullTiles;
  int part = 0;  // (cut, tile) of a tail workgroup
  if (tail) {
    part = g - p.fullTiles;
    const int cut = part / p.tailTiles, r = xcd_run(part - cut * p.tailTiles, p.tailTiles);
    part = cut * p.tailTiles + r;
    g = p.fullTiles + r;
    kbeg = cut * p.tailChunk;
    klen = p.tailChunk;
  } else {
    g = xcd_run(g, p.fullTiles);
  }
  constexpr int GM = 1024 / BM;  // M-tiles of a group: 1024 rows
  int tm, tn;
  tile_of(g, p.tilesM, p.tilesN, GM, tm, tn);
  const int64_t m0 = static_cast<int64_t>(tm) * BM;
  const int64_t n0 = static_cast<int64_t>(tn) * BN;
  const int64_t kend = min(p.K, kbeg + klen);
  const int nstages = kend > kbeg ? static_cast<int>((kend - kbeg + BK - 1) / BK) : 0;

  auto a_m = [&](int i) { return AKC ? (t / BK + i * (NT / BK)) : (t % BM); };
  auto a_k = [&](int i) { return AKC ? (t % BK) : (t / BM + i * (NT / BM)); };
  auto b_n = [&](int i) { return BKC ? (t / BK + i * (NT / BK)) : (t % BN); };
  auto b_k = [&](int i) { return BKC ? (t % BK) : (t / BN + i * (NT / BN)); };

  // byte addresses of this thread's rows of A and columns of B; one past the
  // edge reads the last row (its products are never stored)
  const char *aRow[NRA];
#pragma unroll
  for (int i = 0; i < NRA; ++i) {
    const int64_t m = min(m0 + a_m(i), p.M - 1);
    aRow[i] = reinterpret_cast<const char *>(p.A) + p.rowA[m] * static_cast<int64_t>(sizeof(T));
  }
  const char *bCol[NRB];
#pragma unroll
  for (int i = 0; i < NRB; ++i) {
    const int64_t n = min(n0 + b_n(i), p.N - 1);
    bCol[i] = reinterpret_cast<const char *>(p.B) + p.colB[n] * static_cast<int64_t>(sizeof(T));
  }

  // K offsets of the next stage to load: its loads take them from the
  // registers as they are issued, and the following stage's offsets are then
  // loaded into the same registers, a whole stage before their use.  Where the
  // waves run along M (N), an element's k is the same over a wave: lane i holds
  // the offset of the wave's element i (A's, then B's), one load and two registers
  // instead of one and two per element, and the loads take it through scalar
  // registers (real 7533^3, both operands so: 14.5 -> 13.1 ms; complex 40.1 ->
  // 39.7, 720^3 66 -> 64 us).  The K tables are padded with a valid offset
  // (kTablePad entries past whole stages), so neither these loads nor the operand
  // loads they address need a bound; what lies past K is zeroed when it is stored
  // to LDS, in the one stage that holds K's end
  constexpr bool UA = !AKC && BM % 64 == 0, UB = !BKC && BN % 64 == 0;
  constexpr int LA = UA ? EA : 0, LANES = LA + (UB ? EB : 0);
  static_assert(LANES <= 64, "one lane per element");
  int64_t aK[UA ? 1 : NKA], bK[UB ? 1 : NKB], kLane = 0;
  const int kIndex = [&] {  // k of this lane's element
    const int l = min(t & 63, LANES - 1), t0 = t & ~63;
    return UA && l < LA ? t0 / BM + l * (NT / BM) : t0 / BN + (l - LA) * (NT / BN);
  }();
  auto k_lane = [&](int l) {
    const int lo32 = __builtin_amdgcn_readlane(static_cast<int>(kLane), l);
    const int hi32 = __builtin_amdgcn_readlane(static_cast<int>(kLane >> 32), l);
    return static_cast<int64_t>(hi32) << 32 | static_cast<uint32_t>(lo32);
  };
  auto a_off = [&](int i) { return UA ? k_lane(i) : aK[AKC ? 0 : UA ? 0 : i]; };
  auto b_off = [&](int i) { return UB ? k_lane(LA + i) : bK[BKC ? 0 : UB ? 0 : i]; };
  auto load_koff = [&](int s) {
    const int64_t kb = kbeg + static_cast<int64_t>(s) * BK;
    const int64_t *ca = p.colA, *rb = p.rowB;
    if constexpr (LANES > 0) kLane = (UA && (!UB || (t & 63) < LA) ? ca : rb)[kb + kIndex];
    if constexpr (!UA) {
#pragma unroll
      for (int i = 0; i < NKA; ++i) aK[i] = ca[kb + a_k(i)];
    }
    if constexpr (!UB) {
#pragma unroll
      for (int i = 0; i < NKB; ++i) bK[i] = rb[kb + b_k(i)];
    }
  };

  // staging registers; DEEP uses two sets, always indexed by constants
  constexpr int NSET = DEEP ? 2 : 1;
  T ra[NSET][EA], rb[NSET][EB];
  // the stage's EA + EB elements in PARTS parts, part q in [lo(q), lo(q + 1))
  constexpr int PARTS = BK / 4 - 1;
  auto lo = [](int q) { return q * (EA + EB) / PARTS; };
  auto load_part = [&](auto set_c, int part) {
    constexpr int q = decltype(set_c)::value;
#pragma unroll
    for (int i = 0; i < EA; ++i)
      if (i >= lo(part) && i < lo(part + 1))
        ra[q][i] = reinterpret_cast<const T *>(aRow[AKC ? i : 0])[a_off(i)];
#pragma unroll
    for (int i = 0; i < EB; ++i)
      if (EA + i >= lo(part) && EA + i < lo(part + 1))
        rb[q][i] = reinterpret_cast<const T *>(bCol[BKC ? i : 0])[b_off(i)];
  };
  auto load_data = [&](auto set_c) {
#pragma unroll
    for (int part = 0; part < PARTS; ++part) load_part(set_c, part);
  };
  // conjugation flips the sign bit of the imaginary part (an integer operation:
  // FP64 multiplies would take the MFMAs' cycles)
  const int flipA = p.signA < 0.0 ? static_cast<int>(0x80000000u) : 0;
  const int flipB = p.signB < 0.0 ? static_cast<int>(0x80000000u) : 0;
  auto flip = [](double x, int mask) {
    return __hiloint2double(__double2hiint(x) ^ mask, __double2loint(x));
  };
  // stage s from its registers to LDS: conjugation applied, elements past K zeroed
  auto store_part = [&](int s, int buf, auto set_c, int part) {
    constexpr int q = decltype(set_c)::value;
    if (part == 0) {
      const int64_t left = p.K - kbeg - static_cast<int64_t>(s) * BK;  // k of this stage within K
      if (left < BK) {
#pragma unroll
        for (int i = 0; i < EA; ++i)
          if (a_k(i) >= left) ra[q][i] = T{};
#pragma unroll
        for (int i = 0; i < EB; ++i)
          if (b_k(i) >= left) rb[q][i] = T{};
      }
    }
#pragma unroll
    for (int i = 0; i < EA; ++i)
      if (i >= lo(part) && i < lo(part + 1)) {
        if constexpr (CPLX)
          As[buf][a_k(i)][a_m(i)] = make_double2(ra[q][i].x, flip(ra[q][i].y, flipA));
        else
          As[buf][a_k(i)][a_m(i)] = ra[q][i];
      }
#pragma unroll
    for (int i = 0; i < EB; ++i)
      if (EA + i >= lo(part) && EA + i < lo(part + 1)) {
        if constexpr (CPLX)
          Bs[buf][b_k(i)][b_n(i)] = make_double2(rb[q][i].x, flip(rb[q][i].y, flipB));
        else
          Bs[buf][b_k(i)][b_n(i)] = rb[q][i];
      }
  };
  auto store_lds = [&](int s, int buf, auto set_c) {
#pragma unroll
    for (int part = 0; part < PARTS; ++part) store_part(s, buf, set_c, part);
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, DEEP ? 1 : 0>;
  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;

  const int lane = t & 63;
  const int w = t >> 6;
  const int wm = w / WAVES_N, wn = w % WAVES_N;
  // real: accR; four-product: accR = re, accI = im; M3: accR = P1, accI = P2,
  // accS = P3
  dbl4 accR[MB][NB], accI[CPLX ? MB : 1][CPLX ? NB : 1], accS[M3 ? MB : 1][M3 ? NB : 1];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      accR[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
      if constexpr (CPLX) accI[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
      if constexpr (M3) accS[i][j] = dbl4{0.0, 0.0, 0.0, 0.0};
    }

  // prologue: stage 0 in LDS buffer 0; stage 1 in registers (DEEP: stage 1
  // in set 1, stage 2 in set 0), the offsets of the stage after it under way
  if (nstages > 0) {
    load_koff(0);
    load_data(S0{});
    load_koff(1);
    if constexpr (DEEP) {
      load_data(S1{});
      load_koff(2);
    }
    store_lds(0, 0, S0{});
    load_data(S0{});
    load_koff(DEEP ? 3 : 2);
    __syncthreads();
  }
  // operand fragments of two k steps: step kq + 1 is read from LDS before the
  // MFMAs of step kq are issued, so a wave does not wait for LDS between them
  constexpr int KQ = BK / 4;
  T fa[2][MB], fb[2][NB];
  auto load_frag = [&](int buf, int kq, int q) {
    const int kr = kq * 4 + (lane >> 4);
#pragma unroll
    for (int i = 0; i < MB; ++i) fa[q][i] = As[buf][kr][wm * WM + i * 16 + (lane & 15)];
#pragma unroll
    for (int j = 0; j < NB; ++j) fb[q][j] = Bs[buf][kr][wn * WN + j * 16 + (lane & 15)];
  };
  auto multiply = [&](int q) {
    const T(&a)[MB] = fa[q];
    const T(&b)[NB] = fb[q];
    if constexpr (!CPLX) {
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], accR[i][j], 0, 0, 0);
    } else if constexpr (M3) {
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].x, b[j].x, accR[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].y, b[j].y, accI[i][j], 0, 0, 0);
      double bs[NB];
#pragma unroll
      for (int j = 0; j < NB; ++j) bs[j] = b[j].x + b[j].y;
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const double as = a[i].x + a[i].y;
#pragma unroll
        for (int j = 0; j < NB; ++j)
          accS[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(as, bs[j], accS[i][j], 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].x, b[j].x, accR[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].x, b[j].y, accI[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const double nai = -a[i].y;
#pragma unroll
        for (int j = 0; j < NB; ++j)
          accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(nai, b[j].y, accR[i][j], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].y, b[j].x, accI[i][j], 0, 0, 0);
    }
  };
  // one K-stage: multiply LDS buffer s&1, move stage s+1 from its
  // registers to the other buffer and load a later stage into them, a part after
  // each k step but the last: the two waves of a SIMD reach their memory
  // instructions together, and the matrix pipe idles while both issue them (all
  // after one k step: complex ring 7533^3 41.1 ms, in parts 39.6; real 15.2 and
  // 13.7).  Nothing here stands under a branch (a stage past the
  // end reads valid elements that are never used): at a branch's end the
  // compiler would wait for every LDS operation in flight.  The stage's one
  // barrier stands before the MFMAs of its last k step, whose fragments are in
  // registers: behind it the other buffer is complete, so the next stage's
  // first fragments are read under those MFMAs, and this stage's buffer is
  // free, every wave having read its last step
  auto stage = [&](int s, auto set_c, auto par_c) {
    constexpr int par = decltype(par_c)::value;  // s & 1
    constexpr int AHEAD = DEEP ? 3 : 2;  // stage loaded into the freed registers
#pragma unroll
    for (int kq = 0; kq < KQ; ++kq) {
      if (kq + 1 < KQ) {
        load_frag(par, kq + 1, (kq + 1) & 1);
      } else {
        __syncthreads();
        load_frag(par ^ 1, 0, 0);
      }
      // the scheduler would sink the reads below the MFMAs to their uses, and
      // raise what waits for the loads above them
      __builtin_amdgcn_sched_barrier(0);
      multiply(kq & 1);
      if (kq < PARTS) {
        store_part(s + 1, par ^ 1, set_c, kq);
        load_part(set_c, kq);  // of stage s+AHEAD
        if (kq == PARTS - 1) load_koff(s + AHEAD + 1);
      }
    }
  };
  if (nstages > 0) load_frag(0, 0, 0);
  // stage s+1 sits in set (s+1)&1 (DEEP) or in the single set
  for (int s = 0; s < nstages; s += 2) {
    stage(s, S1{}, P0{});
    if (s + 1 < nstages) stage(s + 1, S0{}, P1{});
  }

  if (tail) {
    T *w = reinterpret_cast<T *>(p.Wt) + static_cast<int64_t>(part) * (BM * BN);
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          T x;
          if constexpr (!CPLX) {
            x = accR[i][j][r];
          } else if constexpr (M3) {
            const double p1 = accR[i][j][r], p2 = accI[i][j][r];
            x = make_double2(p1 - p2, accS[i][j][r] - (p1 + p2));
          } else {
            x = make_double2(accR[i][j][r], accI[i][j][r]);
          }
          w[(wm * WM + i * 16 + 4 * r + (lane >> 4)) * BN + wn * WN + j * 16 + (lane & 15)] = x;
        }
    return;
  }
  int64_t cCol[NB], dCol[NB];
  bool cColOk[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int64_t n = n0 + wn * WN + j * 16 + (lane & 15);
    cColOk[j] = n < p.N;
    cCol[j] = (cColOk[j] && !p.W) ? p.colC[n] : 0;
    dCol[j] = (cColOk[j] && !p.W) ? p.colD[n] : 0;
  }
#pragma unroll
  for (int i = 0; i < MB; ++i) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t m = m0 + wm * WM + i * 16 + 4 * r + (lane >> 4);
      if (m >= p.M) continue;
      const int64_t rc = p.W ? 0 : p.rowC[m], rd = p.W ? 0 : p.rowD[m];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        if (!cColOk[j]) continue;
        const int64_t n = n0 + wn * WN + j * 16 + (lane & 15);
        T x;
        if constexpr (!CPLX) {
          x = accR[i][j][r];
        } else if constexpr (M3) {
          const double p1 = accR[i][j][r], p2 = accI[i][j][r];
          x = make_double2(p1 - p2, accS[i][j][r] - (p1 + p2));
        } else {
          x = make_double2(accR[i][j][r], accI[i][j][r]);
        }
        if (p.W)
          reinterpret_cast<T *>(p.W)[(static_cast<int64_t>(slice) * p.M + m) * p.N + n] = x;
        else
          store_result(p, x, rc + cCol[j], rd + dCol[j]);
      }
    }
  }
}

template <bool CPLX, int NT, int BM, int BN, int BK, int WM, int WN, bool AKC, bool BKC,
          bool M3, bool DEEP, int MINW = 1>
__global__ __launch_bounds__(NT, MINW) void zgett_kernel(
    KArgs p) {
  __shared__ Scalar<CPLX> As[2][BK][BM + kRowPad<CPLX>];
  __shared__ Scalar<CPLX> Bs[2][BK][BN + kRowPad<CPLX>];
  gett_tile<CPLX, NT, BM, BN, BK, WM, WN, AKC, BKC, M3, DEEP>(p, blockIdx.x, blockIdx.y, As,
                                                                   Bs);
}

// Several independent contractions with small results in one launch: blocks
// first[i] ... of the grid are contraction i's tiles times its K splits.  Alone,
// each is bound by latency (4 to 6 us for a launch, one stage's loads and the
// stores), which the group pays once.  Always the 32x32 tile: four waves, 34 KB of
// LDS, so four blocks of different contractions share a CU.  Measured, one
// iteration, launched one by one -> grouped: complex No=4 Nv=16 455 -> 337 us,
// No=12 Nv=60 1.82 -> 1.62 ms; eleven real ones, No=8 Nv=40, 10.6 -> 8.7 ms.
constexpr int kGroup = 16;
struct GroupArgs {
  KArgs k[kGroup];
  int first[kGroup + 1];
  int orient[kGroup];  // 2 a_kcontig + b_kcontig
  int count;
};
static_assert(sizeof(GroupArgs) <= 4096, "kernel arguments");

__device__ __forceinline__ int group_item(const GroupArgs &g) {
  int i = 0;
  while (i + 1 < g.count && static_cast<int>(blockIdx.x) >= g.first[i + 1]) ++i;
  return i;
}

template <bool CPLX>
__global__ __launch_bounds__(256, 4) void gett_group_kernel(GroupArgs g) {
  __shared__ Scalar<CPLX> As[2][16][32 + kRowPad<CPLX>];
  __shared__ Scalar<CPLX> Bs[2][16][32 + kRowPad<CPLX>];
  const int i = group_item(g);
  const KArgs &p = g.k[i];
  const int b = static_cast<int>(blockIdx.x) - g.first[i], tiles = p.tilesM * p.tilesN;
  const int slice = b / tiles, block = b - slice * tiles;
  switch (g.orient[i]) {
    case 0:
      gett_tile<CPLX, 256, 32, 32, 16, 16, 16, false, false, CPLX, false>(p, block, slice, As, Bs);
      break;
    case 1:
      gett_tile<CPLX, 256, 32, 32, 16, 16, 16, false, true, CPLX, false>(p, block, slice, As, Bs);
      break;
    case 2:
      gett_tile<CPLX, 256, 32, 32, 16, 16, 16, true, false, CPLX, false>(p, block, slice, As, Bs);
      break;
    default:
      gett_tile<CPLX, 256, 32, 32, 16, 16, 16, true, true, CPLX, false>(p, block, slice, As, Bs);
  }
}

// C[rowC[m] + colC[n]] = alpha * sum_s W[s][m][n] + beta * C.  Bound by the
// partials' HBM (or L2) reads, or, for few elements and many splits, by their
// latency: a block takes 256 / G consecutive elements and G interleaved groups
// of splits, four loads in flight per thread; the group sums are added in LDS.
// Both orders are fixed, so the result is reproducible.
template <bool CPLX, int G>
__device__ __forceinline__ void splitk_reduce(const KArgs &p, int splits, uint32_t block,
                                              uint32_t blocks) {
  const uint32_t total = static_cast<uint32_t>(p.M * p.N), N = static_cast<uint32_t>(p.N);
  using T = std::conditional_t<CPLX, double2, double>;
  constexpr uint32_t E = 256 / G;
  __shared__ T part[G][E];
  const uint32_t u = threadIdx.x % E, g = threadIdx.x / E;
  const T *w = reinterpret_cast<const T *>(p.W);
  for (uint32_t e0 = block * E; e0 < total; e0 += blocks * E) {
    const uint32_t e = e0 + u;
    const uint32_t ec = e < total ? e : total - 1;
    T acc[4] = {};
    auto add = [](T &a, const T &b) {
      if constexpr (CPLX) {
        a.x += b.x;
        a.y += b.y;
      } else {
        a += b;
      }
    };
    int s = g;
    for (; s + 3 * G < splits; s += 4 * G)
#pragma unroll
      for (int q = 0; q < 4; ++q) add(acc[q], w[static_cast<int64_t>(s + q * G) * total + ec]);
    for (; s < splits; s += G) add(acc[0], w[static_cast<int64_t>(s) * total + ec]);
    add(acc[0], acc[1]);
    add(acc[2], acc[3]);
    add(acc[0], acc[2]);
    if constexpr (G > 1) {
      part[g][u] = acc[0];
      __syncthreads();
      if (g == 0)
#pragma unroll
        for (int q = 1; q < G; ++q) add(acc[0], part[q][u]);
    }
    if (g == 0 && e < total) {
      const uint32_t m = e / N, n = e - m * N;
      store_result(p, acc[0], p.rowC[m] + p.colC[n], p.rowD[m] + p.colD[n]);
    }
    if constexpr (G > 1) __syncthreads();  // part is written again
  }
}

template <bool CPLX, int G>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(KArgs p, int splits) {
  splitk_reduce<CPLX, G>(p, splits, blockIdx.x, gridDim.x);
}

// the reductions of a group's split contractions, 64 elements per block
template <bool CPLX>
__global__ __launch_bounds__(256) void group_reduce_kernel(GroupArgs g) {
  const int i = group_item(g);
  splitk_reduce<CPLX, 4>(g.k[i], g.orient[i], blockIdx.x - g.first[i], g.first[i + 1] - g.first[i]);
}

// Results of the tail tiles from their parts, in order.  One block takes 256
// elements of one tile; HBM-bound by the parts, which are a few per cent of the
// launch's traffic
template <bool CPLX>
__global__ __launch_bounds__(256) void tail_reduce_kernel(KArgs p, int BM, int BN, int GM) {
  using T = std::conditional_t<CPLX, double2, double>;
  const int per = BM * BN / 256;  // blocks of a tile
  const int r = blockIdx.x / per;
  const int e = (blockIdx.x - r * per) * 256 + threadIdx.x;
  int tm, tn;
  tile_of(p.fullTiles + r, p.tilesM, p.tilesN, GM, tm, tn);
  const int64_t m = static_cast<int64_t>(tm) * BM + e / BN;
  const int64_t n = static_cast<int64_t>(tn) * BN + e % BN;
  if (m >= p.M || n >= p.N) return;
  const int64_t stride = static_cast<int64_t>(p.tailTiles) * BM * BN;
  const T *w = reinterpret_cast<const T *>(p.Wt) + static_cast<int64_t>(r) * BM * BN + e;
  T acc = w[0];
#pragma unroll 4
  for (int s = 1; s < p.tailSplits; ++s) {
    const T x = w[s * stride];
    if constexpr (CPLX) {
      acc.x += x.x;
      acc.y += x.y;
    } else {
      acc += x;
    }
  }
  store_result(p, acc, p.rowC[m] + p.colC[n], p.rowD[m] + p.colD[n]);
}

constexpr int kMaxRank = 8;
struct SumArgs {
  const double *A;
  double *C;
  int rank;
  int64_t lens[kMaxRank];
  int64_t sA[kMaxRank];
  int64_t sC[kMaxRank];
  int64_t total;
  double alpha, beta, signA;
};

// C = alpha * op(A) + beta * C over C's index space (first index fastest)
template <bool CPLX>
__global__ __launch_bounds__(256) void sum_kernel(SumArgs p) {
  for (int64_t e = blockIdx.x * 256ll + threadIdx.x; e < p.total;
       e += static_cast<int64_t>(gridDim.x) * 256) {
    int64_t r = e, oa = 0, oc = 0;
    for (int d = 0; d < p.rank; ++d) {
      const int64_t q = r / p.lens[d];
      const int64_t i = r - q * p.lens[d];
      r = q;
      oa += i * p.sA[d];
      oc += i * p.sC[d];
    }
    if constexpr (CPLX) {
      double2 a = p.A ? reinterpret_cast<const double2 *>(p.A)[oa]
                      : make_double2(0.0, 0.0);
      double2 *c = reinterpret_cast<double2 *>(p.C) + oc;
      double2 out = make_double2(p.alpha * a.x, p.alpha * p.signA * a.y);
      if (p.beta != 0.0) {
        const double2 old = *c;
        out.x += p.beta * old.x;
        out.y += p.beta * old.y;
      }
      *c = out;
    } else {
      double out = p.A ? p.alpha * p.A[oa] : 0.0;
      if (p.beta != 0.0) out += p.beta * p.C[oc];
      p.C[oc] = out;
    }
  }
}

template <int BM, int BN, int BK, int WM, int WN>
void dispatch_gett(const GettLaunch &L, const KArgs &args, dim3 grid, hipStream_t s) {
  if (L.a_kcontig && L.b_kcontig)
    gett_kernel<BM, BN, BK, WM, WN, true, true><<<grid, kThreads, 0, s>>>(args);
  else if (L.a_kcontig)
    gett_kernel<BM, BN, BK, WM, WN, true, false><<<grid, kThreads, 0, s>>>(args);
  else if (L.b_kcontig)
    gett_kernel<BM, BN, BK, WM, WN, false, true><<<grid, kThreads, 0, s>>>(args);
  else
    gett_kernel<BM, BN, BK, WM, WN, false, false><<<grid, kThreads, 0, s>>>(args);
}

template <bool CPLX, int NT, int BM, int BN, int BK, int WM, int WN, bool M3,
          bool DEEP = false, int MINW = 1>
void dispatch_zgett(const GettLaunch &L, const KArgs &args,
                    dim3 grid, hipStream_t s) {
  if (L.a_kcontig && L.b_kcontig)
    zgett_kernel<CPLX, NT, BM, BN, BK, WM, WN, true, true, M3, DEEP, MINW>
        <<<grid, NT, 0, s>>>(args);
  else if (L.a_kcontig)
    zgett_kernel<CPLX, NT, BM, BN, BK, WM, WN, true, false, M3, DEEP, MINW>
        <<<grid, NT, 0, s>>>(args);
  else if (L.b_kcontig)
    zgett_kernel<CPLX, NT, BM, BN, BK, WM, WN, false, true, M3, DEEP, MINW>
        <<<grid, NT, 0, s>>>(args);
  else
    zgett_kernel<CPLX, NT, BM, BN, BK, WM, WN, false, false, M3, DEEP, MINW>
        <<<grid, NT, 0, s>>>(args);
}

// Tiles of the GETT kernel (complex: generation 3).  The waves of a workgroup
// own 32 x 32 (complex) or 64 x 64 (real) of a large tile, 32 x 32 of a medium
// and 16 x 16 of a small one; `cap` workgroups share a CU (LDS and registers),
// so one's barriers, first loads and epilogue pass under another's MFMAs.
// Measured times in microseconds: `stage`, one 16-k stage of one workgroup on a
// CU that is full of them (its MFMAs alone take 64 cycles per 16x16x4 block,
// three per complex block, on four SIMDs); `lone`, the same where it has the CU
// to itself and nothing hides a stage's latencies but nothing delays it either
// (a real 320^3 on 100 small tiles: 8.3 us whole, 10.2 cut in five along K);
// `cold`, what each of the first eight stages takes longer; `ends`, the first
// loads and the epilogue.
enum class Tile : int { Large = 0, Medium = 1, Small = 2 };
struct TileShape {
  int BM, BN, cap;
  double stage, lone, cold, ends;
};
constexpr int kZ3BK = 16;  // K-stage of every tile
constexpr TileShape kComplexTiles[3] = {
    {128, 64, 1, 3.3, 3.3, 0.0, 8.0},
    {64, 64, 2, 1.72, 2.0, 0.0, 6.0},
    {32, 32, 4, 0.55, 0.5, 0.0, 4.0}};
constexpr TileShape kRealTiles[3] = {
    {128, 128, 2, 2.4, 2.4, 2.3, 8.0},
    {64, 64, 3, 0.68, 0.76, 0.0, 5.7},
    {32, 32, 4, 0.3, 0.22, 0.0, 4.0}};
// other complex generations: first 128x64; second 128x128; fourth and fifth 128x64
constexpr int kCBM = 128, kCBN = 64, kCBK = 16, kCWM = 64, kCWN = 32;
constexpr int kZBM = 128, kZBN = 128, kZBK = 16, kZWM = 64, kZWN = 32;

TileShape tile_shape(Field f, Tile t, int generation) {
  if (f == Field::Real) return kRealTiles[static_cast<int>(t)];
  if (generation == 2) return {kZBM, kZBN, 1, 6.6, 6.6, 0.0, 10.0};
  if (generation == 1) return {kCBM, kCBN, 2, 4.0, 4.0, 0.0, 10.0};
  return kComplexTiles[static_cast<int>(t)];
}

inline int grid_for(int64_t n) {
  return static_cast<int>(std::min<int64_t>((n + 255) / 256, 256 * 64));
}

}  // namespace

std::string gett_variant(const GettLaunch &L) {
  std::string n = L.field == Field::Complex ? "gett_c64" : "gett_f64";
  n += L.a_kcontig ? "_ak" : "_am";
  n += L.b_kcontig ? "_bk" : "_bn";
  if (L.tile == 1) n += "_t64";
  if (L.tile == 2) n += "_t32";
  return n;
}

namespace {
void reduce_partials(bool cplx, const KArgs &a, int splits, hipStream_t s);

KArgs kernel_args(const GettLaunch &L) {
  const bool cplx = L.field == Field::Complex;
  const TileShape shape = tile_shape(L.field, static_cast<Tile>(L.tile), L.generation);
  const int BM = shape.BM, BN = shape.BN, BK = kZ3BK;
  KArgs a{};
  a.A = static_cast<const double *>(L.A);
  a.B = static_cast<const double *>(L.B);
  a.C = static_cast<double *>(L.C);
  a.W = L.splits > 1 ? static_cast<double *>(L.W) : nullptr;
  a.rowA = L.rowA; a.colA = L.colA; a.rowB = L.rowB; a.colB = L.colB;
  a.rowC = L.rowC; a.colC = L.colC;
  a.D = L.D ? static_cast<const double *>(L.D) : a.C;
  a.rowD = L.D ? L.rowD : L.rowC;
  a.colD = L.D ? L.colD : L.colC;
  a.signD = L.conjD ? -1.0 : 1.0;
  CC4S_ASSERT(!L.D || !cplx || L.generation != 1,
              "the first-generation kernel adds to its own result only");
  a.M = L.M; a.N = L.N; a.K = L.K;
  const int64_t kstages = (L.K + BK - 1) / BK;
  a.kChunk = ((kstages + L.splits - 1) / L.splits) * BK;
  a.alpha = L.alpha; a.beta = L.beta;
  a.signA = L.conjA ? -1.0 : 1.0;
  a.signB = L.conjB ? -1.0 : 1.0;
  a.tilesM = static_cast<int>((L.M + BM - 1) / BM);
  a.tilesN = static_cast<int>((L.N + BN - 1) / BN);
  CC4S_ASSERT(static_cast<int64_t>(a.tilesM) * a.tilesN < (int64_t(1) << 31),
              "contraction too large for one launch");
  const int ntiles = a.tilesM * a.tilesN;
  a.fullTiles = L.tail_splits > 1 ? static_cast<int>(L.full_tiles) : ntiles;
  a.tailTiles = ntiles - a.fullTiles;
  a.tailSplits = L.tail_splits;
  a.Wt = static_cast<double *>(L.W);
  a.tailChunk = L.tail_splits > 1 ? (kstages + L.tail_splits - 1) / L.tail_splits * BK : 0;
  CC4S_ASSERT(L.tail_splits <= 1 || (L.splits == 1 && L.W && a.fullTiles > 0 && a.tailTiles > 0),
              "tail split without its workspace");
  return a;
}
}  // namespace

void launch_gett(const GettLaunch &L, hipStream_t s, hipEvent_t start,
                 hipEvent_t stop) {
  const bool cplx = L.field == Field::Complex;
  const Tile tile = static_cast<Tile>(L.tile);
  const TileShape shape = tile_shape(L.field, tile, L.generation);
  const int BM = shape.BM, BN = shape.BN;
  const KArgs a = kernel_args(L);
  dim3 grid(a.fullTiles + a.tailTiles * std::max(1, L.tail_splits), L.splits);
  if (start) CC4S_HIP(hipEventRecord(start, s));
  if (cplx && L.generation == 3) {
    if (tile == Tile::Large)
      dispatch_zgett<true, 512, 128, 64, 16, 32, 32, true>(L, a, grid, s);
    else if (tile == Tile::Medium)
      dispatch_zgett<true, 256, 64, 64, 16, 32, 32, true, false, 2>(L, a, grid, s);
    else
      dispatch_zgett<true, 256, 32, 32, 16, 16, 16, true, false, 4>(L, a, grid, s);
  } else if (cplx && L.generation == 2) {
    dispatch_zgett<true, kZThreads, kZBM, kZBN, kZBK, kZWM, kZWN, false>(L, a, grid, s);
  } else if (cplx && L.generation == 4) {
    dispatch_zgett<true, 256, 128, 64, 16, 64, 32, true>(L, a, grid, s);
  } else if (cplx && L.generation == 5) {
    dispatch_zgett<true, 512, 128, 64, 16, 32, 32, true, true>(L, a, grid, s);
  } else if (cplx) {
    dispatch_gett<kCBM, kCBN, kCBK, kCWM, kCWN>(L, a, grid, s);
  } else if (tile == Tile::Large) {
    dispatch_zgett<false, 256, 128, 128, 16, 64, 64, false, false, 2>(L, a, grid, s);
  } else if (tile == Tile::Medium) {
    dispatch_zgett<false, 256, 64, 64, 16, 32, 32, false, false, 3>(L, a, grid, s);
  } else {
    dispatch_zgett<false, 256, 32, 32, 16, 16, 16, false, false, 4>(L, a, grid, s);
  }
  CC4S_HIP(hipGetLastError());
  if (stop) CC4S_HIP(hipEventRecord(stop, s));
  if (L.tail_splits > 1) {
    const int GM = 1024 / BM;
    const unsigned blocks = static_cast<unsigned>(a.tailTiles) * (BM * BN / 256);
    if (cplx)
      tail_reduce_kernel<true><<<blocks, 256, 0, s>>>(a, BM, BN, GM);
    else
      tail_reduce_kernel<false><<<blocks, 256, 0, s>>>(a, BM, BN, GM);
    CC4S_HIP(hipGetLastError());
  }
  if (L.splits > 1) reduce_partials(cplx, a, L.splits, s);
}

namespace {
void reduce_partials(bool cplx, const KArgs &a, int splits, hipStream_t s) {
  CC4S_ASSERT(a.M * a.N < (int64_t(1) << 31), "split-K result too large");
  const int64_t total = a.M * a.N;
  auto run = [&](auto kernel, int G) { kernel<<<grid_for(total * G), 256, 0, s>>>(a, splits); };
  // groups of splits while the elements alone leave the chip idle (under 64 K
  // threads) and every group still has several splits
  if (total < 16384 && splits >= 32)
    cplx ? run(splitk_reduce_kernel<true, 16>, 16) : run(splitk_reduce_kernel<false, 16>, 16);
  else if (total < 65536 && splits >= 8)
    cplx ? run(splitk_reduce_kernel<true, 4>, 4) : run(splitk_reduce_kernel<false, 4>, 4);
  else
    cplx ? run(splitk_reduce_kernel<true, 1>, 1) : run(splitk_reduce_kernel<false, 1>, 1);
  CC4S_HIP(hipGetLastError());
}
}  // namespace

void launch_splitk_reduce(Field f, const double *W, double *C,
                          const int64_t *rowC, const int64_t *colC, int64_t M,
                          int64_t N, int splits, double alpha, double beta,
                          hipStream_t s) {
  KArgs a{};
  a.W = const_cast<double *>(W);
  a.C = C;
  a.D = C;
  a.rowC = a.rowD = rowC;
  a.colC = a.colD = colC;
  a.signD = 1.0;
  a.M = M;
  a.N = N;
  a.alpha = alpha;
  a.beta = beta;
  reduce_partials(f == Field::Complex, a, splits, s);
}

// ---------------------------------------------------------------------------
// planner
// ---------------------------------------------------------------------------

struct GettPlan {
  int generation = 3;  // kernel that tile, splits and tail are for
  int64_t M = 0, N = 0, K = 0;
  bool swap = false, a_kc = true, b_kc = true;
  int splits = 1, tail_splits = 1;
  int64_t full_tiles = 0;
  Tile tile = Tile::Large;
  const int64_t *rowA, *colA, *rowB, *colB, *rowC, *colC;
  const int64_t *rowD = nullptr, *colD = nullptr;  // of an added tensor other than C
};

ContractionEngine::ContractionEngine(hipStream_t s) : stream_(s) { apply_env_overrides(); }

void ContractionEngine::apply_env_overrides() {
  // CC4S_MIXED_SPLIT=half|bf16 and CC4S_MIXED_MAX_K override the split
  // format and the longest FP32 sum of the mixed path
  if (const char *e = std::getenv("CC4S_MIXED_SPLIT")) {
    const std::string v = e;
    CC4S_ASSERT(v == "half" || v == "bf16", "CC4S_MIXED_SPLIT must be half or bf16");
    mixed_half = v == "half";
  }
  // CC4S_GETT_GENERATION selects the complex FP64 kernel of this engine
  if (const char *e = std::getenv("CC4S_GETT_GENERATION")) {
    const int v = std::atoi(e);
    complex_generation = v >= 1 && v <= 5 ? v : 3;
  }
  if (const char *e = std::getenv("CC4S_MIXED_TERMS")) {
    const int v = std::atoi(e);
    CC4S_ASSERT(v == 9 || v == 12 || v == 16, "CC4S_MIXED_TERMS must be 9, 12 or 16");
    mixed_terms = v;
  }
  if (const char *e = std::getenv("CC4S_MIXED_MAX_K")) {
    const long long v = std::atoll(e);
    CC4S_ASSERT(v >= 16, "CC4S_MIXED_MAX_K must be at least 16");
    mixed_max_k = v;
  }
  // CC4S_MIXED_MIN_FLOPS: smaller complex contractions stay FP64
  if (const char *e = std::getenv("CC4S_MIXED_TILE")) set_mixed_tile(std::atoi(e));
  if (const char *e = std::getenv("CC4S_MIXED_MIN_FLOPS")) {
    const double v = std::atof(e);
    CC4S_ASSERT(v >= 0.0, "CC4S_MIXED_MIN_FLOPS must not be negative");
    mixed_min_flops = v;
  }
}

// a timing event from the pool of recorded and read ones, else a new one
hipEvent_t ContractionEngine::take_event() {
  hipEvent_t e;
  if (!event_pool_.empty()) {
    e = event_pool_.back();
    event_pool_.pop_back();
  } else {
    CC4S_HIP(hipEventCreate(&e));
  }
  return e;
}

ContractionEngine::~ContractionEngine() {
  for (auto &p : pending_) {
    (void)hipEventDestroy(p.start);
    (void)hipEventDestroy(p.stop);
  }
  for (auto e : event_pool_) (void)hipEventDestroy(e);
}

void ContractionEngine::set_profiling(bool on) { profiling_ = on; }

void ContractionEngine::reset_timings() {
  (void)timings();
  timings_.clear();
}

const std::unordered_map<std::string, KernelTiming> &ContractionEngine::timings() {
  if (!pending_.empty()) {
    CC4S_HIP(hipStreamSynchronize(stream_));
    for (auto &p : pending_) {
      float ms = 0;
      CC4S_HIP(hipEventElapsedTime(&ms, p.start, p.stop));
      auto &t = timings_[p.name];
      t.launches += 1;
      t.ms += ms;
      t.flops += p.flops;
      event_pool_.push_back(p.start);
      event_pool_.push_back(p.stop);
    }
    pending_.clear();
  }
  return timings_;
}

namespace {

std::string plan_key(const View &A, const View &B, const View &C) {
  std::ostringstream k;
  for (const View *v : {&A, &B, &C}) {
    k << v->idx << (v->conj ? "*" : "") << ':';
    for (size_t d = 0; d < v->lens.size(); ++d)
      k << v->lens[d] << '/' << v->strides[d] << ',';
    k << '|';
  }
  k << static_cast<int>(C.field);
  return k.str();
}

// K offset tables are padded with their first entry, a valid offset, to whole
// K-stages and past them: a kernel reads its table up to four stages ahead
constexpr int64_t kTablePad = 5 * kZ3BK;

// Offset tables of a plan, built where they are read: table t holds the offset of
// every multi-index of its modes (first mode fastest), entries n[t] ... of a padded
// one its first offset, which is 0.  One launch instead of an allocation, a host
// loop over every entry and a blocking copy (25 to 40 us a plan, about 50 plans in
// a residuum's first pass): that pass took 1378 -> 675 us (complex No=4 Nv=16) and
// 6.7 -> 3.2 ms (No=12 Nv=60).
constexpr int kTables = 8, kTableModes = 8;
struct TableArgs {
  int64_t *out;
  int64_t first[kTables + 1];  // table t at out + first[t], padded length by difference
  int64_t n[kTables], block[kTables];  // entries; entries per step of the first mode here
  int64_t len[kTables][kTableModes], stride[kTables][kTableModes];
  int modes[kTables];
  int count;
  bool add;  // modes beyond the first kTableModes are added in further launches
};

__global__ __launch_bounds__(256) void offsets_kernel(TableArgs p) {
  for (int64_t e = blockIdx.x * int64_t(256) + threadIdx.x; e < p.first[p.count];
       e += gridDim.x * int64_t(256)) {
    int t = 0;
    while (e >= p.first[t + 1]) ++t;
    const int64_t i = e - p.first[t];
    int64_t off = 0;
    if (i < p.n[t]) {
      int64_t rest = i / p.block[t];
      for (int m = 0; m < p.modes[t]; ++m) {
        const int64_t q = rest / p.len[t][m];
        off += (rest - q * p.len[t][m]) * p.stride[t][m];
        rest = q;
      }
    }
    p.out[e] = p.add ? p.out[e] + off : off;
  }
}

}  // namespace

// a table of `group`'s multi-indices (first listed fastest) with v's strides
struct OffsetTable {
  const View *v;
  std::string group;
  bool padded;
  const int64_t **out;
  int64_t entries() const {
    int64_t n = 1;
    for (char c : group) n *= v->len(c);
    return n;
  }
  int64_t size() const {
    const int64_t n = entries();
    return padded && n ? (n + kZ3BK - 1) / kZ3BK * kZ3BK + kTablePad : n;
  }
};

namespace {

// Tile and split count with the smallest estimated time (microseconds):
//   - workgroups run in waves of 256 CUs x cap; a wave takes its K-stages at the
//     full CU's rate for the workgroups that share a CU, or at a lone
//     workgroup's latency where that is longer, and its ends, half of them under
//     another workgroup where several share a CU;
//   - split-K adds a reduction launch and its partials' traffic (4 TB/s).
// Measured over the statements of one pass, fixed choice (128 x 64 complex,
// 128 x 128 real, split to four workgroups per slot) -> this one; the fixed
// choice stays the better one only where it is also this one's:
//   complex No=4 Nv=16 221 -> 103 us, No=12 Nv=60 774 -> 605 us, No=20 Nv=150
//   21.7 -> 19.4 ms; real No=8 Nv=40 346 -> 167 us, No=20 Nv=150 10.4 -> 9.1 ms.
//   - where whole waves are followed by a partial one, the partial wave's tiles
//     can be cut along K instead, so that their parts fill the chip: the same
//     reduction costs for them alone.  Ladder products 37179 x 496 x 29646: real
//     21.0 -> 18.1 ms, complex 57.7 -> 52.7 ms; ring 2227^3 complex 1.19 -> 1.15
//     ms; energy and gradient of No=24, Nv=192, NG=1100 (4608 x 1100 x 4608) 9.2
//     -> 8.2 ms.
void choose_tile(Field f, int64_t M, int64_t N, int64_t K, size_t max_workspace, GettPlan &plan) {
  const int generation = plan.generation;
  constexpr double kReduce = 3.5, kBytesPerUs = 4e6;
  plan.tile = Tile::Large;
  plan.splits = plan.tail_splits = 1;
  plan.full_tiles = 0;
  if (M <= 0 || N <= 0 || K <= 0) return;
  const int64_t kstages = (K + kZ3BK - 1) / kZ3BK;
  const double es = static_cast<double>(scalar_bytes(f));
  const bool fixed_tile = f == Field::Complex && generation != 3;
  double best = -1;
  for (int t = 0; t < (fixed_tile ? 1 : 3); ++t) {
    const TileShape s = tile_shape(f, static_cast<Tile>(t), generation);
    const int64_t tiles = ((M + s.BM - 1) / s.BM) * ((N + s.BN - 1) / s.BN);
    if (tiles >= (int64_t(1) << 31)) continue;
    const int64_t per = 256 * s.cap;
    // one wave of c workgroups per CU over n stages
    auto wave = [&](double n, double c) {
      return n * (c > 1 ? std::max(c * s.stage, s.lone) : s.lone) + std::min(n, 8.0) * s.cold +
             (s.cap > 1 && c > 1 ? 0.5 : 1.0) * s.ends;
    };
    // every count to 16, then steps of about 6 %
    for (int64_t sp = 1; sp <= std::min<int64_t>(1024, std::max<int64_t>(1, kstages / 2));
         sp += std::max<int64_t>(1, sp / 16)) {
      if (sp > 1 && (static_cast<double>(sp) * M * N * es > static_cast<double>(max_workspace) ||
                     M * N >= (int64_t(1) << 31) || tiles * sp > 4 * per))
        break;
      const double n = static_cast<double>((kstages + sp - 1) / sp);
      const int64_t W = tiles * sp, full = W / per, rem = W % per;
      double cost = static_cast<double>(full) * wave(n, s.cap);
      if (rem) cost += wave(n, static_cast<double>((rem + 255) / 256));
      if (sp > 1) cost += kReduce + 2.0 * static_cast<double>(sp) * M * N * es / kBytesPerUs;
      if (best < 0 || cost < best) {
        best = cost;
        plan.tile = static_cast<Tile>(t);
        plan.splits = static_cast<int>(sp);
        plan.tail_splits = 1;
      }
    }
    // whole waves, and the rest cut along K
    const int64_t full = tiles / per, rem = tiles % per;
    if (fixed_tile || full == 0 || rem == 0) continue;
    for (int64_t cut = 2; cut <= std::min<int64_t>(32, kstages / 4); ++cut) {
      const double n = static_cast<double>((kstages + cut - 1) / cut);
      const double bytes = static_cast<double>(cut * rem) * s.BM * s.BN * es;
      if (bytes > static_cast<double>(max_workspace)) break;
      const int64_t W = rem * cut, waves = W / per, last = W % per;
      double cost = static_cast<double>(full) * wave(static_cast<double>(kstages), s.cap) +
                    static_cast<double>(waves) * wave(n, s.cap) + kReduce +
                    2.0 * bytes / kBytesPerUs;
      if (last) cost += wave(n, static_cast<double>((last + 255) / 256));
      if (cost < best) {
        best = cost;
        plan.tile = static_cast<Tile>(t);
        plan.splits = 1;
        plan.tail_splits = static_cast<int>(cut);
        plan.full_tiles = full * per;
      }
    }
  }
}

}  // namespace

// the tables' entries go to the arena; `stream_` builds them and reads them
void ContractionEngine::build_tables(const OffsetTable *tables, int count) {
  CC4S_ASSERT(count <= kTables, "too many offset tables");
  TableArgs a{};
  a.count = count;
  size_t rounds = 1;
  for (int t = 0; t < count; ++t) {
    a.first[t + 1] = a.first[t] + tables[t].size();
    a.n[t] = tables[t].entries();
    a.block[t] = 1;
    rounds = std::max(rounds, (tables[t].group.size() + kTableModes - 1) / kTableModes);
  }
  const int64_t total = a.first[count];
  const size_t bytes = (static_cast<size_t>(total) * sizeof(int64_t) + 255) / 256 * 256;
  if (arena_.empty() || arena_used_ + bytes > arena_.back().bytes()) {
    DeviceBuffer chunk;
    chunk.allocate(std::max(bytes, kArenaChunk));
    arena_.push_back(std::move(chunk));
    arena_used_ = 0;
  }
  a.out = reinterpret_cast<int64_t *>(arena_.back().as<char>() + arena_used_);
  arena_used_ += bytes;
  for (int t = 0; t < count; ++t) *tables[t].out = a.out + a.first[t];
  if (total == 0) return;
  for (size_t r = 0; r < rounds; ++r) {
    a.add = r > 0;
    for (int t = 0; t < count; ++t) {
      const std::string &g = tables[t].group;
      a.modes[t] = 0;
      for (size_t m = r * kTableModes; m < std::min(g.size(), (r + 1) * kTableModes); ++m) {
        a.len[t][a.modes[t]] = std::max<int64_t>(1, tables[t].v->len(g[m]));
        a.stride[t][a.modes[t]++] = tables[t].v->stride(g[m]);
      }
    }
    const int64_t blocks = std::min<int64_t>((total + 255) / 256, 4096);
    offsets_kernel<<<static_cast<unsigned>(blocks), 256, 0, stream_>>>(a);
    CC4S_HIP(hipGetLastError());
    for (int t = 0; t < count; ++t)
      for (int m = 0; m < a.modes[t]; ++m) a.block[t] *= a.len[t][m];
  }
}

GettPlan &ContractionEngine::plan_for(const View &A0, const View &B0,
                                      const View &C, const View *D) {
  std::string key = plan_key(A0, B0, C);
  if (D) key += "+" + plan_key(*D, *D, *D);
  if (C.field == Field::Complex) key += "g" + std::to_string(complex_generation);
  auto it = plans_.find(key);
  if (it != plans_.end()) return *it->second;

  auto plan = std::make_unique<GettPlan>();
  plan->generation = complex_generation;
  std::string Mi, Ni, Ki;
  for (char c : C.idx) {
    const bool inA = A0.find(c) >= 0, inB = B0.find(c) >= 0;
    CC4S_ASSERT(!(inA && inB), std::string("index '") + c +
                                   "' in both operands and result is not a contraction");
    CC4S_ASSERT(inA || inB, std::string("result index '") + c + "' not in any operand");
    (inA ? Mi : Ni) += c;
  }
  for (char c : A0.idx) {
    if (C.find(c) >= 0) continue;
    CC4S_ASSERT(B0.find(c) >= 0, std::string("index '") + c + "' only in one operand");
    Ki += c;
  }
  for (char c : B0.idx)
    CC4S_ASSERT(C.find(c) >= 0 || A0.find(c) >= 0,
                std::string("index '") + c + "' only in one operand");
  for (char c : Ki)
    CC4S_ASSERT(A0.len(c) == B0.len(c), std::string("length mismatch of '") + c + "'");
  if (D) {
    CC4S_ASSERT(D->rank() == C.rank(), "added tensor has other indices");
    for (char c : C.idx)
      CC4S_ASSERT(D->find(c) >= 0 && D->len(c) == C.len(c), "length mismatch (added tensor)");
  }
  for (char c : Mi) CC4S_ASSERT(A0.len(c) == C.len(c), "length mismatch (A, C)");
  for (char c : Ni) CC4S_ASSERT(B0.len(c) == C.len(c), "length mismatch (B, C)");

  // make C contiguous along N: if its fastest index belongs to A, exchange
  // the operands and compute the transposed problem
  char cfast = 0;
  int64_t cmin = INT64_MAX;
  for (int d = 0; d < C.rank(); ++d)
    if (C.lens[d] > 1 && C.strides[d] < cmin) { cmin = C.strides[d]; cfast = C.idx[d]; }
  plan->swap = cfast && Mi.find(cfast) != std::string::npos;
  const View &A = plan->swap ? B0 : A0;
  const View &B = plan->swap ? A0 : B0;
  if (plan->swap) std::swap(Mi, Ni);

  auto by = [](const View &v) {
    return [&v](char x, char y) { return v.stride(x) < v.stride(y); };
  };
  std::stable_sort(Mi.begin(), Mi.end(), by(A));
  std::stable_sort(Ni.begin(), Ni.end(), by(C));
  bool a_unit_k = false;
  for (char c : Ki) a_unit_k |= A.stride(c) == 1 && A.len(c) > 1;
  std::stable_sort(Ki.begin(), Ki.end(), a_unit_k ? by(A) : by(B));

  auto unit = [](const View &v, const std::string &g) {
    return !g.empty() && v.stride(g[0]) == 1 && v.len(g[0]) > 1;
  };
  plan->a_kc = unit(A, Ki) || !unit(A, Mi);
  plan->b_kc = unit(B, Ki) || !unit(B, Ni);

  const std::vector<OffsetTable> tables = [&] {
    std::vector<OffsetTable> t = {{&A, Mi, false, &plan->rowA}, {&A, Ki, true, &plan->colA},
                            {&B, Ki, true, &plan->rowB},  {&B, Ni, false, &plan->colB},
                            {&C, Mi, false, &plan->rowC}, {&C, Ni, false, &plan->colC}};
    if (D) {
      t.push_back({D, Mi, false, &plan->rowD});
      t.push_back({D, Ni, false, &plan->colD});
    }
    return t;
  }();
  plan->M = tables[0].entries();
  plan->N = tables[3].entries();
  plan->K = tables[1].entries();  // an outer product has one k with offset 0
  build_tables(tables.data(), static_cast<int>(tables.size()));

  choose_tile(C.field, plan->M, plan->N, plan->K, max_workspace, *plan);

  auto &ref = *plan;
  plans_.emplace(key, std::move(plan));
  return ref;
}

// the workspace for a plan's partial sums, or null
void *ContractionEngine::reserve_partials(const GettPlan &P, Field f) {
  size_t elements = 0;
  if (P.splits > 1) {
    elements = static_cast<size_t>(P.splits) * P.M * P.N;
  } else if (P.tail_splits > 1) {
    const TileShape t = tile_shape(f, P.tile, P.generation);
    const int64_t tiles = ((P.M + t.BM - 1) / t.BM) * ((P.N + t.BN - 1) / t.BN);
    elements = static_cast<size_t>(P.tail_splits) * (tiles - P.full_tiles) * t.BM * t.BN;
  }
  if (elements == 0) return nullptr;
  workspace_.reserve(elements * scalar_bytes(f));
  return workspace_.get();
}

void ContractionEngine::contract(double alpha, const View &A, const View &B,
                                 double beta, const View &C, const View *D,
                                 const OperandMax *maxA) {
  CC4S_ASSERT(A.field == C.field && B.field == C.field, "mixed scalar fields");
  CC4S_ASSERT(!C.conj, "conjugated result view");
  CC4S_ASSERT(!D || (D->field == C.field && !mixed_), "added tensor in a split pass");
  if (D && C.field == Field::Complex && complex_generation == 1) {
    sum(1.0, *D, 0.0, C);
    D = nullptr;
  }
  GettPlan &P = plan_for(A, B, C, D);
  if (P.M == 0 || P.N == 0) return;
  GettLaunch L;
  L.field = C.field;
  L.A = P.swap ? B.ptr : A.ptr;
  L.B = P.swap ? A.ptr : B.ptr;
  L.conjA = P.swap ? B.conj : A.conj;
  L.conjB = P.swap ? A.conj : B.conj;
  L.C = C.ptr;
  L.rowA = P.rowA; L.colA = P.colA; L.rowB = P.rowB; L.colB = P.colB;
  L.rowC = P.rowC; L.colC = P.colC;
  if (D) {
    L.D = D->ptr;
    L.conjD = D->conj;
    L.rowD = P.rowD; L.colD = P.colD;
  }
  L.M = P.M; L.N = P.N; L.K = P.K;
  L.splits = P.splits;
  L.tile = static_cast<int>(P.tile);
  L.generation = P.generation;
  L.full_tiles = P.full_tiles;
  L.tail_splits = P.tail_splits;
  L.alpha = alpha; L.beta = beta;
  L.a_kcontig = P.a_kc; L.b_kcontig = P.b_kc;
  const double flops = (C.field == Field::Complex ? 8.0 : 2.0) * double(P.M) *
                       double(P.N) * double(P.K);
  if (mixed_ && C.field == Field::Complex && flops >= mixed_min_flops) {
    contract_mixed(P, alpha, A, B, beta, C, flops, maxA);
    stats.flops += flops;
    stats.launches += 1;
    return;
  }
  // a small contraction of a group waits for its end
  if (grouping_ && !profiling_ && P.tile == Tile::Small && P.tail_splits == 1 &&
      P.M * P.N * P.splits < kGroupElements &&
      (C.field == Field::Real || P.generation == 3)) {
    group_.push_back(L);
    stats.flops += flops;
    stats.launches += 1;
    return;
  }
  L.W = reserve_partials(P, C.field);
  if (profiling_) {
    Pending p{take_event(), take_event(), gett_variant(L), flops};
    launch_gett(L, stream_, p.start, p.stop);
    pending_.push_back(p);
    if (pending_.size() > 4096) (void)timings();
  } else {
    launch_gett(L, stream_);
  }
  stats.flops += flops;
  stats.launches += 1;
}

void ContractionEngine::launch_group() {
  std::vector<GettLaunch> all;
  all.swap(group_);
  for (size_t first = 0; first < all.size(); first += kGroup) {
    const size_t n = std::min<size_t>(kGroup, all.size() - first);
    size_t bytes = 0;
    for (size_t i = 0; i < n; ++i)
      if (all[first + i].splits > 1)
        bytes += static_cast<size_t>(all[first + i].splits) * all[first + i].M *
                 all[first + i].N * scalar_bytes(all[first + i].field);
    workspace_.reserve(bytes);
    const bool cplx = all[first].field == Field::Complex;
    GroupArgs g{}, r{};
    size_t used = 0;
    for (size_t i = 0; i < n; ++i) {
      GettLaunch &L = all[first + i];
      if (L.splits > 1) {
        L.W = workspace_.as<char>() + used;
        used += static_cast<size_t>(L.splits) * L.M * L.N * scalar_bytes(L.field);
      }
      const KArgs a = kernel_args(L);
      g.k[i] = a;
      g.orient[i] = 2 * (L.a_kcontig ? 1 : 0) + (L.b_kcontig ? 1 : 0);
      g.first[i + 1] = g.first[i] + a.tilesM * a.tilesN * L.splits;
      if (L.splits > 1) {
        r.k[r.count] = a;
        r.orient[r.count] = L.splits;
        r.first[r.count + 1] = r.first[r.count] + static_cast<int>((L.M * L.N + 63) / 64);
        ++r.count;
      }
    }
    g.count = static_cast<int>(n);
    if (n == 1 && !r.count) {
      launch_gett(all[first], stream_);
      continue;
    }
    if (cplx)
      gett_group_kernel<true><<<g.first[n], 256, 0, stream_>>>(g);
    else
      gett_group_kernel<false><<<g.first[n], 256, 0, stream_>>>(g);
    CC4S_HIP(hipGetLastError());
    if (!r.count) continue;
    if (cplx)
      group_reduce_kernel<true><<<r.first[r.count], 256, 0, stream_>>>(r);
    else
      group_reduce_kernel<false><<<r.first[r.count], 256, 0, stream_>>>(r);
    CC4S_HIP(hipGetLastError());
  }
}

void ContractionEngine::contract_mixed(GettPlan &P, double alpha, const View &A,
                                       const View &B, double beta, const View &C,
                                       double flops, const OperandMax *maxA) {
  // 9 products per complex MAC: half parts plus a third plane of Re + Im
  const bool nine = mixed_half && mixed_terms == 9;
  const int terms = mixed_terms == 9 && !mixed_half ? 12 : mixed_terms;
  const size_t eb = nine ? 12 : 8;  // packed bytes per element and k
  const MixedTile T = mixed_tile(terms);
  const int64_t Mp = (P.M + T.BM - 1) / T.BM * T.BM;
  const int64_t Np = (P.N + T.BN - 1) / T.BN * T.BN;
  const int64_t Kfull = (P.K + T.BK - 1) / T.BK * T.BK;
  const View &Aop = P.swap ? B : A;
  const View &Bop = P.swap ? A : B;
  // an operand marked constant (a cache slot holds its pointer) is packed
  // once over the full K range
  auto slot_of = [&](const View &v) {
    for (int s = 0; s < kCacheSlots; ++s)
      if (cache_ptr_[s] && v.ptr == cache_ptr_[s] &&
          (cache_idx_[s].empty() || v.idx == cache_idx_[s]))
        return s;
    return -1;
  };
  const int slotA = slot_of(Aop);
  const int slotB = slotA < 0 ? slot_of(Bop) : -1;
  const bool cacheA = slotA >= 0, cacheB = slotB >= 0;
  const int slot = cacheA ? slotA : slotB;
  // half split: per-operand scales (A, B, the cache slots) and reduction room
  double *scA = nullptr, *scB = nullptr, *scC = nullptr, *scPart = nullptr;
  if (mixed_half) {
    scales_.reserve((2 + kCacheSlots) * sizeof(double) + split_scale_partials_bytes());
    scA = scales_.as<double>();
    scB = scA + 1;
    scC = scA + 2 + (slot > 0 ? slot : 0);
    scPart = scA + 2 + kCacheSlots;
  }
  if (cacheA || cacheB) {
    const int64_t rows = cacheA ? Mp : Np;
    if (cache_plan_[slot] != &P || cache_is_a_[slot] != cacheA || cache_eb_[slot] != eb) {
      cache_plan_[slot] = nullptr;  // not that plan's operand any more
      cache_[slot].reserve(static_cast<size_t>(rows) * Kfull * eb);
      char *cs = nine ? cache_[slot].as<char>() + static_cast<size_t>(rows) * Kfull * 8
                      : nullptr;
      if (cacheA) {
        if (mixed_half)
          launch_split_scale(static_cast<const double *>(Aop.ptr), P.rowA, P.colA, P.M,
                             P.K, P.a_kc, nine, scPart, scC, stream_);
        launch_pack(static_cast<const double *>(Aop.ptr), P.rowA, P.colA, P.M, P.K, 0,
                    Kfull, Mp, Aop.conj, P.a_kc, cache_[slot].get(), cs, scC, stream_);
      } else {
        if (mixed_half)
          launch_split_scale(static_cast<const double *>(Bop.ptr), P.colB, P.rowB, P.N,
                             P.K, P.b_kc, nine, scPart, scC, stream_);
        launch_pack(static_cast<const double *>(Bop.ptr), P.colB, P.rowB, P.N, P.K, 0,
                    Kfull, Np, Bop.conj, P.b_kc, cache_[slot].get(), cs, scC, stream_);
      }
      cache_plan_[slot] = &P;
      cache_is_a_[slot] = cacheA;
      cache_eb_[slot] = eb;
    }
  }
  const OperandMax *known = uses_operand_max() ? maxA : nullptr;  // of A, Bop where P.swap
  if (mixed_half && !cacheA && known && !P.swap)
    launch_split_scale_of(known->parts, known->count, scA, stream_);
  else if (mixed_half && !cacheA)
    launch_split_scale(static_cast<const double *>(Aop.ptr), P.rowA, P.colA, P.M, P.K,
                       P.a_kc, nine, scPart, scA, stream_);
  if (mixed_half && !cacheB && known && P.swap)
    launch_split_scale_of(known->parts, known->count, scB, stream_);
  else if (mixed_half && !cacheB)
    launch_split_scale(static_cast<const double *>(Bop.ptr), P.colB, P.rowB, P.N, P.K,
                       P.b_kc, nine, scPart, scB, stream_);
  const double *useScA = mixed_half ? (cacheA ? scC : scA) : nullptr;
  const double *useScB = mixed_half ? (cacheB ? scC : scB) : nullptr;
  const int64_t packed_rows = (cacheA ? 0 : Mp) + (cacheB ? 0 : Np);
  int64_t Kc = packed_rows > 0
                   ? static_cast<int64_t>(pack_budget / (static_cast<size_t>(packed_rows) * eb))
                   : Kfull;
  Kc = std::max<int64_t>(T.BK, Kc / T.BK * T.BK);
  Kc = std::min(Kc, Kfull);
  // split K inside a chunk when the tile grid cannot fill the CUs twice
  const int64_t tiles = (Mp / T.BM) * (Np / T.BN);
  int splits = 1;
  if (tiles < 512) {
    int64_t sp = std::min<int64_t>((1024 + tiles - 1) / tiles, Kc / (4 * T.BK));
    while (sp > 1 && static_cast<size_t>(sp) * P.M * P.N * 16 > max_workspace) --sp;
    splits = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(sp, 256)));
  }
  // no FP32 sum (one split of one chunk) runs over more than mixed_max_k
  Kc = std::min<int64_t>(Kc, std::max<int64_t>(T.BK, mixed_max_k * splits / T.BK * T.BK));
  const int64_t chunks = (P.K + Kc - 1) / Kc;
  pack_.reserve(static_cast<size_t>(packed_rows) * Kc * eb);
  char *Apk = pack_.as<char>();
  char *Bpk = Apk + (cacheA ? 0 : static_cast<size_t>(Mp) * Kc * 8);
  // the Re + Im planes follow the main planes
  char *Aps = nine ? Apk + static_cast<size_t>(packed_rows) * Kc * 8 : nullptr;
  char *Bps = nine ? Aps + (cacheA ? 0 : static_cast<size_t>(Mp) * Kc * 4) : nullptr;
  const char *cacheS =
      nine && (cacheA || cacheB)
          ? cache_[slot].as<char>() + static_cast<size_t>(cacheA ? Mp : Np) * Kfull * 8
          : nullptr;
  double *W = nullptr;
  if (splits > 1) {
    workspace_.reserve(static_cast<size_t>(splits) * P.M * P.N * (nine ? 16 : 8));
    W = workspace_.as<double>();
  }
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (profiling_) {
    e0 = take_event();
    e1 = take_event();
    CC4S_HIP(hipEventRecord(e0, stream_));
  }
  for (int64_t c = 0; c < chunks; ++c) {
    const int64_t k0 = c * Kc;
    const int64_t kc = std::min(Kc, (P.K - k0 + T.BK - 1) / T.BK * T.BK);
    const void *Ause = cacheA ? static_cast<const void *>(cache_[slot].as<char>() +
                                                          static_cast<size_t>(k0) * Mp * 8)
                              : Apk;
    const void *Buse = cacheB ? static_cast<const void *>(cache_[slot].as<char>() +
                                                          static_cast<size_t>(k0) * Np * 8)
                              : Bpk;
    const void *AuseS = !nine ? nullptr
                        : cacheA ? static_cast<const void *>(cacheS + static_cast<size_t>(k0) * Mp * 4)
                                 : Aps;
    const void *BuseS = !nine ? nullptr
                        : cacheB ? static_cast<const void *>(cacheS + static_cast<size_t>(k0) * Np * 4)
                                 : Bps;
    if (!cacheA)
      launch_pack(static_cast<const double *>(Aop.ptr), P.rowA, P.colA, P.M, P.K, k0,
                  kc, Mp, Aop.conj, P.a_kc, Apk, Aps, useScA, stream_);
    if (!cacheB)
      launch_pack(static_cast<const double *>(Bop.ptr), P.colB, P.rowB, P.N, P.K, k0,
                  kc, Np, Bop.conj, P.b_kc, Bpk, Bps, useScB, stream_);
    const double bc = c == 0 ? beta : 1.0;
    launch_bgemm(Ause, Buse, static_cast<double *>(C.ptr), W, P.rowC, P.colC, P.M,
                 P.N, Mp, Np, kc, splits, alpha, bc, useScA, useScB, terms, AuseS, BuseS,
                 stream_);
    if (splits > 1 && nine)
      launch_splitk_reduce(Field::Complex, W, static_cast<double *>(C.ptr), P.rowC,
                           P.colC, P.M, P.N, splits, alpha, bc, stream_);
    else if (splits > 1)
      launch_split_reduce(W, static_cast<double *>(C.ptr), P.rowC, P.colC, P.M, P.N,
                          splits, alpha, bc, useScA, useScB, stream_);
  }
  if (profiling_) {
    CC4S_HIP(hipEventRecord(e1, stream_));
    pending_.push_back(Pending{e0, e1, "mixed_c64", flops});
    if (pending_.size() > 4096) (void)timings();
  }
}

void ContractionEngine::sum(double alpha, const View &A, double beta,
                            const View &C) {
  CC4S_ASSERT(A.field == C.field, "mixed scalar fields");
  CC4S_ASSERT(C.rank() <= kMaxRank, "rank too large");
  CC4S_ASSERT(!C.conj, "conjugated result view");
  SumArgs a;
  a.A = static_cast<const double *>(A.ptr);
  a.C = static_cast<double *>(C.ptr);
  a.rank = C.rank();
  a.total = C.size();
  for (int d = 0; d < C.rank(); ++d) {
    const char c = C.idx[d];
    CC4S_ASSERT(A.find(c) >= 0 && A.len(c) == C.lens[d],
                std::string("sum: index '") + c + "' mismatch");
    a.lens[d] = C.lens[d];
    a.sC[d] = C.strides[d];
    a.sA[d] = A.stride(c);
  }
  CC4S_ASSERT(A.rank() == C.rank(), "sum: operand has extra indices");
  a.alpha = alpha;
  a.beta = beta;
  a.signA = A.conj ? -1.0 : 1.0;
  if (a.total == 0) return;
  if (C.field == Field::Complex)
    sum_kernel<true><<<grid_for(a.total), 256, 0, stream_>>>(a);
  else
    sum_kernel<false><<<grid_for(a.total), 256, 0, stream_>>>(a);
  CC4S_HIP(hipGetLastError());
}

void ContractionEngine::scale(double beta, const View &C) {
  SumArgs a;
  a.A = nullptr;
  a.C = static_cast<double *>(C.ptr);
  a.rank = C.rank();
  a.total = C.size();
  for (int d = 0; d < C.rank(); ++d) {
    a.lens[d] = C.lens[d];
    a.sC[d] = C.strides[d];
    a.sA[d] = 0;
  }
  a.alpha = 0.0;
  a.beta = beta;
  a.signA = 1.0;
  if (a.total == 0) return;
  if (C.field == Field::Complex)
    sum_kernel<true><<<grid_for(a.total), 256, 0, stream_>>>(a);
  else
    sum_kernel<false><<<grid_for(a.total), 256, 0, stream_>>>(a);
  CC4S_HIP(hipGetLastError());
}

}  // namespace cc4s_amd
