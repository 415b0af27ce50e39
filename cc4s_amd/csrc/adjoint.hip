// Energy adjoint kernels: the energy weights as a tensor (the FP64 gradient
// products and the structure factor contract it on the GETT), the FP32 gradient
// products with the weights recomputed from the amplitudes inside the product,
// and the per-G block dots of the structure factor.
#include "adjoint.hpp"

#include <type_traits>

namespace cc4s_amd {

namespace {

constexpr int kBlock = 256;
constexpr int kDotChunks = 64;  // fixed: deterministic reduction order

__device__ inline double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// Z from T1 and T2 [a,b,i,j] (CoupledCluster.cxx:223-231): complex
// Z_abij = 2 tau_abij - tau_baij, real Z_abij + Z_baji, tau = T2 + T1 T1.
// HBM-bound: a block takes the (a, b) tile pair {(A, B), (B, A)} at fixed
// (i, j), reads T2 along its contiguous index and meets the transposed element
// in LDS (real: also the tiles at (j, i), whose pair is read once more).
constexpr int kTile = 32;

template <bool CPLX>
__global__ __launch_bounds__(kBlock) void weights_kernel(
    const std::conditional_t<CPLX, double2, double> *__restrict__ T1,
    const std::conditional_t<CPLX, double2, double> *__restrict__ T2,
    std::conditional_t<CPLX, double2, double> *__restrict__ Z, int64_t No, int64_t Nv) {
  using T = std::conditional_t<CPLX, double2, double>;
  // [0]: (A, B), [1]: (B, A) at (i, j); [2], [3]: the same at (j, i)
  __shared__ T t[CPLX ? 2 : 4][kTile][kTile + 1];
  const int64_t nt = (Nv + kTile - 1) / kTile;
  const int64_t ntiles = nt * nt * No * No;
  for (int64_t tid = blockIdx.x; tid < ntiles; tid += gridDim.x) {
    const int64_t ta = tid % nt, tb = (tid / nt) % nt, ij = tid / (nt * nt);
    if (ta > tb) continue;  // the partner's block does it (uniform per block)
    const int64_t i = ij % No, j = ij / No;
    const int64_t a0 = ta * kTile, b0 = tb * kTile;
    const int64_t off = Nv * Nv * ij, offT = Nv * Nv * (j + No * i);
    __syncthreads();
    for (int e = threadIdx.x; e < kTile * kTile; e += kBlock) {
      const int u = e % kTile, w = e / kTile;
      const bool ox = a0 + u < Nv && b0 + w < Nv, oy = b0 + u < Nv && a0 + w < Nv;
      const int64_t x = (a0 + u) + Nv * (b0 + w), y = (b0 + u) + Nv * (a0 + w);
      t[0][u][w] = ox ? T2[off + x] : T{};
      t[1][u][w] = oy ? T2[off + y] : T{};
      if constexpr (!CPLX) {
        t[2][u][w] = ox ? T2[offT + x] : T{};
        t[3][u][w] = oy ? T2[offT + y] : T{};
      }
    }
    __syncthreads();
    // element (f0 + u, s0 + w) from its own tile p and the transposed one q
    auto put = [&](int64_t f0, int64_t s0, int p, int q, int u, int w) {
      const int64_t a = f0 + u, b = s0 + w;
      if (a >= Nv || b >= Nv) return;
      const T ai = T1[a + Nv * i], bj = T1[b + Nv * j], bi = T1[b + Nv * i], aj = T1[a + Nv * j];
      T z;
      if constexpr (CPLX) {
        const double2 d = cmul(ai, bj), x = cmul(bi, aj);
        z.x = 2.0 * (t[p][u][w].x + d.x) - (t[q][w][u].x + x.x);
        z.y = 2.0 * (t[p][u][w].y + d.y) - (t[q][w][u].y + x.y);
      } else {
        const double d = ai * bj, x = bi * aj;
        z = 2.0 * (t[p][u][w] + d) - (t[q][w][u] + x) + 2.0 * (t[q + 2][w][u] + d) -
            (t[p + 2][u][w] + x);
      }
      Z[off + a + Nv * b] = z;
    };
    for (int e = threadIdx.x; e < kTile * kTile; e += kBlock) {
      const int u = e % kTile, w = e / kTile;
      put(a0, b0, 0, 1, u, w);
      if (ta != tb) put(b0, a0, 1, 0, u, w);
    }
  }
}

// ---------------------------------------------------------------------------
// FP32 gradient products: C[G, n] = sum_k Gamma_blk[G, k] W(k, n), with the
// energy weights W recomputed from T1 and T2 for every tile as it is staged
// into LDS (no Z tensor exists).  Tile 128 (G) x 64 (n), 16 k per stage,
// double-buffered LDS, 8 waves of 32 x 32 on 16x16x4 MFMA, the four-product
// complex multiply (FP32 sums cancel too much in the three-product form's
// P3 - P1 - P2).  C is complex FP64, G fastest.  The FP64 products, which ran on
// this kernel at 55 % of the matrix rate (four amplitude reads and two complex
// multiplies per weight, once per 128 G), run on the GETT over Z instead: No=24,
// Nv=192, NG=1100 4.2 -> 2.4 ms per product, Z itself 0.3 ms.
//   kHP (complex): k = (b,j), n = (a,i), A = Gamma[G, No+b, j],
//                  W = conj Z_abij, C at G + NG (i + No a)
//   kPH (complex): k = (a,i), n = (b,j), A = Gamma[G, i, No+a],
//                  W = Z_abij, C at G + NG (b + Nv j)
//   kRE (real):    k = (b,j), n = (a,i), A = Gamma[G, No+b, j] (Re and Im are
//                  the two real vertex components), W = Z_abij + Z_baji (real),
//                  C at G + NG (a + Nv i)
enum { kHP = 0, kPH = 1, kRE = 2 };

typedef float flt4 __attribute__((ext_vector_type(4)));

__device__ inline flt4 mma(float a, float b, flt4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

struct GradArgs {
  const double2 *gamma;  // [NG, Np, Np]
  const double2 *T1c, *T2c;  // complex amplitudes
  const double *T1r, *T2r;   // real amplitudes
  double2 *C;
  int64_t NG, Np, No, Nv;
};

constexpr int kAT = 512;                  // 8 waves
constexpr int kABM = 128, kABN = 64, kABK = 16;
constexpr int kALA = kABM + 1, kALW = kABN + 1;

template <int MODE>
__global__ __launch_bounds__(kAT, 1) void grad_kernel(GradArgs p) {
  using P = float2;
  __shared__ P As[2][kABK][kALA];
  __shared__ P Ws[2][kABK][kALW];

  const int64_t NG = p.NG, No = p.No, Nv = p.Nv, Np = p.Np;
  const int64_t K = No * Nv, N = No * Nv;
  const uint32_t nv32 = static_cast<uint32_t>(Nv);
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int64_t g0 = static_cast<int64_t>(blockIdx.x) * kABM;
  const int64_t n0 = static_cast<int64_t>(blockIdx.y) * kABN;
  const int nst = static_cast<int>((K + kABK - 1) / kABK);

  // A elements of this thread: G = g0 + t % 128, k = 4e + t / 128 of a stage
  const int ag = t % kABM, ak = t / kABM;
  const bool gOk = g0 + ag < NG;
  const int64_t gIdx = gOk ? g0 + ag : 0;
  // W elements: n = n0 + t % 64, k = 8e + t / 64 of a stage
  const int wn = t % kABN, wk = t / kABN;
  const int64_t nn = n0 + wn;
  const bool nOk = nn < N;
  // the n index pair: (a, i) for kHP and kRE, (b, j) for kPH; fastest first
  const int64_t nf = nOk ? nn % Nv : 0, ns = nOk ? nn / Nv : 0;

  double2 ra[4];
  bool kaOk[4];
  // amplitude values of the two W elements, combined at the LDS store
  double2 t2a[2], t2b[2], t1a[2], t1b[2], t1c[2], t1d[2];
  double r2a[2], r2b[2], r2c[2], r2d[2], r1a[2], r1b[2], r1c[2], r1d[2];
  bool kwOk[2];

  auto t2c = [&](int64_t a, int64_t b, int64_t i, int64_t j) {
    return p.T2c[a + Nv * (b + Nv * (i + No * j))];
  };
  auto t2r = [&](int64_t a, int64_t b, int64_t i, int64_t j) {
    return p.T2r[a + Nv * (b + Nv * (i + No * j))];
  };
  auto load = [&](int s) {
    const int64_t kb = static_cast<int64_t>(s) * kABK;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t k = kb + 4 * e + ak;
      kaOk[e] = k < K;
      const int64_t kk = kaOk[e] ? k : 0;
      // (b, j) or (a, i); 32-bit division (No Nv < 2^31)
      const int64_t kf = static_cast<uint32_t>(kk) % nv32, ks = static_cast<uint32_t>(kk) / nv32;
      // Gamma[G, P, Q] at G + NG (P + Np Q)
      const int64_t P = MODE == kPH ? ks : No + kf, Q = MODE == kPH ? No + kf : ks;
      ra[e] = p.gamma[gIdx + NG * (P + Np * Q)];
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int64_t k = kb + 8 * e + wk;
      kwOk[e] = k < K && nOk;
      const int64_t kk = k < K ? k : 0;
      const int64_t kf = static_cast<uint32_t>(kk) % nv32, ks = static_cast<uint32_t>(kk) / nv32;
      int64_t a, b, i, j;
      if (MODE == kPH) {
        a = kf; i = ks; b = nf; j = ns;
      } else {
        b = kf; j = ks; a = nf; i = ns;
      }
      if constexpr (MODE != kRE) {
        t2a[e] = t2c(a, b, i, j);
        t2b[e] = t2c(b, a, i, j);
        t1a[e] = p.T1c[a + Nv * i];
        t1b[e] = p.T1c[b + Nv * j];
        t1c[e] = p.T1c[b + Nv * i];
        t1d[e] = p.T1c[a + Nv * j];
      } else {
        r2a[e] = t2r(a, b, i, j);
        r2b[e] = t2r(b, a, j, i);
        r2c[e] = t2r(b, a, i, j);
        r2d[e] = t2r(a, b, j, i);
        r1a[e] = p.T1r[a + Nv * i];
        r1b[e] = p.T1r[b + Nv * j];
        r1c[e] = p.T1r[b + Nv * i];
        r1d[e] = p.T1r[a + Nv * j];
      }
    }
  };
  auto cmul = [](double2 x, double2 y) {
    return make_double2(x.x * y.x - x.y * y.y, x.x * y.y + x.y * y.x);
  };
  // out-of-range elements are zeroed here, component by component (a select
  // of whole pairs would go through scratch memory)
  auto store = [&](int buf) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool ok = gOk && kaOk[e];
      As[buf][4 * e + ak][ag] = make_float2(ok ? ra[e].x : 0.0, ok ? ra[e].y : 0.0);
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      double zr, zi;
      if constexpr (MODE != kRE) {
        // Z_abij = 2 tau_abij - tau_baij, tau = T2 + T1 T1 (CoupledCluster.cxx:223-231)
        const double2 p1 = cmul(t1a[e], t1b[e]), p2 = cmul(t1c[e], t1d[e]);
        zr = 2.0 * (t2a[e].x + p1.x) - (t2b[e].x + p2.x);
        zi = 2.0 * (t2a[e].y + p1.y) - (t2b[e].y + p2.y);
        if (MODE == kHP) zi = -zi;
      } else {
        // Z_abij + Z_baji
        const double p1 = r1a[e] * r1b[e], p2 = r1c[e] * r1d[e];
        zr = 2.0 * (r2a[e] + p1) - (r2c[e] + p2) + 2.0 * (r2b[e] + p1) - (r2d[e] + p2);
        zi = 0.0;
      }
      Ws[buf][8 * e + wk][wn] = make_float2(kwOk[e] ? zr : 0.0, kwOk[e] ? zi : 0.0);
    }
  };

  const int wr = w / 2, wc = w % 2;  // the wave's 32 x 32 part of the tile
  flt4 a1[2][2], a2[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      a1[i][j] = flt4{0, 0, 0, 0};
      a2[i][j] = flt4{0, 0, 0, 0};
    }
  load(0);
  store(0);
  __syncthreads();
  for (int s = 0; s < nst; ++s) {
    const int buf = s & 1;
    if (s + 1 < nst) load(s + 1);
#pragma unroll
    for (int kq = 0; kq < kABK / 4; ++kq) {
      const int kr = kq * 4 + (lane >> 4);
      P x[2], y[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) x[i] = As[buf][kr][wr * 32 + i * 16 + (lane & 15)];
#pragma unroll
      for (int j = 0; j < 2; ++j) y[j] = Ws[buf][kr][wc * 32 + j * 16 + (lane & 15)];
      if constexpr (MODE == kRE) {
        // real W: re and im of Gamma times W
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            a1[i][j] = mma(x[i].x, y[j].x, a1[i][j]);
            a2[i][j] = mma(x[i].y, y[j].x, a2[i][j]);
          }
      } else {
        // four products: a1 = re, a2 = im
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            a1[i][j] = mma(x[i].x, y[j].x, a1[i][j]);
            a2[i][j] = mma(x[i].x, y[j].y, a2[i][j]);
          }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            a1[i][j] = mma(-x[i].y, y[j].y, a1[i][j]);
            a2[i][j] = mma(x[i].y, y[j].x, a2[i][j]);
          }
      }
    }
    // the other buffer was read in stage s-1, released by its barrier
    if (s + 1 < nst) store(buf ^ 1);
    __syncthreads();
  }

#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int64_t n = n0 + wc * 32 + j * 16 + (lane & 15);
    if (n >= N) continue;
    const int64_t f = n % Nv, sl = n / Nv;
    // output column of n: (i + No a) for kHP, (b + Nv j) for kPH, (a + Nv i) for kRE
    const int64_t col = MODE == kHP ? sl + No * f : n;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t G = g0 + wr * 32 + i * 16 + 4 * (lane >> 4) + r;
        if (G >= NG) continue;
        const double re = a1[i][j][r], im = a2[i][j][r];
        p.C[G + NG * col] = make_double2(re, im);
      }
  }
}

// partials[c * NG + G]: chunk c of the flattened (x, y) range of one block
__global__ __launch_bounds__(kBlock) void block_dots_kernel(
    const double2 *gamma, int64_t NG, int64_t Np, int64_t row0, int64_t rows,
    int64_t col0, int64_t cols, const double2 *g, double *partials) {
  const int64_t G = blockIdx.x * int64_t(kBlock) + threadIdx.x;
  if (G >= NG) return;
  const int64_t n = rows * cols;
  const int64_t c = blockIdx.y;
  const int64_t e0 = n * c / kDotChunks, e1 = n * (c + 1) / kDotChunks;
  double s = 0.0;
  for (int64_t e = e0; e < e1; ++e) {
    const int64_t x = e % rows, y = e / rows;
    const double2 v = gamma[G + NG * ((row0 + x) + Np * (col0 + y))];
    const double2 w = g[G + NG * e];
    s += v.x * w.x + v.y * w.y;  // Re(conj(v) w)
  }
  partials[c * NG + G] = s;
}

__global__ __launch_bounds__(kBlock) void block_dots_finish_kernel(
    const double *partials, int64_t NG, double factor, int accumulate, double *out) {
  const int64_t G = blockIdx.x * int64_t(kBlock) + threadIdx.x;
  if (G >= NG) return;
  double s = 0.0;
  for (int c = 0; c < kDotChunks; ++c) s += partials[c * NG + G];
  out[G] = (accumulate ? out[G] : 0.0) + factor * s;
}

}  // namespace

void energy_weights(hipStream_t s, Field f, const void *T, int64_t No,
                    int64_t Nv, void *Z) {
  const int64_t nt = (Nv + kTile - 1) / kTile;
  const int blocks = static_cast<int>(std::min<int64_t>(nt * nt * No * No, 256 * 32));
  if (f == Field::Complex) {
    const double2 *t = static_cast<const double2 *>(T);
    weights_kernel<true><<<blocks, kBlock, 0, s>>>(t, t + Nv * No, static_cast<double2 *>(Z), No,
                                                   Nv);
  } else {
    const double *t = static_cast<const double *>(T);
    weights_kernel<false><<<blocks, kBlock, 0, s>>>(t, t + Nv * No, static_cast<double *>(Z), No,
                                                    Nv);
  }
  CC4S_HIP(hipGetLastError());
}

void energy_gradient_product_fp32(hipStream_t s, Field f, GradientBlock blk,
                                  const void *gamma, const void *T, int64_t NG, int64_t No,
                                  int64_t Nv, void *C) {
  CC4S_ASSERT(NG > 0 && No > 0 && Nv > 0, "empty gradient product");
  CC4S_ASSERT(f == Field::Complex || blk == GradientBlock::PH,
              "the real field has the ph gradient block only");
  GradArgs a{};
  a.gamma = static_cast<const double2 *>(gamma);
  a.C = static_cast<double2 *>(C);
  a.NG = NG;
  a.No = No;
  a.Nv = Nv;
  a.Np = No + Nv;
  if (f == Field::Complex) {
    a.T1c = static_cast<const double2 *>(T);
    a.T2c = a.T1c + Nv * No;
  } else {
    a.T1r = static_cast<const double *>(T);
    a.T2r = a.T1r + Nv * No;
  }
  const int64_t gy = (No * Nv + kABN - 1) / kABN;
  CC4S_ASSERT(gy <= 65535 && No * Nv < (int64_t(1) << 31), "gradient product too wide");
  const dim3 grid(static_cast<unsigned>((NG + kABM - 1) / kABM), static_cast<unsigned>(gy));
  const int mode = f == Field::Real ? kRE : (blk == GradientBlock::HP ? kHP : kPH);
  if (mode == kHP)
    grad_kernel<kHP><<<grid, dim3(kAT), 0, s>>>(a);
  else if (mode == kPH)
    grad_kernel<kPH><<<grid, dim3(kAT), 0, s>>>(a);
  else
    grad_kernel<kRE><<<grid, dim3(kAT), 0, s>>>(a);
  CC4S_HIP(hipGetLastError());
}

size_t block_dots_partials_size(int64_t NG) {
  return static_cast<size_t>(kDotChunks) * NG * sizeof(double);
}

void block_dots(hipStream_t s, const void *gamma, int64_t NG, int64_t Np,
                int64_t row0, int64_t rows, int64_t col0, int64_t cols,
                const void *g, double factor, bool accumulate, void *partials,
                double *out) {
  CC4S_ASSERT(row0 >= 0 && col0 >= 0 && row0 + rows <= Np && col0 + cols <= Np,
              "vertex block out of range");
  const unsigned gx = static_cast<unsigned>((NG + kBlock - 1) / kBlock);
  block_dots_kernel<<<dim3(gx, kDotChunks), kBlock, 0, s>>>(
      static_cast<const double2 *>(gamma), NG, Np, row0, rows, col0, cols,
      static_cast<const double2 *>(g), static_cast<double *>(partials));
  CC4S_HIP(hipGetLastError());
  block_dots_finish_kernel<<<gx, kBlock, 0, s>>>(static_cast<const double *>(partials),
                                                 NG, factor, accumulate ? 1 : 0, out);
  CC4S_HIP(hipGetLastError());
}

}  // namespace cc4s_amd
