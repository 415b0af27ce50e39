// Paired particle-particle ladder: the slab contraction of Ccsd.cxx:590 over
// pairs c <= d and i <= j (complex).
//
// tau has the pair symmetry tau_cdij = tau_dcji (T1 x T1 has it, and T2 where it
// holds to rounding; other amplitudes take the slab contraction), so with
//   tau+_cd(ij) = (tau_cdij + tau_cdji) / 2   symmetric in (c, d),
//   tau-_cd(ij) = (tau_cdij - tau_cdji) / 2   antisymmetric in (c, d),
// the slab contraction R_xyij = sum_cd V_xycd tau_cdij becomes
//   Rp_xy(ij) = sum_{c<=d} Vp_xy(cd) tau+_(cd)(ij),
//               Vp = V_xycd + V_xydc (c < d), V_xycc (c = d);
//   Rm_xy(ij) = sum_{c<d}  Vm_xy(cd) tau-_(cd)(ij),  Vm = V_xycd - V_xydc;
//   R_xyij = Rp + Rm and R_xyji = Rp - Rm (i < j), R_xyii = Rp_xy(ii):
// two contractions over about Nv^2/2 k and No^2/2 columns each, half the
// multiply-adds of the one over Nv^2 k and No^2 columns.
//
// Resident integrals (both fields).  For a Hermitian (symmetric) vertex the
// undressed integrals V_xycd do not change during a run, V_xycd = V_yxdc and
// V_cdxy = conj(V_xycd), so their pair combinations are two Hermitian matrices
//   S_(xy)(cd) = V_xycd + V_xydc   (x <= y, c <= d),
//   A_(xy)(cd) = V_xycd - V_xydc   (x < y, c < d)
// that are formed once (only the triangle d <= max(x, y): a quarter of the
// Nv^4 NG multiply-adds, half of what every pass spends on the dressed slabs)
// and kept in HBM.  The T1 dressing of Ccsd.cxx:509-510, 560-561 moves to the
// result: with the same combinations of V_kacd (k a hole) as further columns
// (k, a), one product per combination gives, for tau+- (tau+ halved at c = d),
//   R_abij = Rp + Rm  and  U_kaij = sum_cd V_kacd tau_cdij,
// and the dressed ladder is R_abij - T_ak U_kbij - T_bk U_kaji +
// T_ak T_bl (V_klcd tau_cdij), whose last term is the hole ladder's over tau
// instead of T2 (Ccsd.cxx:541-546).  The products are MFMA-bound GETTs over
// Nv^2/2 k; the three kernels here are HBM-bound and take under 5 % of them.
// Measured (one pass and the amplitudes read back, slabs -> resident): complex
// No=32, Nv=256, NG=1500 0.968 -> 0.570 s (the first pass, which forms S and A,
// 1.07 -> 0.85 s), No=12, Nv=60, NG=300 4.18 -> 2.57 ms; real No=31, Nv=243,
// NG=1201 0.578 -> 0.284 s.
//
// Triangular pair indices (column-major upper triangles): (c, d), c <= d ->
// c + d(d+1)/2; c < d -> c + d(d-1)/2; the same for (i, j).  Layouts, k
// fastest: tau+ [Kp][Np], tau- [Km][Nm], Vp [Kp][x][y], Vm [Km][x][y]; Rp
// [x][y][Np], Rm [x][y][Nm].
#include "ladder.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace cc4s_amd {

namespace {

// (i, j) of the upper-triangle pair index n (i <= j)
__device__ __forceinline__ void tri_pair(int64_t n, int64_t &i, int64_t &j) {
  int64_t jj = static_cast<int64_t>((sqrt(8.0 * static_cast<double>(n) + 1.0) - 1.0) * 0.5);
  while (jj * (jj + 1) / 2 > n) --jj;
  while ((jj + 1) * (jj + 2) / 2 <= n) ++jj;
  j = jj;
  i = n - jj * (jj + 1) / 2;
}

__device__ __forceinline__ double2 add2(double2 a, double2 b) {
  return make_double2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ double2 sub2(double2 a, double2 b) {
  return make_double2(a.x - b.x, a.y - b.y);
}

template <bool CPLX>
struct Num;
template <>
struct Num<true> {
  using T = double2;
  __device__ static T zero() { return make_double2(0.0, 0.0); }
  __device__ static T lin(double x, T a, double y, T b) {
    return make_double2(x * a.x + y * b.x, x * a.y + y * b.y);
  }
  __device__ static T conj(T a) { return make_double2(a.x, -a.y); }
};
template <>
struct Num<false> {
  using T = double;
  __device__ static T zero() { return 0.0; }
  __device__ static T lin(double x, T a, double y, T b) { return x * a + y * b; }
  __device__ static T conj(T a) { return a; }
};

// grid (ceil(v/256), v, Np): thread c, block row d, block column n = (i, j);
// the diagonal c = d of tau+ times `diag`
template <bool CPLX>
__global__ __launch_bounds__(256) void tau_pairs_kernel(const typename Num<CPLX>::T *tau,
                                                        typename Num<CPLX>::T *Tp,
                                                        typename Num<CPLX>::T *Tm, double diag,
                                                        int64_t v, int64_t o, int64_t Kp,
                                                        int64_t Km) {
  using N = Num<CPLX>;
  const int64_t c = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t d = blockIdx.y;
  if (c > d) return;
  int64_t i, j;
  tri_pair(blockIdx.z, i, j);
  const int64_t vv = v * v;
  const auto t1 = tau[c + v * d + vv * (i + o * j)];
  const auto t2 = tau[c + v * d + vv * (j + o * i)];
  const int64_t n = blockIdx.z;
  const double h = c == d ? 0.5 * diag : 0.5;
  Tp[c + d * (d + 1) / 2 + Kp * n] = N::lin(h, t1, h, t2);
  if (c < d && i < j)
    Tm[c + d * (d - 1) / 2 + Km * (i + j * (j - 1) / 2)] = N::lin(0.5, t1, -0.5, t2);
}

constexpr int kT = 32;  // (c, d) tile of the vertex fold

// one 32 x 32 tile (cb <= db) of the (c, d) plane of one (x, y): both
// orientations are read along their contiguous first index and meet in LDS.
// grid (tiles, cx * Ny)
__global__ __launch_bounds__(256) void vertex_pairs_kernel(const double2 *slab, double2 *Vp,
                                                           double2 *Vm, int64_t v, int64_t cx,
                                                           int64_t Kp, int64_t Km,
                                                           unsigned long long *maxima) {
  __shared__ double2 t1[kT][kT + 1];  // [d][c]: V_xycd
  __shared__ double2 t2[kT][kT + 1];  // [c][d]: V_xydc
  int64_t cb, db;
  tri_pair(blockIdx.x, cb, db);
  const int64_t xy = blockIdx.y;
  const int64_t x = xy % cx, y = xy / cx;
  const int64_t c0 = cb * kT, d0 = db * kT;
  // slab[c, x, d, y] at c + v (x + cx (d + v y))
  const int64_t sd = v * cx;
  const double2 *base = slab + v * (x + cx * v * y);
  const int t = threadIdx.x;
  for (int e = t; e < kT * kT; e += 256) {
    const int a = e % kT, b = e / kT;
    // V_xycd at c = c0 + a, d = d0 + b; V_xydc at d = d0 + a (first index), c = c0 + b
    const int64_t c1 = c0 + a, d1 = d0 + b;
    t1[b][a] = (c1 < v && d1 < v) ? base[c1 + sd * d1] : make_double2(0.0, 0.0);
    const int64_t d2 = d0 + a, c2 = c0 + b;
    t2[b][a] = (c2 < v && d2 < v) ? base[d2 + sd * c2] : make_double2(0.0, 0.0);
  }
  __syncthreads();
  const int64_t ox = xy;  // (x, y) column of Vp / Vm
  double mp = 0.0, mm = 0.0;
  auto larger = [](double m, double2 z) { return fmax(m, fmax(fabs(z.x), fabs(z.y))); };
  for (int e = t; e < kT * kT; e += 256) {
    const int a = e % kT, b = e / kT;
    const int64_t c = c0 + a, d = d0 + b;
    if (c > d || d >= v) continue;
    const double2 vcd = t1[b][a];
    if (c == d) {
      Vp[c + d * (d + 1) / 2 + Kp * ox] = vcd;
      mp = larger(mp, vcd);
    } else {
      const double2 vdc = t2[a][b], p = add2(vcd, vdc), m = sub2(vcd, vdc);
      Vp[c + d * (d + 1) / 2 + Kp * ox] = p;
      Vm[c + d * (d - 1) / 2 + Km * ox] = m;
      mp = larger(mp, p);
      mm = larger(mm, m);
    }
  }
  if (!maxima) return;
  // magnitudes order as their bits do
  mp = wave_max(mp);
  mm = wave_max(mm);
  if ((t & 63) == 0) {
    const int slot = (blockIdx.x + gridDim.x * blockIdx.y) % kLadderMaxima;
    atomicMax(maxima + slot, static_cast<unsigned long long>(__double_as_longlong(mp)));
    atomicMax(maxima + kLadderMaxima + slot,
              static_cast<unsigned long long>(__double_as_longlong(mm)));
  }
}

// grid (ceil(cx Ny / 256), o * o): R_xyij from Rp and Rm
__global__ __launch_bounds__(256) void unpack_pairs_kernel(const double2 *Rp, const double2 *Rm,
                                                           double2 *R, int64_t nxy, int64_t o) {
  const int64_t xy = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (xy >= nxy) return;
  const int64_t ij = blockIdx.y;
  const int64_t i = ij % o, j = ij / o;
  double2 r;
  if (i == j) {
    r = Rp[xy + nxy * (i + i * (i + 1) / 2)];
  } else if (i < j) {
    r = add2(Rp[xy + nxy * (i + j * (j + 1) / 2)], Rm[xy + nxy * (i + j * (j - 1) / 2)]);
  } else {
    r = sub2(Rp[xy + nxy * (j + i * (i + 1) / 2)], Rm[xy + nxy * (j + i * (i - 1) / 2)]);
  }
  R[xy + nxy * ij] = r;
}

// ---------------------------------------------------------------------------
// resident pair integrals
// ---------------------------------------------------------------------------

// One 32 x 32 tile (cb <= db) of the (c, d) plane (n values each) of one (x, y)
// of a slab V[c,x,d,y], folded into columns of S and A: S = V_xycd + V_xydc,
// A = sign (V_xycd - V_xydc).  HBM-bound: both orientations are read along
// their contiguous index and meet in LDS.  grid (tiles, cx * Ny)
//   particle pairs (PP): X = x0 + x >= Y = y, the column of the pair (Y, X) with
//     Y first, V_YXcd = V_xydc, so sign = -1; pairs Y > X are skipped;
//   (hole X, particle Y): the column v X + Y after the pair columns, sign = 1.
template <bool CPLX, bool PP>
__global__ __launch_bounds__(256) void pair_fold_kernel(
    const typename Num<CPLX>::T *__restrict__ slab, typename Num<CPLX>::T *__restrict__ S,
    typename Num<CPLX>::T *__restrict__ A, int64_t n, int64_t cx, int64_t x0, int64_t v) {
  using N = Num<CPLX>;
  __shared__ typename N::T t1[kT][kT + 1];  // [d][c]: V_xycd
  __shared__ typename N::T t2[kT][kT + 1];  // [c][d]: V_xydc
  const int64_t X = x0 + blockIdx.y % cx, Y = blockIdx.y / cx;
  if (PP && Y > X) return;  // uniform per block
  int64_t cb, db;
  tri_pair(blockIdx.x, cb, db);
  const int64_t Kp = v * (v + 1) / 2, Km = v * (v - 1) / 2;
  const int64_t mp = PP ? X * (X + 1) / 2 + Y : Kp + v * X + Y;
  const int64_t mm = PP ? X * (X - 1) / 2 + Y : Km + v * X + Y;
  const bool anti = !PP || Y < X;
  const double s = PP ? -1.0 : 1.0;
  const int64_t c0 = cb * kT, d0 = db * kT;
  const int64_t sd = n * cx;
  const auto *base = slab + n * (X - x0 + cx * n * Y);
  const int t = threadIdx.x;
  for (int e = t; e < kT * kT; e += 256) {
    const int a = e % kT, b = e / kT;
    const int64_t c1 = c0 + a, d1 = d0 + b;
    t1[b][a] = (c1 < n && d1 < n) ? base[c1 + sd * d1] : N::zero();
    const int64_t d2 = d0 + a, c2 = c0 + b;
    t2[b][a] = (c2 < n && d2 < n) ? base[d2 + sd * c2] : N::zero();
  }
  __syncthreads();
  for (int e = t; e < kT * kT; e += 256) {
    const int a = e % kT, b = e / kT;
    const int64_t c = c0 + a, d = d0 + b;
    if (c > d || d >= n) continue;
    const auto vcd = t1[b][a], vdc = t2[a][b];
    S[c + d * (d + 1) / 2 + Kp * mp] = N::lin(1.0, vcd, 1.0, vdc);
    if (anti && c < d) A[c + d * (d - 1) / 2 + Km * mm] = N::lin(s, vcd, -s, vdc);
  }
}

// M[k + n m] = conj(M[m + n k]) for k > m, 32 x 32 tiles through LDS; one block
// per tile pair bi <= bj (HBM-bound: n^2/2 elements read, n^2/2 written)
template <bool CPLX>
__global__ __launch_bounds__(256) void mirror_kernel(typename Num<CPLX>::T *M, int64_t n) {
  using N = Num<CPLX>;
  __shared__ typename N::T t[kT][kT + 1];
  int64_t bi, bj;
  tri_pair(blockIdx.x, bi, bj);
  const int64_t r0 = bi * kT, c0 = bj * kT;
  for (int e = threadIdx.x; e < kT * kT; e += 256) {
    const int a = e % kT, b = e / kT;
    const int64_t r = r0 + a, c = c0 + b;
    t[b][a] = (r < n && c < n && r < c) ? M[r + n * c] : N::zero();
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kT * kT; e += 256) {
    const int a = e % kT, b = e / kT;
    const int64_t c = c0 + a, r = r0 + b;  // element (c, r), c > r
    if (r < n && c < n && r < c) M[c + n * r] = N::conj(t[a][b]);
  }
}

// Rp [n][Np], Rm [n][Nm] (n fastest) of the resident ladder into
//   blockIdx.y = b < v:  R2[a,b,i,j] += f (Rp +- Rm) of the pair of a and b;
//   blockIdx.y = v + k:  Q[a,k,i,j] += (Rp -+ Rm) of the row (k, a),
// the sign after the order of (i, j) (and of (a, b)).  A block turns 32 x 32
// (n, a) through LDS: rows are read along n, written along a.
// grid (ceil(v/32), v + o, ceil(Np/32))
template <bool CPLX>
__global__ __launch_bounds__(256) void resident_unpack_kernel(
    const typename Num<CPLX>::T *__restrict__ Rp, const typename Num<CPLX>::T *__restrict__ Rm,
    typename Num<CPLX>::T *__restrict__ R2, typename Num<CPLX>::T *__restrict__ Q, double f,
    int64_t v, int64_t o) {
  using N = Num<CPLX>;
  __shared__ typename N::T p[kT][kT + 1], q[kT][kT + 1];  // [a][n]
  const int64_t Kp = v * (v + 1) / 2, Km = v * (v - 1) / 2;
  const int64_t Np = o * (o + 1) / 2, Nm = o * (o - 1) / 2;
  const int64_t a0 = static_cast<int64_t>(blockIdx.x) * kT;
  const int64_t n0 = static_cast<int64_t>(blockIdx.z) * kT;
  const bool ring = blockIdx.y >= v;
  const int64_t b = ring ? blockIdx.y - v : blockIdx.y;  // k for Q
  for (int e = threadIdx.x; e < kT * kT; e += 256) {
    const int u = e % kT, w = e / kT;
    const int64_t n = n0 + u, a = a0 + w;
    typename N::T x = N::zero(), y = N::zero();
    if (n < Np && a < v) {
      int64_t i, j;
      tri_pair(n, i, j);
      const int64_t lo = a < b ? a : b, hi = a < b ? b : a;
      const int64_t mp = ring ? Kp + a + v * b : hi * (hi + 1) / 2 + lo;
      const int64_t mm = ring ? Km + a + v * b : hi * (hi - 1) / 2 + lo;
      x = Rp[n + Np * mp];
      // (i, j), i < j, is column n - j of the antisymmetric part
      if (i < j && (ring || lo < hi)) y = Rm[n - j + Nm * mm];
    }
    p[w][u] = x;
    q[w][u] = y;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kT * kT; e += 256) {
    const int u = e % kT, w = e / kT;
    const int64_t a = a0 + u, n = n0 + w;
    if (n >= Np || a >= v) continue;
    int64_t i, j;
    tri_pair(n, i, j);
    const auto x = p[u][w], y = q[u][w];
    // Q_akij takes U_kaji: the order (j, i) of the row (k, a)
    const double s = ring ? -1.0 : (a < b ? f : -f), g = ring ? 1.0 : f;
    auto *out = ring ? Q + a + v * b : R2 + a + v * b;
    const int64_t st = ring ? v * o : v * v;
    auto *c1 = out + st * (i + o * j);
    *c1 = N::lin(1.0, *c1, 1.0, N::lin(g, x, s, y));
    if (i < j) {
      auto *c2 = out + st * (j + o * i);
      *c2 = N::lin(1.0, *c2, 1.0, N::lin(g, x, -s, y));
    }
  }
}

}  // namespace

void ladder_tau_pairs(Field f, const void *tau, void *Tp, void *Tm, double diag, int64_t v,
                      int64_t o, hipStream_t s) {
  const int64_t Kp = v * (v + 1) / 2, Km = v * (v - 1) / 2, Np = o * (o + 1) / 2;
  CC4S_ASSERT(v > 0 && o > 0 && Np < 65536 && v < 65536, "paired ladder: shape out of range");
  const dim3 grid(static_cast<unsigned>((v + 255) / 256), static_cast<unsigned>(v),
                  static_cast<unsigned>(Np));
  if (f == Field::Complex)
    tau_pairs_kernel<true><<<grid, 256, 0, s>>>(
        static_cast<const double2 *>(tau), static_cast<double2 *>(Tp),
        static_cast<double2 *>(Tm), diag, v, o, Kp, Km);
  else
    tau_pairs_kernel<false><<<grid, 256, 0, s>>>(
        static_cast<const double *>(tau), static_cast<double *>(Tp),
        static_cast<double *>(Tm), diag, v, o, Kp, Km);
  CC4S_HIP(hipGetLastError());
}

void resident_fold(Field f, bool particles, const void *slab, void *S, void *A, int64_t n,
                   int64_t cx, int64_t Ny, int64_t x0, int64_t v, hipStream_t s) {
  const int64_t nb = (n + kT - 1) / kT;
  CC4S_ASSERT(n > 0 && n <= v && Ny <= v && cx * Ny < 65536,
              "resident ladder: slab chunk out of range");
  const dim3 grid(static_cast<unsigned>(nb * (nb + 1) / 2), static_cast<unsigned>(cx * Ny));
  auto launch = [&](auto kernel, auto *zero) {
    using T = std::remove_pointer_t<decltype(zero)>;
    kernel<<<grid, 256, 0, s>>>(static_cast<const T *>(slab), static_cast<T *>(S),
                                static_cast<T *>(A), n, cx, x0, v);
  };
  double2 *z2 = nullptr;
  double *z1 = nullptr;
  if (f == Field::Complex)
    particles ? launch(pair_fold_kernel<true, true>, z2) : launch(pair_fold_kernel<true, false>, z2);
  else
    particles ? launch(pair_fold_kernel<false, true>, z1)
              : launch(pair_fold_kernel<false, false>, z1);
  CC4S_HIP(hipGetLastError());
}

void resident_mirror(Field f, void *M, int64_t n, hipStream_t s) {
  const int64_t nb = (n + kT - 1) / kT;
  CC4S_ASSERT(n > 0 && nb * (nb + 1) / 2 < (int64_t(1) << 31), "resident ladder: too large");
  const unsigned grid = static_cast<unsigned>(nb * (nb + 1) / 2);
  if (f == Field::Complex)
    mirror_kernel<true><<<grid, 256, 0, s>>>(static_cast<double2 *>(M), n);
  else
    mirror_kernel<false><<<grid, 256, 0, s>>>(static_cast<double *>(M), n);
  CC4S_HIP(hipGetLastError());
}

void resident_unpack(Field f, const void *Rp, const void *Rm, void *R2, void *Q, double factor,
                     int64_t v, int64_t o, hipStream_t s) {
  const int64_t Np = o * (o + 1) / 2;
  CC4S_ASSERT(v + o < 65536 && (Np + kT - 1) / kT < 65536, "resident ladder: shape out of range");
  const dim3 grid(static_cast<unsigned>((v + kT - 1) / kT), static_cast<unsigned>(v + o),
                  static_cast<unsigned>((Np + kT - 1) / kT));
  if (f == Field::Complex)
    resident_unpack_kernel<true><<<grid, 256, 0, s>>>(
        static_cast<const double2 *>(Rp), static_cast<const double2 *>(Rm),
        static_cast<double2 *>(R2), static_cast<double2 *>(Q), factor, v, o);
  else
    resident_unpack_kernel<false><<<grid, 256, 0, s>>>(
        static_cast<const double *>(Rp), static_cast<const double *>(Rm),
        static_cast<double *>(R2), static_cast<double *>(Q), factor, v, o);
  CC4S_HIP(hipGetLastError());
}

void ladder_vertex_pairs(const void *slab, void *Vp, void *Vm, int64_t v, int64_t cx,
                         int64_t Ny, double *maxima, hipStream_t s) {
  const int64_t Kp = v * (v + 1) / 2, Km = v * (v - 1) / 2;
  const int64_t nb = (v + kT - 1) / kT;
  if (maxima) CC4S_HIP(hipMemsetAsync(maxima, 0, 2 * kLadderMaxima * sizeof(double), s));
  CC4S_ASSERT(cx * Ny < 65536, "paired ladder: slab chunk out of range");
  const dim3 grid(static_cast<unsigned>(nb * (nb + 1) / 2), static_cast<unsigned>(cx * Ny));
  vertex_pairs_kernel<<<grid, 256, 0, s>>>(static_cast<const double2 *>(slab),
                                           static_cast<double2 *>(Vp),
                                           static_cast<double2 *>(Vm), v, cx, Kp, Km,
                                           reinterpret_cast<unsigned long long *>(maxima));
  CC4S_HIP(hipGetLastError());
}

void ladder_unpack_pairs(const void *Rp, const void *Rm, void *R, int64_t nxy, int64_t o,
                         hipStream_t s) {
  CC4S_ASSERT(o * o < 65536, "paired ladder: No out of range");
  const dim3 grid(static_cast<unsigned>((nxy + 255) / 256), static_cast<unsigned>(o * o));
  unpack_pairs_kernel<<<grid, 256, 0, s>>>(static_cast<const double2 *>(Rp),
                                           static_cast<const double2 *>(Rm),
                                           static_cast<double2 *>(R), nxy, o);
  CC4S_HIP(hipGetLastError());
}

}  // namespace cc4s_amd
