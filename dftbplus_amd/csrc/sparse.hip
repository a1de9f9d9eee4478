// Sparse (atom-pair block) kernels of the SCC-DFTB path:
//  * Slater-Koster H0/S assembly over the neighbour blocks (nonscc.F90 buildH0/buildS):
//    8-point Neville interpolation on the equidistant grid, 5th-order tail to zero over the
//    last bohr (slakoeqgrid.F90:183-244), s/p rotation to the bond direction (sk.F90:35-289);
//  * sparse -> dense unpack (both triangles written, periodic images folded) and the dense ->
//    sparse pack of the lower triangle (sparse2dense.F90:266-321, 1024-1097);
//  * H = H0 + 1/2 S (V_mu + V_nu) (shift.F90:132-229), Mulliken charges and the non-SCC energy
//    (populations.F90:120-193);
//  * the pair part of the forces 2 sum(rho dH0 - W dS + rho (V_mu+V_nu)/2 dS)
//    (forces.F90:548-672) with finite-difference (nonscc.F90:428-484) or analytic SK derivatives.
//
// Orbital order within an atom: s, p_y, p_z, p_x. Species carry at most two shells with l <= 1,
// i.e. at most 4 orbitals per atom.
#include "common.h"
#include "gamma_dev.h"
#include "sparse.h"

#include <cmath>

namespace dftbhip {

constexpr double kDistFudge = 1.0;
constexpr double kDeltaR = 1.0e-5;

// a[k], k variable: a chain of selects keeps the array in registers
template <int N>
__device__ __forceinline__ double pick(const double (&a)[N], int n, int k) {
  double v = a[0];
#pragma unroll
  for (int j = 1; j < N; ++j) {
    const double x = a[j];
    v = j < n && j == k ? x : v;
  }
  return v;
}

// Neville interpolation as polyInterU2 (interpolation.F90:182-239) on 8 uniform points
// xa_i = (i0 + i) * dx, values y_i = tab[(i0 - 1 + i) * nint + col]. kMid: xx lies in the fourth
// interval, as it does away from the ends of a table: the path through the tableau is then known
// at compile time. Every rounding is written out (no contraction beyond the fma's here): past the
// end of a table a second difference over 1e-5 divides by 1e-10, so that an ulp of a value is
// 1e-11 in H0 and S there, whose last bits would otherwise change with the compiler's choice of
// contractions, from kernel to kernel (and did: 8e-12, which a tail far from convergence made
// 1e-4 of its charges).
template <bool kDeriv, bool kMid>
__device__ __forceinline__ double neville8(const double* tab, int nint, int col, int i0, double dx,
                                           double xx, int icl, double* dydx) {
#pragma clang fp contract(off)
  double x[8], cc[8], dd[8], cp[8], dp[8], r2[8];   // x: xa_i - xx
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    x[i] = fma((double)(i0 + i), dx, -xx);
    cc[i] = dd[i] = tab[(long)(i0 - 1 + i) * nint + col];
    cp[i] = dp[i] = 0.0;
  }
  const double x0 = (double)i0 * dx;
  double delta[7];
#pragma unroll
  for (int i = 0; i < 7; ++i) {
    const double h = i < 2 ? fma((double)(i0 + i + 1), dx, -x0) : (double)(i0 + i + 1) * dx - x0;
    delta[i] = 1.0 / h;
  }
  if (kMid) icl = 4;
  double yy = pick(cc, 8, icl - 1);
  double yp = 0.0;
  icl -= 1;
#pragma unroll
  for (int mm = 1; mm < 8; ++mm) {
#pragma unroll
    for (int ii = 0; ii < 8 - mm; ++ii) {
      const double diff = mm == 2 ? fma(r2[ii], x[ii + 1], -cc[ii + 1]) : dd[ii] - cc[ii + 1];
      r2[ii] = diff * delta[mm - 1];
      if (kDeriv) {
        const double r2p = (dp[ii] - cp[ii + 1]) * delta[mm - 1];
        // derivative of c = (x_i - x) r2 and d = (x_{i+m} - x) r2
        cp[ii] = fma(x[ii], r2p, -r2[ii]);
        dp[ii] = fma(x[ii + mm], r2p, -r2[ii]);
      }
      cc[ii] = x[ii] * r2[ii];
      dd[ii] = x[ii + mm] * r2[ii];
    }
    const bool up = 2 * icl < 8 - mm;
    if (!up) icl -= 1;
    yy += up ? pick(cc, 8 - mm, icl) : pick(dd, 8 - mm, icl);
    if (kDeriv) yp += up ? pick(cp, 8 - mm, icl) : pick(dp, 8 - mm, icl);
  }
  if (kDeriv) *dydx = yp;
  return yy;
}

// the interval of xx among the points from i0 on, 1 .. 8
__device__ __forceinline__ int neville_interval(int i0, double dx, double xx) {
#pragma clang fp contract(off)
  const double x0 = (double)i0 * dx;
  const int icl =
      (int)ceil(fma(-(double)i0, dx, xx) * (1.0 / fma((double)(i0 + 1), dx, -x0)));
  return min(max(icl, 1), 8);
}

// SK integral c (and optionally its radial derivative) at distance r
template <bool kDeriv>
__device__ __forceinline__ double sk_integral(const double* tab, int nrows, int nint, int c,
                                              double dx, double r, double* d) {
  const double rmax = fma((double)nrows, dx, kDistFudge);
  const int ind = (int)floor(r / dx);
  if (kDeriv) *d = 0.0;
  if (r >= rmax) return 0.0;
  if (ind < nrows) {
    int ilast = min(nrows, ind + 4);
    ilast = max(ilast, 8);
    const int icl = neville_interval(ilast - 7, dx, r);
    return icl == 4 ? neville8<kDeriv, true>(tab, nint, c, ilast - 7, dx, r, icl, d)
                    : neville8<kDeriv, false>(tab, nint, c, ilast - 7, dx, r, icl, d);
  }
  const int i0 = nrows - 7;
  const double dr = r - rmax;
  double y[2];
#pragma unroll 1
  for (int q = 0; q < 2; ++q) {
    const double x = fma((double)nrows, dx, q == 0 ? -kDeltaR : kDeltaR);
    const double v =
        neville8<false, false>(tab, nint, c, i0, dx, x, neville_interval(i0, dx, x), nullptr);
    if (q == 0) y[0] = v;
    else y[1] = v;
  }
  const double y0 = y[0], y2 = y[1];
  const double y1 = tab[(long)(nrows - 1) * nint + c];
  const double y1p = (y2 - y0) / (2.0 * kDeltaR);
  const double y1pp = (y2 + y0 - 2.0 * y1) / (kDeltaR * kDeltaR);
  // poly5ToZero (interpolation.F90:31-67) with dx = -distFudge
  const double ddx = -kDistFudge;
  const double dx1 = y1p * ddx, dx2 = y1pp * ddx * ddx;
  const double a3 = 10.0 * y1 - 4.0 * dx1 + 0.5 * dx2;
  const double a4 = -15.0 * y1 + 7.0 * dx1 - 1.0 * dx2;
  const double a5 = 6.0 * y1 - 3.0 * dx1 + 0.5 * dx2;
  const double xr = dr * (-1.0 / kDistFudge);
  if (kDeriv) {
    const double dpoly = ((5.0 * a5 * xr + 4.0 * a4) * xr + 3.0 * a3) * xr * xr;
    *d = dpoly * (-1.0 / kDistFudge);
  }
  return ((a5 * xr + a4) * xr + a3) * xr * xr * xr;
}

// An SK block is worked out by kBlkLanes lanes: lane q interpolates integral q & 7 of H (lanes 0
// to 7) or S (8 to 15), the lanes read what they need of each other's integrals, and lane
// e = r + c n2 forms element (r, c) of the column-major n2 x n1 block. The element's place:
struct SkElem {
  int l1, l2, p, q, ind;   // shells' momenta, orbitals within them (row, column), first integral
};

__device__ __forceinline__ SkElem sk_elem(const SpeciesDev& s1, const SpeciesDev& s2, int r,
                                          int c) {
  SkElem x{0, 0, 0, 0, 0};
  int ind = 0, icol = 0;
  for (int a = 0; a < s1.nshell; ++a) {
    const int l1 = s1.ang[a];
    int irow = 0;
    for (int b = 0; b < s2.nshell; ++b) {
      const int l2 = s2.ang[b];
      if (r >= irow && r < irow + 2 * l2 + 1 && c >= icol && c < icol + 2 * l1 + 1)
        x = {l1, l2, r - irow, c - icol, ind};
      ind += min(l1, l2) + 1;
      irow += 2 * l2 + 1;
    }
    icol += 2 * l1 + 1;
  }
  return x;
}

// cartesian index of orbital p of a p shell (order y, z, x)
__device__ __forceinline__ int p_cart(int p) { return p == 0 ? 1 : (p == 1 ? 2 : 0); }
__device__ __forceinline__ double comp(const double u[3], int c) {
  return c == 0 ? u[0] : (c == 1 ? u[1] : u[2]);
}

// Element of the rotated block for the bond unit vector u, v0 and v1 its integrals
__device__ __forceinline__ double sk_value(const SkElem& x, const double u[3], double v0,
                                           double v1) {
  if (x.l1 == 0 && x.l2 == 0) return v0;
  if (x.l1 + x.l2 == 1) {   // (-1)^(l1+l2) transpose for p on atom 1
    const double sg = x.l1 == 0 ? 1.0 : -1.0;
    return sg * comp(u, p_cart(x.l1 == 0 ? x.p : x.q)) * v0;
  }
  return (v0 - v1) * comp(u, p_cart(x.p)) * comp(u, p_cart(x.q)) + (x.p == x.q ? v1 : 0.0);
}

// its derivative w.r.t. component c of the bond vector; d0, d1: radial derivatives
__device__ __forceinline__ double sk_slope(const SkElem& x, const double u[3], double r, int c,
                                           double v0, double v1, double d0, double d1) {
  const double uc = comp(u, c);
  if (x.l1 == 0 && x.l2 == 0) return d0 * uc;
  const int pc = p_cart(x.l1 + x.l2 == 1 && x.l1 != 0 ? x.q : x.p), qc = p_cart(x.q);
  const double up = comp(u, pc), dup = ((pc == c ? 1.0 : 0.0) - up * uc) / r;
  if (x.l1 + x.l2 == 1) {
    const double sg = x.l1 == 0 ? 1.0 : -1.0;
    return sg * (dup * v0 + up * uc * d0);
  }
  const double uq = comp(u, qc), duq = ((qc == c ? 1.0 : 0.0) - uq * uc) / r;
  return (d0 - d1) * uc * up * uq + (x.p == x.q ? d1 * uc : 0.0) +
         (v0 - v1) * (dup * uq + up * duq);
}

// The species pair's tables, and lane q's integral for the bond vector vec (u, r: its direction
// and length)
struct SkPair {
  const double* tab;
  int nint, c;
};
__device__ __forceinline__ SkPair sk_pair(const SkDev& sk, int sp1, int sp2, int q) {
  const int pair = sp1 * sk.nsp + sp2;
  return {(q < 8 ? sk.htab : sk.stab) + sk.tabOff[pair], sk.nint[pair], q & 7};
}
template <bool kDeriv>
__device__ __forceinline__ double sk_lane(const SkDev& sk, const SkPair& pr, const double vec[3],
                                          double u[3], double* r, double* d) {
  *r = sqrt(vec[0] * vec[0] + vec[1] * vec[1] + vec[2] * vec[2]);
  for (int c = 0; c < 3; ++c) u[c] = vec[c] / *r;
  if (kDeriv) *d = 0.0;
  if (pr.c >= pr.nint) return 0.0;
  return sk_integral<kDeriv>(pr.tab, sk.nrows, pr.nint, pr.c, sk.dist, *r, d);
}

constexpr int kBlkLanes = 16;

// H0 and S blocks. Bound by the arithmetic of one interpolation per lane: 102 us for the blocks
// of 1000 molecules, 114 us for 2744 atoms (760 and 903 us with a thread per block, its arrays in
// scratch memory).
__global__ __launch_bounds__(256) void build_h0s_kernel(SkDev sk, PairsDev pr, const double* coords, double* h0,
                                 double* s) {
  const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const int k = (int)(t / kBlkLanes), e = (int)(t % kBlkLanes);
  if (k >= pr.nblk) return;   // whole groups of lanes
  const int a1 = pr.at1[k], i2 = pr.img2[k], a2 = pr.at2[k];
  const int sp1 = pr.species[a1], sp2 = pr.species[a2];
  const SpeciesDev& S1 = sk.sp[sp1];
  const SpeciesDev& S2 = sk.sp[sp2];
  const int n1 = S1.norb, n2 = S2.norb;
  const int r = e % n2, c = e / n2;
  const long i = pr.start[k] + e;
  if (i2 == a1) {
    if (e < n1 * n2) {
      h0[i] = (r == c) ? S1.onsite[c] : 0.0;
      s[i] = (r == c) ? 1.0 : 0.0;
    }
    return;
  }
  double vec[3], u[3], len;
  for (int q = 0; q < 3; ++q) vec[q] = coords[3 * (long)i2 + q] - coords[3 * (long)a1 + q];
  const double v = sk_lane<false>(sk, sk_pair(sk, sp1, sp2, e), vec, u, &len, nullptr);
  const SkElem x = sk_elem(S1, S2, r, c);
  const double h0v = __shfl(v, x.ind, kBlkLanes), h1v = __shfl(v, x.ind + 1, kBlkLanes);
  const double s0v = __shfl(v, x.ind + 8, kBlkLanes),
               s1v = __shfl(v, (x.ind + 9) & 15, kBlkLanes);
  if (e >= n1 * n2) return;
  h0[i] = sk_value(x, u, h0v, h1v);
  s[i] = sk_value(x, u, s0v, s1v);
}

// The per-iteration sparse kernels below give each SK block kBlkLanes lanes too, lane e holding
// element e (lanes past n1 n2 idle): the blocks of a wave are consecutive in the sparse arrays,
// so their loads and stores are contiguous.

template <typename T>
__global__ void pack_kernel(PairsDev pr, const int* norbAtom, const long* iAtomStart,
                            const T* dense, long ld, double* x) {
  const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const int k = (int)(t / kBlkLanes), e = (int)(t % kBlkLanes);
  if (k >= pr.nblk) return;
  const int a1 = pr.at1[k], a2 = pr.at2[k];
  const int n1 = norbAtom[a1], n2 = norbAtom[a2];
  if (e >= n1 * n2) return;
  const int r = e % n2, c = e / n2;
  const long o1 = iAtomStart[a1], o2 = iAtomStart[a2];
  long rr = r, cc = c;
  if (a1 == a2 && r < c) {   // on-site block symmetrised from its lower triangle
    rr = c;
    cc = r;
  }
  x[pr.start[k] + e] = (double)dense[(o2 + rr) + (o1 + cc) * ld];
}

// phase factor exp(i 2 pi kf.T) of block k; at a time-reversal-invariant point (m = 2 kf
// integral) it is (-1)^(m.T), taken exactly from the parity
__device__ inline void block_phase(const double* blkT, int k, double kx, double ky, double kz,
                                   int real2k, int m0, int m1, int m2, double& sn, double& cs) {
  if (real2k) {
    const long par = llround(m0 * blkT[3 * k] + m1 * blkT[3 * k + 1] + m2 * blkT[3 * k + 2]);
    cs = (par & 1) ? -1.0 : 1.0;
    sn = 0.0;
  } else {
    sincos(2.0 * M_PI * (kx * blkT[3 * k] + ky * blkT[3 * k + 1] + kz * blkT[3 * k + 2]), &sn,
           &cs);
  }
}

// Complex matrix at the k-point kf (fractional) into its real 2n x 2n embedding
// [[Re, -Im], [Im, Re]]: blocks times exp(i 2 pi kf.T) at (atom2 rows, atom1 columns) and the
// Hermitian counterpart; on-site blocks contribute their lower triangle with a real diagonal
// ('L' storage of unpackHS_cmplx_kpts, sparse2dense.F90:185-262). At a time-reversal-invariant
// point (real2k) the matrix is real: n x n, both triangles. The dense array is zeroed
// beforehand.
__global__ void unpack_kpt_kernel(PairsDev pr, const int* norbAtom, const long* iAtomStart,
                                  const double* blkT, double kx, double ky, double kz,
                                  int real2k, int m0, int m1, int m2, const double* x,
                                  double* dense, long ld, long n) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= pr.nblk) return;
  const int a1 = pr.at1[k], a2 = pr.at2[k];
  const int n1 = norbAtom[a1], n2 = norbAtom[a2];
  const long o1 = iAtomStart[a1], o2 = iAtomStart[a2];
  const long st = pr.start[k];
  double sn, cs;
  block_phase(blkT, k, kx, ky, kz, real2k, m0, m1, m2, sn, cs);
  for (int c = 0; c < n1; ++c)
    for (int r = 0; r < n2; ++r) {
      if (a1 == a2 && r < c) continue;
      const double v = x[st + r + c * n2];
      const double re = v * cs, im = v * sn;
      const long i = o2 + r, j = o1 + c;
      if (real2k) {
        atomicAdd(&dense[i + j * ld], re);
        if (i != j) atomicAdd(&dense[j + i * ld], re);
        continue;
      }
      atomicAdd(&dense[i + j * ld], re);
      atomicAdd(&dense[(n + i) + (n + j) * ld], re);
      if (i == j) continue;
      atomicAdd(&dense[(n + i) + j * ld], im);
      atomicAdd(&dense[i + (n + j) * ld], -im);
      atomicAdd(&dense[j + i * ld], re);
      atomicAdd(&dense[(n + j) + (n + i) * ld], re);
      atomicAdd(&dense[(n + j) + i * ld], -im);
      atomicAdd(&dense[j + (n + i) * ld], im);
    }
}

// x += w Re(exp(-i 2 pi kf.T) P) per block, P = TL + i BL read from the lower triangle of the
// embedded 2n x 2n matrix; on-site blocks completed from their lower triangle by conjugation
// (packHS_cmplx_kpts, sparse2dense.F90:820-918)
__global__ void pack_kpt_kernel(PairsDev pr, const int* norbAtom, const long* iAtomStart,
                                const double* blkT, double kx, double ky, double kz, int real2k,
                                int m0, int m1, int m2, double w, const double* dense, long ld,
                                long n, double* x) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= pr.nblk) return;
  const int a1 = pr.at1[k], a2 = pr.at2[k];
  const int n1 = norbAtom[a1], n2 = norbAtom[a2];
  const long o1 = iAtomStart[a1], o2 = iAtomStart[a2];
  const long st = pr.start[k];
  double sn, cs;
  block_phase(blkT, k, kx, ky, kz, real2k, m0, m1, m2, sn, cs);
  for (int c = 0; c < n1; ++c)
    for (int r = 0; r < n2; ++r) {
      double re, im = 0.0;
      if (a1 == a2 && r < c) {
        const long i = o2 + c, j = o1 + r;
        re = dense[i + j * ld];
        if (!real2k) im = -dense[(n + i) + j * ld];
      } else {
        const long i = o2 + r, j = o1 + c;
        re = dense[i + j * ld];
        if (!real2k) im = dense[(n + i) + j * ld];
      }
      x[st + r + c * n2] += w * (re * cs + im * sn);
    }
}

__global__ void shift_kernel(PairsDev pr, const int* norbAtom, const long* iAtomStart,
                             const double* h0, const double* s, const double* vorb, double* h) {
  const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const int k = (int)(t / kBlkLanes), e = (int)(t % kBlkLanes);
  if (k >= pr.nblk) return;
  const int a1 = pr.at1[k], a2 = pr.at2[k];
  const int n1 = norbAtom[a1], n2 = norbAtom[a2];
  if (e >= n1 * n2) return;
  const int r = e % n2, c = e / n2;
  const long o1 = iAtomStart[a1], o2 = iAtomStart[a2];
  const long i = pr.start[k] + e;
  h[i] = h0[i] + 0.5 * s[i] * (vorb[o2 + r] + vorb[o1 + c]);
}

// Pair forces: gradient contribution of every off-site block. mode 0: central finite
// differences with step delta on the bond vector (the reference default); mode 1: analytic
// derivative of the interpolated and rotated blocks (the adjoint of the assembly).
// Lanes as above: six interpolations per lane in mode 0, one in mode 1, the element's
// contribution summed over the block's lanes. A thread per pair (60 interpolations one after the
// other, blocks in scratch memory) took 3.9 ms for 1000 molecules and 4.6 ms for 2744 atoms; now
// 0.45 and 0.50 ms.
template <int kMode>
__global__ __launch_bounds__(256) void pair_force_kernel(SkDev sk, PairsDev pr, const int* norbAtom,
                                  const long* iAtomStart, const double* coords, const double* rho,
                                  const double* erho, const double* vorb, double delta,
                                  double* grad) {
  const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const int k = (int)(t / kBlkLanes), e = (int)(t % kBlkLanes);
  if (k >= pr.nblk) return;   // whole groups of lanes, here and below
  const int a1 = pr.at1[k], i2 = pr.img2[k], a2 = pr.at2[k];
  if (a1 == a2) return;
  const int sp1 = pr.species[a1], sp2 = pr.species[a2];
  const int n1 = norbAtom[a1], n2 = norbAtom[a2];
  const int r = e % n2, cc = e / n2;
  const bool in = e < n1 * n2;
  double wH = 0.0, wS = 0.0, wV = 0.0;   // rho, W and rho (V_mu + V_nu) / 2 of the element
  if (in) {
    const long i = pr.start[k] + e;
    wH = rho[i];
    wS = erho[i];
    wV = wH * (0.5 * (vorb[iAtomStart[a2] + r] + vorb[iAtomStart[a1] + cc]));
  }
  double vec[3];
  for (int c = 0; c < 3; ++c) vec[c] = coords[3 * (long)i2 + c] - coords[3 * (long)a1 + c];
  const SkPair tabs = sk_pair(sk, sp1, sp2, e);
  const SkElem x = sk_elem(sk.sp[sp1], sk.sp[sp2], r, cc);
  const int j0 = x.ind, j1 = x.ind + 1, j2 = x.ind + 8, j3 = (x.ind + 9) & 15;
  double g[3] = {0, 0, 0};
  if (kMode == 0) {
#pragma unroll 1
    for (int c = 0; c < 3; ++c) {
      double hp = 0.0, sp = 0.0, hm = 0.0, sm = 0.0;
#pragma unroll 1
      for (int side = 0; side < 2; ++side) {
        double w[3], u[3], len;
        for (int q = 0; q < 3; ++q)
          w[q] = vec[q] + (q == c ? (side == 0 ? delta : -delta) : 0.0);
        const double v = sk_lane<false>(sk, tabs, w, u, &len, nullptr);
        hp = hm;
        sp = sm;
        hm = sk_value(x, u, __shfl(v, j0, kBlkLanes), __shfl(v, j1, kBlkLanes));
        sm = sk_value(x, u, __shfl(v, j2, kBlkLanes), __shfl(v, j3, kBlkLanes));
      }
      const double dH = (hm - hp) / (2.0 * delta), dS = (sm - sp) / (2.0 * delta);
      const double acc = in ? wH * dH - wS * dS + wV * dS : 0.0;
      if (c == 0) g[0] = acc;
      else if (c == 1) g[1] = acc;
      else g[2] = acc;
    }
  } else {
    double u[3], len, d;
    const double v = sk_lane<true>(sk, tabs, vec, u, &len, &d);
    const double h0 = __shfl(v, j0, kBlkLanes), h1 = __shfl(v, j1, kBlkLanes);
    const double s0 = __shfl(v, j2, kBlkLanes), s1 = __shfl(v, j3, kBlkLanes);
    const double dh0 = __shfl(d, j0, kBlkLanes), dh1 = __shfl(d, j1, kBlkLanes);
    const double ds0 = __shfl(d, j2, kBlkLanes), ds1 = __shfl(d, j3, kBlkLanes);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      // derivative w.r.t. atom 1 = - d/dR
      const double dH = -sk_slope(x, u, len, c, h0, h1, dh0, dh1);
      const double dS = -sk_slope(x, u, len, c, s0, s1, ds0, ds1);
      g[c] = in ? wH * dH - wS * dS + wV * dS : 0.0;
    }
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
#pragma unroll
    for (int o = kBlkLanes / 2; o > 0; o >>= 1) g[c] += __shfl_xor(g[c], o, kBlkLanes);
    g[c] *= 2.0;
  }
  if (e < 6) {
    const double gc = comp(g, e % 3);
    atomicAdd(&grad[3 * (long)(e < 3 ? a1 : a2) + e % 3], e < 3 ? gc : -gc);
  }
}

__global__ void invr_cluster_kernel(int nat, const double* coords, double* g) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y;
  if (i >= nat) return;
  double v = 0.0;
  if (i != j) {
    const double dx = coords[3 * i] - coords[3 * j], dy = coords[3 * i + 1] - coords[3 * j + 1],
                 dz = coords[3 * i + 2] - coords[3 * j + 2];
    v = 1.0 / sqrt(dx * dx + dy * dy + dz * dz);
  }
  g[i + (long)j * nat] = v;
}

// Ewald real-space sum over translations, plus the constant -pi/(V alpha^2) and the self term.
__global__ void ewald_real_kernel(int nat, const double* coords, int ntr, const double* tr,
                                  double alpha, double maxr, double cst, double self, double* g) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y;
  if (i >= nat) return;
  const double dx = coords[3 * i] - coords[3 * j], dy = coords[3 * i + 1] - coords[3 * j + 1],
               dz = coords[3 * i + 2] - coords[3 * j + 2];
  double acc = 0.0;
  for (int t = 0; t < ntr; ++t) {
    const double x = dx - tr[3 * t], y = dy - tr[3 * t + 1], z = dz - tr[3 * t + 2];
    const double r = sqrt(x * x + y * y + z * z);
    if (r <= maxr && r > 1.0e-8) acc += erfc(alpha * r) / r;
  }
  acc += cst;
  if (i == j) acc += self;
  g[i + (long)j * nat] += acc;
}

// structure factor matrices C(i,g) = cos(G.r_i), S(i,g) = sin(G.r_i)
__global__ void strucfac_kernel(int nat, const double* coords, int ng, const double* G,
                                double* cs) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int g = blockIdx.y;
  if (i >= nat) return;
  const double ph =
      G[3 * g] * coords[3 * i] + G[3 * g + 1] * coords[3 * i + 1] + G[3 * g + 2] * coords[3 * i + 2];
  double sn, cn;
  sincos(ph, &sn, &cn);
  cs[i + (long)g * nat] = cn;
  cs[i + (long)(g + ng) * nat] = sn;
}

// gamma(jc, i) and gamma(i, jc) -= expGamma for every neighbour within its cutoff
__global__ void short_gamma_kernel(NeighDev nb, const double* coords, const double* hubbu,
                                   const double* gcut, int nsp, int nat, double* g) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nb.n) return;
  const int i = nb.at1[k], j = nb.img2[k], jc = nb.at2[k];
  const int si = nb.species[i], sj = nb.species[jc];
  const double dx = coords[3 * (long)i] - coords[3 * (long)j],
               dy = coords[3 * (long)i + 1] - coords[3 * (long)j + 1],
               dz = coords[3 * (long)i + 2] - coords[3 * (long)j + 2];
  const double r = sqrt(dx * dx + dy * dy + dz * dz);
  if (j != i && r > gcut[sj * nsp + si]) return;
  const double v = expgamma(r, hubbu[sj], hubbu[si]);
  atomicAdd(&g[jc + (long)i * nat], -v);
  if (jc != i) atomicAdd(&g[i + (long)jc * nat], -v);
}

// gradient of 1/2 dq^T gamma dq from the short-range part and (cluster) 1/R part per neighbour
__global__ void short_gamma_grad_kernel(NeighDev nb, const double* coords, const double* hubbu,
                                        const double* gcut, int nsp, const double* dq,
                                        double* grad) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nb.n) return;
  const int i = nb.at1[k], j = nb.img2[k], jc = nb.at2[k];
  if (jc == i) return;
  const int si = nb.species[i], sj = nb.species[jc];
  const double d[3] = {coords[3 * (long)i] - coords[3 * (long)j],
                       coords[3 * (long)i + 1] - coords[3 * (long)j + 1],
                       coords[3 * (long)i + 2] - coords[3 * (long)j + 2]};
  const double r = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
  if (r > gcut[sj * nsp + si]) return;
  const double f = -expgamma_prime(r, hubbu[sj], hubbu[si]) * dq[i] * dq[jc] / r;
  for (int c = 0; c < 3; ++c) {
    atomicAdd(&grad[3 * (long)i + c], f * d[c]);
    atomicAdd(&grad[3 * (long)jc + c], -f * d[c]);
  }
}

// cluster 1/R gradient: one thread per atom i, loop over j
__global__ void invr_cluster_grad_kernel(int nat, const double* coords, const double* dq,
                                         double* grad) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nat) return;
  double g[3] = {0, 0, 0};
  for (int j = 0; j < nat; ++j) {
    if (j == i) continue;
    const double d[3] = {coords[3 * i] - coords[3 * j], coords[3 * i + 1] - coords[3 * j + 1],
                         coords[3 * i + 2] - coords[3 * j + 2]};
    const double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
    const double f = -dq[i] * dq[j] / (r2 * sqrt(r2));
    for (int c = 0; c < 3; ++c) g[c] += f * d[c];
  }
  for (int c = 0; c < 3; ++c) grad[3 * i + c] += g[c];
}

// Ewald gradient: real space over translations + reciprocal from structure factors
// Ewald gradient of atom i (one 256-thread workgroup per atom): real-space sum over all atoms
// and lattice translations within maxr, reciprocal sum over the G vectors with the structure
// factors C_G = sum_j dq_j cos(G r_j), S_G = sum_j dq_j sin(G r_j) (CS = [C; S])
__global__ __launch_bounds__(256) void ewald_grad_kernel(int nat, const double* coords, int ntr,
                                                         const double* tr, double alpha,
                                                         double maxr, int ng, const double* G,
                                                         const double* w, const double* CS,
                                                         const double* dq, double* grad) {
  __shared__ double red[3][4];
  const int i = blockIdx.x;
  if (i >= nat) return;
  const int tid = threadIdx.x;
  const double xi = coords[3 * i], yi = coords[3 * i + 1], zi = coords[3 * i + 2];
  const double ta = 2.0 * alpha / sqrt(M_PI);
  const double maxr2 = maxr * maxr;
  double g0 = 0.0, g1 = 0.0, g2 = 0.0;
  for (int j = tid; j < nat; j += 256) {
    const double dx = xi - coords[3 * j], dy = yi - coords[3 * j + 1], dz = zi - coords[3 * j + 2];
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
    for (int t = 0; t < ntr; ++t) {
      const double x = dx - tr[3 * t], y = dy - tr[3 * t + 1], z = dz - tr[3 * t + 2];
      const double r2 = x * x + y * y + z * z;
      if (r2 <= maxr2 && r2 > 1.0e-16) {
        const double r = sqrt(r2);
        const double dfdr = -(ta * exp(-alpha * alpha * r2) / r + erfc(alpha * r) / r2);
        const double f = dfdr / r;
        a0 += f * x;
        a1 += f * y;
        a2 += f * z;
      }
    }
    g0 += a0 * dq[j];
    g1 += a1 * dq[j];
    g2 += a2 * dq[j];
  }
  for (int q = tid; q < ng; q += 256) {
    const double ph = G[3 * q] * xi + G[3 * q + 1] * yi + G[3 * q + 2] * zi;
    double sn, cn;
    sincos(ph, &sn, &cn);
    const double fac = (sn * CS[q] - cn * CS[ng + q]) * w[q];
    g0 -= fac * G[3 * q];
    g1 -= fac * G[3 * q + 1];
    g2 -= fac * G[3 * q + 2];
  }
  for (int o = 32; o > 0; o >>= 1) {
    g0 += __shfl_down(g0, o, 64);
    g1 += __shfl_down(g1, o, 64);
    g2 += __shfl_down(g2, o, 64);
  }
  const int lane = tid & 63, wv = tid >> 6;
  if (lane == 0) {
    red[0][wv] = g0;
    red[1][wv] = g1;
    red[2][wv] = g2;
  }
  __syncthreads();
  if (tid < 3)
    grad[3 * i + tid] += dq[i] * (red[tid][0] + red[tid][1] + red[tid][2] + red[tid][3]);
}

// repulsive energy and gradient over neighbours within the repulsive cutoff
__device__ void rep_value(const RepDev& rp, double r, double* e, double* de) {
  *e = 0.0;
  *de = 0.0;
  if (r < 1.0e-2 || r >= rp.cutoff) return;
  if (r < rp.xs[0]) {
    const double ex = exp(-rp.expc[0] * r + rp.expc[1]);
    *e = ex + rp.expc[2];
    *de = -rp.expc[0] * ex;
    return;
  }
  int im = 0;
  while (im + 1 < rp.nint && rp.xs[im + 1] <= r) ++im;
  const double dr = r - rp.xs[im];
  const double* c = (im < rp.nint - 1) ? rp.coef + 4 * im : rp.last;
  const int nc = (im < rp.nint - 1) ? 4 : 6;
  double en = 0.0, dv = 0.0;
  for (int q = nc - 1; q >= 0; --q) en = en * dr + c[q];
  for (int q = nc - 1; q >= 1; --q) dv = dv * dr + q * c[q];
  *e = en;
  *de = dv;
}

__global__ void repulsive_kernel(NeighDev nb, const double* coords, const RepDev* reps, int nsp,
                                 double* eatom, double* grad) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nb.n) return;
  const int i = nb.at1[k], j = nb.img2[k], jc = nb.at2[k];
  if (j == i) return;
  const double d[3] = {coords[3 * (long)i] - coords[3 * (long)j],
                       coords[3 * (long)i + 1] - coords[3 * (long)j + 1],
                       coords[3 * (long)i + 2] - coords[3 * (long)j + 2]};
  const double r = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
  const RepDev& rp = reps[nb.species[i] * nsp + nb.species[jc]];
  if (r >= rp.cutoff) return;
  double e, de;
  rep_value(rp, r, &e, &de);
  atomicAdd(&eatom[i], 0.5 * e);
  if (jc != i) {
    atomicAdd(&eatom[jc], 0.5 * e);
    for (int c = 0; c < 3; ++c) {
      atomicAdd(&grad[3 * (long)i + c], de * d[c] / r);
      atomicAdd(&grad[3 * (long)jc + c], -de * d[c] / r);
    }
  }
}

// ------------------------------------------------------------------------------------------
// launch wrappers
// ------------------------------------------------------------------------------------------
int launch_build_h0s(hipStream_t s, const SkDev& sk, const PairsDev& pr, const double* coords,
                     double* h0, double* ov) {
  if (pr.nblk == 0) return 0;
  hipLaunchKernelGGL(build_h0s_kernel, dim3(cdiv((long)pr.nblk * kBlkLanes, 256)), dim3(256), 0, s,
                     sk, pr, coords, h0, ov);
  DH_LAUNCH_CHECK();
  return 0;
}

template <typename T>
int launch_pack(hipStream_t s, const PairsDev& pr, const int* norb, const long* iAtomStart,
                const T* dense, long ld, double* x) {
  if (pr.nblk == 0) return 0;
  hipLaunchKernelGGL((pack_kernel<T>), dim3(cdiv((long)pr.nblk * kBlkLanes, 256)),
                     dim3(256), 0, s, pr, norb,
                     iAtomStart, dense, ld, x);
  DH_LAUNCH_CHECK();
  return 0;
}

bool kpoint_is_real(const double* kf) {
  for (int q = 0; q < 3; ++q)
    if (std::fabs(2.0 * kf[q] - std::nearbyint(2.0 * kf[q])) > 1e-12) return false;
  return true;
}

int kpoint_dim(const double* kf, int n) { return kpoint_is_real(kf) ? n : 2 * n; }

int launch_unpack_kpt(hipStream_t s, const PairsDev& pr, const int* norb, const long* iAtomStart,
                      const double* blkT, const double* kf, const double* x, double* dense,
                      long ld, int n) {
  const int nd = kpoint_dim(kf, n);
  DH_CHECK(ld >= nd, "unpack_kpt: leading dimension too small");
  DH_TRY(fill2d<double>(s, dense, ld, nd, nd, 0.0));
  if (pr.nblk == 0) return 0;
  const int re = kpoint_is_real(kf) ? 1 : 0;
  hipLaunchKernelGGL(unpack_kpt_kernel, dim3(cdiv(pr.nblk, 128)), dim3(128), 0, s, pr, norb,
                     iAtomStart, blkT, kf[0], kf[1], kf[2], re, (int)std::nearbyint(2.0 * kf[0]),
                     (int)std::nearbyint(2.0 * kf[1]), (int)std::nearbyint(2.0 * kf[2]), x,
                     dense, ld, (long)n);
  DH_LAUNCH_CHECK();
  return 0;
}

int launch_pack_kpt(hipStream_t s, const PairsDev& pr, const int* norb, const long* iAtomStart,
                    const double* blkT, const double* kf, double w, const double* dense, long ld,
                    int n, double* x) {
  if (pr.nblk == 0) return 0;
  DH_CHECK(ld >= kpoint_dim(kf, n), "pack_kpt: leading dimension too small");
  const int re = kpoint_is_real(kf) ? 1 : 0;
  hipLaunchKernelGGL(pack_kpt_kernel, dim3(cdiv(pr.nblk, 128)), dim3(128), 0, s, pr, norb,
                     iAtomStart, blkT, kf[0], kf[1], kf[2], re, (int)std::nearbyint(2.0 * kf[0]),
                     (int)std::nearbyint(2.0 * kf[1]), (int)std::nearbyint(2.0 * kf[2]), w,
                     dense, ld, (long)n, x);
  DH_LAUNCH_CHECK();
  return 0;
}

int launch_shift(hipStream_t s, const PairsDev& pr, const int* norb, const long* iAtomStart,
                 const double* h0, const double* ov, const double* vorb, double* h) {
  if (pr.nblk == 0) return 0;
  hipLaunchKernelGGL(shift_kernel, dim3(cdiv((long)pr.nblk * kBlkLanes, 256)),
                     dim3(256), 0, s, pr, norb,
                     iAtomStart, h0, ov, vorb, h);
  DH_LAUNCH_CHECK();
  return 0;
}

int launch_pair_forces(hipStream_t s, const SkDev& sk, const PairsDev& pr, const int* norb,
                       const long* iAtomStart, const double* coords, const double* rho,
                       const double* erho, const double* vorb, int mode, double delta,
                       double* grad) {
  if (pr.nblk == 0) return 0;
  const dim3 grid(cdiv((long)pr.nblk * kBlkLanes, 256));
  if (mode == 0)
    hipLaunchKernelGGL(pair_force_kernel<0>, grid, dim3(256), 0, s, sk, pr, norb, iAtomStart,
                       coords, rho, erho, vorb, delta, grad);
  else
    hipLaunchKernelGGL(pair_force_kernel<1>, grid, dim3(256), 0, s, sk, pr, norb, iAtomStart,
                       coords, rho, erho, vorb, delta, grad);
  DH_LAUNCH_CHECK();
  return 0;
}

int launch_invr_cluster(hipStream_t s, int nat, const double* coords, double* g) {
  hipLaunchKernelGGL(invr_cluster_kernel, dim3(cdiv(nat, 256), nat), dim3(256), 0, s, nat, coords,
                     g);
  DH_LAUNCH_CHECK();
  return 0;
}

int launch_ewald_real(hipStream_t s, int nat, const double* coords, int ntr, const double* tr,
                      double alpha, double maxr, double cst, double self, double* g) {
  hipLaunchKernelGGL(ewald_real_kernel, dim3(cdiv(nat, 256), nat), dim3(256), 0, s, nat, coords,
                     ntr, tr, alpha, maxr, cst, self, g);
  DH_LAUNCH_CHECK();
  return 0;
}

int launch_strucfac(hipStream_t s, int nat, const double* coords, int ng, const double* G,
                    double* cs) {
  if (ng == 0) return 0;
  hipLaunchKernelGGL(strucfac_kernel, dim3(cdiv(nat, 256), ng), dim3(256), 0, s, nat, coords, ng,
                     G, cs);
  DH_LAUNCH_CHECK();
  return 0;
}

int launch_short_gamma(hipStream_t s, const NeighDev& nb, const double* coords,
                       const double* hubbu, const double* gcut, int nsp, int nat, double* g) {
  if (nb.n == 0) return 0;
  hipLaunchKernelGGL(short_gamma_kernel, dim3(cdiv(nb.n, 256)), dim3(256), 0, s, nb, coords, hubbu,
                     gcut, nsp, nat, g);
  DH_LAUNCH_CHECK();
  return 0;
}

int launch_short_gamma_grad(hipStream_t s, const NeighDev& nb, const double* coords,
                            const double* hubbu, const double* gcut, int nsp, const double* dq,
                            double* grad) {
  if (nb.n == 0) return 0;
  hipLaunchKernelGGL(short_gamma_grad_kernel, dim3(cdiv(nb.n, 256)), dim3(256), 0, s, nb, coords,
                     hubbu, gcut, nsp, dq, grad);
  DH_LAUNCH_CHECK();
  return 0;
}

int launch_gamma_grad(hipStream_t s, const NeighDev& nb, const double* coords,
                      const double* hubbu, const double* gcut, int nsp, int nat, bool periodic,
                      int ntr, const double* tr, double alpha, double maxr, int ng,
                      const double* G, const double* w, const double* CSq, const double* dq,
                      double* grad) {
  if (nb.n > 0) {
    hipLaunchKernelGGL(short_gamma_grad_kernel, dim3(cdiv(nb.n, 256)), dim3(256), 0, s, nb, coords,
                       hubbu, gcut, nsp, dq, grad);
    DH_LAUNCH_CHECK();
  }
  if (!periodic) {
    hipLaunchKernelGGL(invr_cluster_grad_kernel, dim3(cdiv(nat, 64)), dim3(64), 0, s, nat, coords,
                       dq, grad);
  } else {
    hipLaunchKernelGGL(ewald_grad_kernel, dim3(nat), dim3(256), 0, s, nat, coords, ntr, tr, alpha,
                       maxr, ng, G, w, CSq, dq, grad);
  }
  DH_LAUNCH_CHECK();
  return 0;
}

int launch_repulsive(hipStream_t s, const NeighDev& nb, const double* coords, const RepDev* reps,
                     int nsp, double* eatom, double* grad) {
  if (nb.n == 0) return 0;
  hipLaunchKernelGGL(repulsive_kernel, dim3(cdiv(nb.n, 256)), dim3(256), 0, s, nb, coords, reps,
                     nsp, eatom, grad);
  DH_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------------------------
// Block-sparse products with a transposed dense operand: YH^T = (H X)^T and YS^T = (S X)^T for
// X given as Xt = X^T (nvec x n, column-major, so the nvec coefficients of one orbital are
// contiguous). H and S are the matrices unpack builds from the sparse blocks (image blocks of one
// atom pair summed).
//  * spmm_fold_kernel: once per H and S, the row view's groups (row atom A, column atom B) become
//    dense 4 x 4 blocks of both matrices (image blocks summed with their k-point phases +-1,
//    transposed where the stored block is (B, A), zero-padded past the atoms' orbitals), 32
//    consecutive doubles per group in row order, with the column atom's first orbital beside;
//  * spmm_fold_t_kernel: a workgroup of 4 waves owns one row atom and 256 kVpl consecutive
//    vectors (kVpl per lane, 64 apart). Per group the wave reads the block's 32 values as
//    wave-uniform scalar loads from contiguous memory, the 4 coefficient rows of the column atom
//    (kVpl coalesced loads each) and does 32 kVpl FMAs; the outputs of the atom's 4 orbitals
//    for both matrices stay in registers. Workgroups are numbered so that consecutive ones of an
//    XCD (IDs congruent mod 8) walk the atoms of one vector tile, so the coefficient rows a tile
//    reads stay in that XCD's L2 while its neighbouring row atoms read them.
// ---------------------------------------------------------------------------------------------
constexpr int kXcds = 8;
static int g_spmmVpl = 1;
int set_spmm_cols(int vpl) {
  DH_CHECK(vpl == 1 || vpl == 2 || vpl == 4, "spmm: 1, 2 or 4 vectors per lane");
  g_spmmVpl = vpl;
  return 0;
}

__global__ __launch_bounds__(256) void spmm_fold_kernel(
    const int* __restrict__ gPtr, const int2* __restrict__ grp, const int2* __restrict__ entS,
    const int* __restrict__ norbAtom, const long* __restrict__ iAtomStart,
    const long* __restrict__ blkStart, const double* __restrict__ h,
    const double* __restrict__ ov, const double* __restrict__ blkT, int m0, int m1, int m2,
    double* __restrict__ fold, int* __restrict__ colOff) {
  const int A = blockIdx.x;
  const int nA = norbAtom[A];
  const int g0 = gPtr[A], g1 = gPtr[A + 1];
  for (int t = threadIdx.x; t < (g1 - g0) * 32; t += blockDim.x) {
    const int g = g0 + (t >> 5), el = t & 31;
    const int mat = el >> 4, r = (el >> 2) & 3, c = el & 3;
    const int2 gr = grp[g];
    const int B = entS[gr.x].y, nB = norbAtom[B];
    const double* __restrict__ src = mat ? ov : h;
    double v = 0.0;
    if (r < nA && c < nB) {
      for (int e = gr.x; e < gr.y; ++e) {
        const int k = entS[e].x >> 1, tr = entS[e].x & 1;
        const long q = blkStart[k] + (tr ? (c + (long)r * nB) : (r + (long)c * nA));
        double x = src[q];
        if (blkT) {
          const long par =
              llround(m0 * blkT[3 * k] + m1 * blkT[3 * k + 1] + m2 * blkT[3 * k + 2]);
          if (par & 1) x = -x;
        }
        v += x;
      }
    }
    fold[(long)g * 32 + el] = v;
    if (el == 0) colOff[g] = (int)iAtomStart[B];
  }
}

template <int kVpl>
__global__ __launch_bounds__(256) void spmm_fold_t_kernel(
    int nat, int ntile, int n, const int* __restrict__ gPtr, const int* __restrict__ colOff,
    const double* __restrict__ fold, const int* __restrict__ norbAtom,
    const long* __restrict__ iAtomStart, const double* __restrict__ Xt, long ldx, int nvec,
    double* __restrict__ yh, double* __restrict__ ys, long ldy) {
  const long w = blockIdx.x;
  const int xcd = (int)(w % kXcds);
  const long l = w / kXcds;
  const int tile = xcd + kXcds * (int)(l / nat);
  const int A = (int)(l % nat);
  if (tile >= ntile) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int jb = tile * 256 * kVpl + wave * 64 * kVpl + lane;
  const double* __restrict__ xj[kVpl];
#pragma unroll
  for (int v = 0; v < kVpl; ++v) xj[v] = Xt + min(jb + 64 * v, nvec - 1);
  double ah[kVpl][4], as[kVpl][4];
#pragma unroll
  for (int v = 0; v < kVpl; ++v)
#pragma unroll
    for (int r = 0; r < 4; ++r) ah[v][r] = as[v][r] = 0.0;
  const int g0 = gPtr[A], g1 = gPtr[A + 1];
  // the coefficient rows of the next group are loaded while the current one is multiplied
  // (rows past the column atom's orbitals meet zero block columns; clamped to stay inside Xt)
  double xn[kVpl][4];
  auto load_x = [&](int g) {
    const int oB = colOff[g];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const long row = min(oB + c, n - 1);
#pragma unroll
      for (int v = 0; v < kVpl; ++v) xn[v][c] = xj[v][row * ldx];
    }
  };
  if (g0 < g1) load_x(g0);
  for (int g = g0; g < g1; ++g) {
    double xv[kVpl][4];
#pragma unroll
    for (int v = 0; v < kVpl; ++v)
#pragma unroll
      for (int c = 0; c < 4; ++c) xv[v][c] = xn[v][c];
    if (g + 1 < g1) load_x(g + 1);
    const double* __restrict__ b = fold + (long)g * 32;
    double bh[16], bs[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      bh[q] = b[q];
      bs[q] = b[16 + q];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int v = 0; v < kVpl; ++v) {
          ah[v][r] = fma(bh[r * 4 + c], xv[v][c], ah[v][r]);
          as[v][r] = fma(bs[r * 4 + c], xv[v][c], as[v][r]);
        }
  }
  const int nA = norbAtom[A];
  const long oA = iAtomStart[A];
#pragma unroll
  for (int v = 0; v < kVpl; ++v) {
    const int j = jb + 64 * v;
    if (j >= nvec) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (r >= nA) break;
      yh[j + (oA + r) * ldy] = ah[v][r];
      ys[j + (oA + r) * ldy] = as[v][r];
    }
  }
}

int launch_spmm_fold(hipStream_t s, const RowBlocksDev& rb, const int* norb,
                     const long* iAtomStart, const long* blkStart, const double* h,
                     const double* ov, const double* blkT, const double* kf, double* fold,
                     int* colOff) {
  if (rb.nat == 0) return 0;
  int m[3] = {0, 0, 0};
  if (blkT) {
    DH_CHECK(kf && kpoint_is_real(kf), "spmm: the k-point is not time-reversal invariant");
    for (int q = 0; q < 3; ++q) m[q] = (int)std::nearbyint(2.0 * kf[q]);
  }
  hipLaunchKernelGGL(spmm_fold_kernel, dim3(rb.nat), dim3(256), 0, s, rb.gPtr, rb.grp, rb.entS,
                     norb, iAtomStart, blkStart, h, ov, blkT, m[0], m[1], m[2], fold, colOff);
  DH_LAUNCH_CHECK();
  return 0;
}

int launch_spmm_hs_t(hipStream_t s, const RowBlocksDev& rb, const int* norb,
                     const long* iAtomStart, int n, const double* fold, const int* colOff,
                     const double* Xt, long ldx, int nvec, double* yh, double* ys, long ldy) {
  if (rb.nat == 0 || nvec <= 0) return 0;
  const int vpl = g_spmmVpl;
  const int ntile = (int)cdiv(nvec, 256 * vpl);
  const long tilesPad = (long)cdiv(ntile, kXcds) * kXcds;
  const long nwg = tilesPad * rb.nat;
  DH_CHECK(nwg < (1L << 31), "spmm: grid too large");
#define DH_SPMM(V_)                                                                           \
  hipLaunchKernelGGL(spmm_fold_t_kernel<V_>, dim3((unsigned)nwg), dim3(256), 0, s, rb.nat, ntile, \
                     n, rb.gPtr, colOff, fold, norb, iAtomStart, Xt, ldx, nvec, yh, ys, ldy)
  if (vpl == 1) DH_SPMM(1);
  else if (vpl == 2) DH_SPMM(2);
  else DH_SPMM(4);
#undef DH_SPMM
  DH_LAUNCH_CHECK();
  return 0;
}

// Sparse -> dense from the row view (unpackHS_real, sparse2dense.F90:266-321, both triangles):
// one wave per row atom, a lane per group of entries with one column atom (the image blocks of
// the pair, summed in registers), every element of the atom pair's block written once.
template <typename T>
__global__ __launch_bounds__(256) void unpack_rows_kernel(
    RowBlocksDev rb, const int* __restrict__ norbAtom, const long* __restrict__ iAtomStart,
    const long* __restrict__ blkStart, const double* __restrict__ x, T* __restrict__ dense,
    long ld) {
  const int A = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (A >= rb.nat) return;
  const int nA = norbAtom[A];
  const long oA = iAtomStart[A];
  const int g1 = rb.gPtr[A + 1];
  for (int g = rb.gPtr[A] + lane; g < g1; g += 64) {
    const int2 gr = rb.grp[g];
    const int B = rb.entS[gr.x].y;
    const int nB = norbAtom[B];
    const long oB = iAtomStart[B];
    double v[4][4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c) v[r][c] = 0.0;
    for (int p = gr.x; p < gr.y; ++p) {
      const int2 en = rb.entS[p];
      const int k = en.x >> 1, tr = en.x & 1;
      const long st = blkStart[k];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (r >= nA) break;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          if (c >= nB) break;
          v[r][c] += x[st + (tr ? (c + (long)r * nB) : (r + (long)c * nA))];
        }
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (c >= nB) break;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (r >= nA) break;
        dense[(oA + r) + (oB + c) * ld] = (T)v[r][c];
      }
    }
  }
}

template <typename T>
int launch_unpack_rows(hipStream_t s, const RowBlocksDev& rb, const int* norb,
                       const long* iAtomStart, const long* blkStart, const double* x, T* dense,
                       long ld, int n) {
  DH_TRY(fill2d<T>(s, dense, ld, n, n, T(0)));
  if (rb.nat == 0) return 0;
  hipLaunchKernelGGL((unpack_rows_kernel<T>), dim3(cdiv(rb.nat, 4)), dim3(256), 0, s, rb, norb,
                     iAtomStart, blkStart, x, dense, ld);
  DH_LAUNCH_CHECK();
  return 0;
}
template int launch_unpack_rows<double>(hipStream_t, const RowBlocksDev&, const int*,
                                        const long*, const long*, const double*, double*, long,
                                        int);
template int launch_unpack_rows<float>(hipStream_t, const RowBlocksDev&, const int*, const long*,
                                       const long*, const double*, float*, long, int);

// Mulliken populations and band-structure energy per orbital (mullikenPerOrbital,
// populations.F90:120-193: the block of a pair (atom1, atom2) adds its column sums to atom1's
// orbitals and, when atom1 != atom2 as central atoms, its row sums to atom2's) from the row view:
// one wave per row atom, a lane per entry, the per-orbital partial sums combined by an xor
// butterfly, so every orbital is written once, without atomics, and the result does not depend
// on the order in which the hardware runs the waves. In the row view an entry (k, t, B) of row
// atom A holds element (r of A, c of B) at r + c nA (t = 0, pair (B, A)) or c + r nB (t = 1,
// pair (A, B)); a pair of an atom with itself or its image (t = 0, B = A) adds its column sums,
// i.e. element (c, r) of the stored block.
__global__ __launch_bounds__(256) void mulliken_rows_kernel(
    RowBlocksDev rb, const int* __restrict__ norbAtom, const long* __restrict__ iAtomStart,
    const long* __restrict__ blkStart, const double* __restrict__ ov,
    const double* __restrict__ h0, const double* __restrict__ rho, double* __restrict__ qorb,
    double* __restrict__ eorb) {
  const int A = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (A >= rb.nat) return;
  const int nA = norbAtom[A];
  double q[4] = {0.0, 0.0, 0.0, 0.0}, e[4] = {0.0, 0.0, 0.0, 0.0};
  const int p1 = rb.rowPtr[A + 1];
  for (int p = rb.rowPtr[A] + lane; p < p1; p += 64) {
    const int2 en = rb.ent[p];
    const int k = en.x >> 1, tr = en.x & 1, B = en.y;
    const int nB = norbAtom[B];
    const long st = blkStart[k];
    const bool self = !tr && B == A;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (r >= nA) break;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (c >= nB) break;
        const long idx = st + (tr ? (c + (long)r * nB) : (self ? (c + (long)r * nA)
                                                              : (r + (long)c * nA)));
        const double d = rho[idx];
        q[r] = fma(ov[idx], d, q[r]);
        if (h0) e[r] = fma(h0[idx], d, e[r]);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    for (int o = 32; o > 0; o >>= 1) {
      q[r] += __shfl_xor(q[r], o, 64);
      e[r] += __shfl_xor(e[r], o, 64);
    }
  if (lane == 0) {
    const long oA = iAtomStart[A];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (r >= nA) break;
      qorb[oA + r] = q[r];
      if (eorb) eorb[oA + r] = e[r];
    }
  }
}

int launch_mulliken_rows(hipStream_t s, const RowBlocksDev& rb, const int* norb,
                         const long* iAtomStart, const long* blkStart, const double* ov,
                         const double* h0, const double* rho, double* qorb, double* eorb) {
  if (rb.nat == 0) return 0;
  hipLaunchKernelGGL(mulliken_rows_kernel, dim3(cdiv(rb.nat, 4)), dim3(256), 0, s, rb, norb,
                     iAtomStart, blkStart, ov, h0, rho, qorb, eorb);
  DH_LAUNCH_CHECK();
  return 0;
}

template int launch_pack<double>(hipStream_t, const PairsDev&, const int*, const long*,
                                 const double*, long, double*);
template int launch_pack<float>(hipStream_t, const PairsDev&, const int*, const long*,
                                const float*, long, double*);

}  // namespace dftbhip
