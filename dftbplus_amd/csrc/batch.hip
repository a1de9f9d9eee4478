// Batched SCC kernels for many independent molecules in one launch (batch.hip).
//
// A batch is one block-diagonal system: atoms and orbitals of all molecules are numbered
// consecutively and the neighbour list holds only intra-molecule pairs, so the sparse kernels
// (H0/S assembly, shift, pack, Mulliken, pair forces, repulsive) run unchanged over the union.
// What is per molecule lives here: the dense matrices (packed one after the other, n_m x n_m
// column-major), the generalized eigensolver (Cholesky and the inverse factor once per geometry,
// then per call a direct solve, or parallel cyclic Jacobi by one workgroup: in HBM for molecules
// above kWgBatchMax orbitals, in LDS for those of up to kBatchSmall in a batch without larger
// direct ones), the density matrices and the cluster gamma matrix with its products and gradient.
// The eigensolver and density kernels visit the molecules largest first (BatchLayout::order).
#include "batch.h"
#include "gamma_dev.h"
#include "lanes.h"

namespace dftbhip {

// The two kernels below give each SK block 16 lanes, lane e holding element e = r + c n2 of the
// column-major n2 x n1 block (lanes past n1 n2 idle): a wave's blocks are consecutive in the
// sparse arrays, so their loads and stores are contiguous.
constexpr int kBatchBlkLanes = 16;

// sparse -> per-molecule dense (both triangles); the dense array is zeroed beforehand
__global__ void batch_unpack_kernel(PairsDev pr, const int* norbAtom, const long* iAtomStart,
                                    BatchLayout L, const double* x, double* dense) {
  const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const int k = (int)(t / kBatchBlkLanes), e = (int)(t % kBatchBlkLanes);
  if (k >= pr.nblk) return;
  const int a1 = pr.at1[k], a2 = pr.at2[k];
  const int n1 = norbAtom[a1], n2 = norbAtom[a2];
  if (e >= n1 * n2) return;
  const int r = e % n2, c = e / n2;
  const int m = L.atomMol[a1];
  const long o0 = L.orb0[m];
  const int n = (int)(L.orb0[m + 1] - o0);
  double* d = dense + L.dOff[m];
  const long o1 = iAtomStart[a1] - o0, o2 = iAtomStart[a2] - o0;
  const double v = x[pr.start[k] + e];
  atomicAdd(&d[(o2 + r) + (o1 + c) * n], v);
  if (a1 != a2) atomicAdd(&d[(o1 + c) + (o2 + r) * n], v);
}

// per-molecule dense (lower triangle read for on-site blocks) -> sparse
__global__ void batch_pack_kernel(PairsDev pr, const int* norbAtom, const long* iAtomStart,
                                  BatchLayout L, const double* dense, double* x) {
  const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
  const int k = (int)(t / kBatchBlkLanes), e = (int)(t % kBatchBlkLanes);
  if (k >= pr.nblk) return;
  const int a1 = pr.at1[k], a2 = pr.at2[k];
  const int n1 = norbAtom[a1], n2 = norbAtom[a2];
  if (e >= n1 * n2) return;
  const int r = e % n2, c = e / n2;
  const int m = L.atomMol[a1];
  const long o0 = L.orb0[m];
  const int n = (int)(L.orb0[m + 1] - o0);
  const double* d = dense + L.dOff[m];
  const long o1 = iAtomStart[a1] - o0, o2 = iAtomStart[a2] - o0;
  long rr = r, cc = c;
  if (a1 == a2 && r < c) {
    rr = c;
    cc = r;
  }
  x[pr.start[k] + e] = d[(o2 + rr) + (o1 + cc) * n];
}

// ------------------------------------------------------------------------------------------
// Generalized eigensolver H C = S C E of a large molecule, one 1024-thread workgroup each.
//
// S is fixed for a geometry, so the reduction to standard form is done once: a cold call
// factors S = L L^T and starts from C = L^-T. Every call forms A = C^T H C with two workgroup
// GEMMs and diagonalizes A by parallel cyclic Jacobi, applying each round's rotations to A from
// both sides (one pass over its 2 x 2 blocks) and to the columns of C. Rotations keep
// C^T S C = I, so the rotated C holds the generalized eigenvectors. A warm call starts from the
// C of the previous call, for which A is already nearly diagonal when H changed little.
// Work: 3 n^2 doubles per molecule at 3 dOff[m]: B0 (L, then A), B1 (H C) and Cw (the C above,
// columns in Jacobi order, kept between calls).
// ------------------------------------------------------------------------------------------
constexpr int kJacobiMaxSweeps = 30;

// Rotation test of a Jacobi pair: the off-diagonal element is above the relative level of the
// smaller diagonal entry AND above the rounding level of the matrix (floor = 4 eps max|a_ii| of
// the matrix the sweeps start from). Without the floor, a pair touching a diagonal entry near 0
// would rotate forever on the rounding noise that other rotations leave in its element.
__device__ inline bool jacobi_rotates(double apq, double app, double aqq, double floor) {
  const double eps = 2.220446049250313e-16;
  const double a = fabs(apq);
  return a > 1e-300 && a > floor && 100.0 * a > eps * fmin(fabs(app), fabs(aqq));
}
constexpr int kSygvThreads = 1024;
constexpr int kGT = 64;   // workgroup GEMM output tile
constexpr int kGK = 16;   // workgroup GEMM k chunk

__device__ __forceinline__ void jacobi_pair(int N2, int r, int k, int& p, int& q) {
  p = (k == 0) ? 0 : 1 + (r + k - 1) % (N2 - 1);
  q = 1 + (r + N2 - 2 - k) % (N2 - 1);
}

// Unit u of the unordered pairs (k1, k2), k1 <= k2, numbered k2 (k2 + 1) / 2 + k1.
__device__ __forceinline__ void unit_pairs(int u, int& k1, int& k2) {
  int b = (int)((sqrtf(8.0f * (float)u + 1.0f) - 1.0f) * 0.5f);
  while ((b + 1) * (b + 2) / 2 <= u) ++b;
  while (b * (b + 1) / 2 > u) --b;
  k2 = b;
  k1 = u - b * (b + 1) / 2;
}

// sum_{k < len} x[k * sx] * y[k * sy] with four independent partial sums
__device__ __forceinline__ double dot4(const double* __restrict__ x, long sx,
                                       const double* __restrict__ y, long sy, int len) {
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  int k = 0;
  for (; k + 4 <= len; k += 4) {
    s0 += x[k * sx] * y[k * sy];
    s1 += x[(k + 1) * sx] * y[(k + 1) * sy];
    s2 += x[(k + 2) * sx] * y[(k + 2) * sy];
    s3 += x[(k + 3) * sx] * y[(k + 3) * sy];
  }
  for (; k < len; ++k) s0 += x[k * sx] * y[k * sy];
  return (s0 + s1) + (s2 + s3);
}

// Applies one Jacobi round's rotations (pairs rp/rq with cosines rc and sines rs, s = 0: none)
// to the columns of the n x n column-major C (leading dimension n, global memory or LDS): thread
// t takes row i = t mod n and the pairs g, g + G, ... with g = t / n, G = threads / n, all of
// its kB loads issued before the stores. Needs n <= the workgroup size.
template <int kB>
__device__ __forceinline__ void rotate_columns(double* C, int n, int np, const int* rp,
                                               const int* rq, const double* rc,
                                               const double* rs) {
  const int G = kSygvThreads / n;
  const int g = threadIdx.x / n, i = threadIdx.x - g * n;
  if (g >= G) return;
  for (int k0 = g; k0 < np; k0 += kB * G) {
    double cp[kB], cq[kB];
#pragma unroll
    for (int u = 0; u < kB; ++u) {
      const int k = k0 + u * G;
      cp[u] = 0.0;
      cq[u] = 0.0;
      if (k < np && rs[k] != 0.0) {
        cp[u] = C[i + rp[k] * n];
        cq[u] = C[i + rq[k] * n];
      }
    }
    // the pair data are read again from LDS below rather than held in registers
    __asm__ volatile("" ::: "memory");
#pragma unroll
    for (int u = 0; u < kB; ++u) {
      const int k = k0 + u * G;
      if (k < np && rs[k] != 0.0) {
        const double c = rc[k], sn = rs[k];
        C[i + rp[k] * n] = c * cp[u] - sn * cq[u];
        C[i + rq[k] * n] = sn * cp[u] + c * cq[u];
      }
    }
  }
}


// Workgroup GEMM on n x n column-major matrices (leading dimension n):
//   Z = op(X)(:, 0:kd) diag(wk) op(Y)(0:kd, :),  op(X) = X or X^T, op(Y) = Y or Y^T,
// wk optional. 1024 threads; 64 x 64 output tiles, each thread rows tx, tx + 32 by columns
// ty, ty + 32; k in chunks of 16 staged in LDS, the next chunk's loads issued before the
// current chunk's products. Z must not overlap X or Y.
template <bool TX, bool TY>
__device__ void wg_gemm(int n, int kd, const double* __restrict__ X, const double* __restrict__ Y,
                        const double* __restrict__ wk, double* __restrict__ Z,
                        double (*Xs)[kGT + 1], double (*Ys)[kGT + 1]) {
  const int tid = threadIdx.x;
  const int tx = tid % 32, ty = tid / 32;
  // the element each thread stages per chunk: op(X)(xr, xk) and op(Y)(yk, yc)
  const int xr = TX ? tid / kGK : tid % kGT, xk = TX ? tid % kGK : tid / kGT;
  const int yk = TY ? tid / kGT : tid % kGK, yc = TY ? tid % kGT : tid / kGK;
  const int nt = (n + kGT - 1) / kGT;
  for (int tile = 0; tile < nt * nt; ++tile) {
    const int r0 = (tile % nt) * kGT, c0 = (tile / nt) * kGT;
    auto ldx = [&](int k0) -> double {
      const int r = r0 + xr, k = k0 + xk;
      if (r >= n || k >= kd) return 0.0;
      const double v = TX ? X[k + (long)r * n] : X[r + (long)k * n];
      return wk ? v * wk[k] : v;
    };
    auto ldy = [&](int k0) -> double {
      const int k = k0 + yk, c = c0 + yc;
      if (c >= n || k >= kd) return 0.0;
      return TY ? Y[c + (long)k * n] : Y[k + (long)c * n];
    };
    double a00 = 0.0, a10 = 0.0, a01 = 0.0, a11 = 0.0;
    double xv = ldx(0), yv = ldy(0);
    for (int k0 = 0; k0 < kd; k0 += kGK) {
      __syncthreads();
      Xs[xk][xr] = xv;
      Ys[yk][yc] = yv;
      __syncthreads();
      if (k0 + kGK < kd) {
        xv = ldx(k0 + kGK);
        yv = ldy(k0 + kGK);
      }
#pragma unroll
      for (int k = 0; k < kGK; ++k) {
        const double x0 = Xs[k][tx], x1 = Xs[k][tx + 32];
        const double y0 = Ys[k][ty], y1 = Ys[k][ty + 32];
        a00 += x0 * y0;
        a10 += x1 * y0;
        a01 += x0 * y1;
        a11 += x1 * y1;
      }
    }
    const int ra = r0 + tx, rb = ra + 32, ca = c0 + ty, cb = ca + 32;
    if (ra < n && ca < n) Z[ra + (long)ca * n] = a00;
    if (rb < n && ca < n) Z[rb + (long)ca * n] = a10;
    if (ra < n && cb < n) Z[ra + (long)cb * n] = a01;
    if (rb < n && cb < n) Z[rb + (long)cb * n] = a11;
  }
  __syncthreads();
}

// Cholesky S = L L^T of one molecule (B0 overwritten) and Cw = L^-T: column i of Cw is row i of
// L^-1. False (and info) when a leading minor is not positive definite.
__device__ bool wg_factor(int n, const double* Sm, double* B0, double* Cw, int* info) {
  constexpr int NT = kSygvThreads;
  const long nn = (long)n * n;
  const int tid = threadIdx.x;
  __shared__ int flag;
  if (tid == 0) flag = 0;
  for (long e = tid; e < nn; e += NT) B0[e] = Sm[e];
  __syncthreads();
  // Cholesky S = L L^T (lower, right-looking)
  for (int j = 0; j < n; ++j) {
    if (tid == 0) {
      const double d = B0[j + (long)j * n];
      if (!(d > 0.0)) {
        flag = j + 1;
      } else {
        B0[j + (long)j * n] = sqrt(d);
      }
    }
    __syncthreads();
    if (flag != 0) {
      if (tid == 0) *info = flag;
      return false;
    }
    const double djj = B0[j + (long)j * n];
    for (int i = j + 1 + tid; i < n; i += NT) B0[i + (long)j * n] /= djj;
    __syncthreads();
    const int len = n - j - 1;
    for (long e = tid; e < (long)len * len; e += NT) {
      const int i = j + 1 + (int)(e % len), k = j + 1 + (int)(e / len);
      if (i >= k) B0[i + (long)k * n] -= B0[i + (long)j * n] * B0[k + (long)j * n];
    }
    __syncthreads();
  }
  // L^T into the upper triangle: row i of L is then contiguous (column i of the upper part)
  for (long e = tid; e < nn; e += NT) {
    const int i = (int)(e % n), k = (int)(e / n);
    if (i > k) B0[k + (long)i * n] = B0[i + (long)k * n];
  }
  __syncthreads();
  // Cw = L^-T: thread c forms column c of L^-1 by forward substitution and stores it as row c
  // of Cw, so that the lanes of a wave read and write consecutive addresses
  for (int c = tid; c < n; c += NT)
    for (int i = 0; i < n; ++i) {
      double v = 0.0;
      if (i >= c)
        v = ((i == c ? 1.0 : 0.0) - dot4(B0 + (long)i * n, 1, Cw + c, n, i)) /
            B0[i + (long)i * n];
      Cw[c + (long)i * n] = v;
    }
  __syncthreads();
  return true;
}

__global__ __launch_bounds__(kSygvThreads) void batch_sygv_kernel(BatchLayout L, const int* list,
                                                                  const double* S,
                                                                  const double* H, double* work,
                                                                  double* w, double* C,
                                                                  int* info, const int* active,
                                                                  int warm) {
  constexpr int NT = kSygvThreads;
  const int m = list[blockIdx.x];
  if (active && !active[m]) return;   // converged: eigenpairs stay from the last pass
  __shared__ double Xs[kGK][kGT + 1], Ys[kGK][kGT + 1];
  __shared__ double rc[kBatchMaxOrb / 2], rs[kBatchMaxOrb / 2];
  __shared__ int rp[kBatchMaxOrb / 2], rq[kBatchMaxOrb / 2];
  __shared__ int perm[kBatchMaxOrb];
  __shared__ int nrot, need;
  __shared__ unsigned long long dmaxBits;
  const int tid = threadIdx.x;
  const long base = L.dOff[m];
  const int n = (int)(L.orb0[m + 1] - L.orb0[m]);
  const long nn = (long)n * n;
  const double* Hm = H + base;
  double* B0 = work + 3 * base;
  double* B1 = B0 + nn;
  double* Cw = B1 + nn;
  double* Cm = C + base;
  double* wm = w + L.orb0[m];
  if (!warm) {
    if (!wg_factor(n, S + base, B0, Cw, info + m)) return;
  }
  // A = Cw^T H Cw (symmetrized)
  wg_gemm<false, false>(n, n, Hm, Cw, nullptr, B1, Xs, Ys);
  wg_gemm<true, false>(n, n, Cw, B1, nullptr, B0, Xs, Ys);
  double* A = B0;
  for (long e = tid; e < nn; e += NT) {
    const int i = (int)(e % n), j = (int)(e / n);
    if (i > j) {
      const double v = 0.5 * (A[i + (long)j * n] + A[j + (long)i * n]);
      A[i + (long)j * n] = v;
      A[j + (long)i * n] = v;
    }
  }
  __syncthreads();
  // parallel cyclic Jacobi, round-robin pairing (n odd: index n is a dummy that never rotates)
  const int N2 = n + (n & 1);
  const int np = N2 / 2;
  const int nunit = np * (np + 1) / 2;
  constexpr int kAU = 4;   // A-update units per thread and pass
  const int npair = n * (n - 1) / 2;
  // rounding level of the matrix: 4 eps max |a_ii| (bits of non-negative doubles order as
  // unsigned integers, so the maximum is an integer atomic)
  if (tid == 0) dmaxBits = 0ull;
  __syncthreads();
  {
    double dm = 0.0;
    for (int i = tid; i < n; i += NT) dm = fmax(dm, fabs(A[i + (long)i * n]));
    atomicMax(&dmaxBits, (unsigned long long)__double_as_longlong(dm));
  }
  __syncthreads();
  const double rotFloor = 4.0 * 2.220446049250313e-16 * __longlong_as_double((long long)dmaxBits);
  bool done = n <= 1;
  for (int sweep = 0; sweep < kJacobiMaxSweeps && n > 1; ++sweep) {
    // a sweep in which no pair passes the rotation test changes nothing: test all pairs first
    if (tid == 0) {
      nrot = 0;
      need = 0;
    }
    __syncthreads();
    for (int u = tid; u < npair; u += NT) {
      int k1, k2;
      unit_pairs(u, k1, k2);
      const int p = k1, q = k2 + 1;
      const double apq = A[p + (long)q * n];
      const double app = A[p + (long)p * n], aqq = A[q + (long)q * n];
      if (jacobi_rotates(apq, app, aqq, rotFloor)) need = 1;
    }
    __syncthreads();
    if (need == 0) {
      done = true;
      break;
    }
    for (int r = 0; r < N2 - 1; ++r) {
      for (int k = tid; k < np; k += NT) {
        int p, q;
        jacobi_pair(N2, r, k, p, q);
        double c = 1.0, s = 0.0;
        if (p < n && q < n) {
          const double apq = A[p + (long)q * n];
          const double app = A[p + (long)p * n], aqq = A[q + (long)q * n];
          if (jacobi_rotates(apq, app, aqq, rotFloor)) {
            const double th = (aqq - app) / (2.0 * apq);
            const double t = copysign(1.0, th) / (fabs(th) + sqrt(th * th + 1.0));
            c = 1.0 / sqrt(t * t + 1.0);
            s = t * c;
            atomicAdd(&nrot, 1);
          }
        }
        rp[k] = p;
        rq[k] = q;
        rc[k] = c;
        rs[k] = s;
      }
      __syncthreads();
      // A <- J^T A J over the unordered 2 x 2 blocks (rows of pair k1, columns of pair k2,
      // k1 <= k2; the block and its transpose take the same values), kAU per thread with all
      // loads ahead of the stores; only the loaded values stay in registers in between
      for (int u0 = tid; u0 < nunit; u0 += kAU * NT) {
        double x[kAU][4];
#pragma unroll
        for (int a = 0; a < kAU; ++a) {
          const int u = u0 + a * NT;
          if (u >= nunit) continue;
          int k1, k2;
          unit_pairs(u, k1, k2);
          if (rs[k1] == 0.0 && rs[k2] == 0.0) continue;
          const int row[2] = {rp[k1], rq[k1]}, col[2] = {rp[k2], rq[k2]};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int ri = row[e & 1], ci = col[e >> 1];
            x[a][e] = ri < n && ci < n ? A[ri + ci * n] : 0.0;   // n <= kBatchMaxOrb
          }
        }
        __asm__ volatile("" ::: "memory");
#pragma unroll
        for (int a = 0; a < kAU; ++a) {
          const int u = u0 + a * NT;
          if (u >= nunit) continue;
          int k1, k2;
          unit_pairs(u, k1, k2);
          const double c1 = rc[k1], s1 = rs[k1], c2 = rc[k2], s2 = rs[k2];
          if (s1 == 0.0 && s2 == 0.0) continue;
          // x[e]: e = 0 (p1, p2), 1 (q1, p2), 2 (p1, q2), 3 (q1, q2); columns first
          const double y0 = c2 * x[a][0] - s2 * x[a][2];
          const double y1 = c2 * x[a][1] - s2 * x[a][3];
          const double y2 = s2 * x[a][0] + c2 * x[a][2];
          const double y3 = s2 * x[a][1] + c2 * x[a][3];
          double z[4] = {c1 * y0 - s1 * y1, s1 * y0 + c1 * y1, c1 * y2 - s1 * y3,
                         s1 * y2 + c1 * y3};
          if (k1 == k2) z[1] = z[2];   // (q, p) and (p, q) alike
          const int row[2] = {rp[k1], rq[k1]}, col[2] = {rp[k2], rq[k2]};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int ri = row[e & 1], ci = col[e >> 1];
            if (ri < n && ci < n) {
              A[ri + ci * n] = z[e];
              if (k1 != k2) A[ci + ri * n] = z[e];
            }
          }
        }
      }
      rotate_columns<8>(Cw, n, np, rp, rq, rc, rs);
      __syncthreads();
    }
    if (nrot == 0) {
      done = true;
      break;
    }
    __syncthreads();
  }
  // ascending eigenvalues (stable ranks), C(:, rank) = Cw(:, i)
  for (int i = tid; i < n; i += NT) {
    const double di = A[i + (long)i * n];
    int rank = 0;
    for (int j = 0; j < n; ++j) {
      const double dj = A[j + (long)j * n];
      rank += (dj < di || (dj == di && j < i)) ? 1 : 0;
    }
    perm[rank] = i;
    wm[rank] = di;
  }
  __syncthreads();
  for (long e = tid; e < nn; e += NT) {
    const int i = (int)(e % n), c = (int)(e / n);
    Cm[e] = Cw[i + (long)perm[c] * n];
  }
  // a molecule whose last allowed sweep still rotated is reported (info > 0), not taken as
  // converged
  if (tid == 0) info[m] = done ? 0 : kBatchEigenNoConv;
}

// ------------------------------------------------------------------------------------------
// The same for the smallest molecules with A (upper triangle packed by columns: (i, j), i <= j, at
// i + j (j + 1) / 2) and C in LDS, the whole solve in one launch. The direct solve takes ten, so
// up to kBatchSmall orbitals the sweeps are faster: per iteration of one molecule of 8 to 16
// orbitals 191 against 215 us, of 1024 378 against 403 us; of 17 to 24 orbitals 206 against
// 223 us for one but 572 against 525 us for 1024.
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ int sym_idx(int i, int j) {
  return i <= j ? i + j * (j + 1) / 2 : j + i * (i + 1) / 2;
}

__global__ __launch_bounds__(kSygvThreads) __attribute__((amdgpu_waves_per_eu(8)))
void batch_sygv_small_kernel(BatchLayout L, const int* list, const double* S, const double* H,
                             double* work, double* w, double* C, int* info, const int* active,
                             int warm) {
  constexpr int NT = kSygvThreads, kMaxN = kBatchSmall;
  constexpr int kPacked = kMaxN * (kMaxN + 1) / 2;
  constexpr int kStage = 2 * kGK * (kGT + 1);   // also the staging of the products
  __shared__ double As[kPacked > kStage ? kPacked : kStage];
  __shared__ double Cs[kMaxN * kMaxN];
  __shared__ double rc[kMaxN / 2], rs[kMaxN / 2];
  __shared__ int rp[kMaxN / 2], rq[kMaxN / 2];
  __shared__ int perm[kMaxN];
  __shared__ int nrot, need;
  __shared__ unsigned long long dmaxBits;
  const int m = list[blockIdx.x];
  if (active && !active[m]) return;   // converged: eigenpairs stay from the last pass
  const int tid = threadIdx.x;
  const long base = L.dOff[m];
  const int n = (int)(L.orb0[m + 1] - L.orb0[m]);
  if (n > kMaxN) return;   // not of this class
  const long nn = (long)n * n;
  double* B0 = work + 3 * base;
  double* B1 = B0 + nn;
  double* Cw = B1 + nn;
  if (!warm) {
    if (!wg_factor(n, S + base, B0, Cw, info + m)) return;
  }
  double (*Xs)[kGT + 1] = reinterpret_cast<double (*)[kGT + 1]>(As);
  double (*Ys)[kGT + 1] = reinterpret_cast<double (*)[kGT + 1]>(As + kGK * (kGT + 1));
  wg_gemm<false, false>(n, n, H + base, Cw, nullptr, B1, Xs, Ys);
  wg_gemm<true, false>(n, n, Cw, B1, nullptr, B0, Xs, Ys);
  // A (symmetrized) into LDS
  for (long e = tid; e < nn; e += NT) {
    const int i = (int)(e % n), j = (int)(e / n);
    if (i <= j) As[i + j * (j + 1) / 2] = 0.5 * (B0[i + (long)j * n] + B0[j + (long)i * n]);
    Cs[e] = Cw[e];
  }
  __syncthreads();
  auto lds_barrier = [&]() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0); vmcnt, expcnt untouched (gfx9 encoding)
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  };
  const int N2 = n + (n & 1);
  const int np = N2 / 2;
  const int nunit = np * (np + 1) / 2;
  const int npair = n * (n - 1) / 2;
  // rounding level of the matrix: 4 eps max |a_ii| (bits of non-negative doubles order as
  // unsigned integers, so the maximum is an integer atomic)
  if (tid == 0) dmaxBits = 0ull;
  __syncthreads();
  {
    double dm = 0.0;
    for (int i = tid; i < n; i += NT) dm = fmax(dm, fabs(As[sym_idx(i, i)]));
    atomicMax(&dmaxBits, (unsigned long long)__double_as_longlong(dm));
  }
  __syncthreads();
  const double rotFloor = 4.0 * 2.220446049250313e-16 * __longlong_as_double((long long)dmaxBits);
  bool done = n <= 1;
  for (int sweep = 0; sweep < kJacobiMaxSweeps && n > 1; ++sweep) {
    // a sweep in which no pair passes the rotation test changes nothing: test all pairs first
    if (tid == 0) {
      nrot = 0;
      need = 0;
    }
    lds_barrier();
    for (int u = tid; u < npair; u += NT) {
      int k1, k2;
      unit_pairs(u, k1, k2);
      const int p = k1, q = k2 + 1;
      const double apq = As[sym_idx(p, q)];
      const double app = As[sym_idx(p, p)], aqq = As[sym_idx(q, q)];
      if (jacobi_rotates(apq, app, aqq, rotFloor)) need = 1;
    }
    lds_barrier();
    if (need == 0) {
      done = true;
      break;
    }
    for (int r = 0; r < N2 - 1; ++r) {
      for (int k = tid; k < np; k += NT) {
        int p, q;
        jacobi_pair(N2, r, k, p, q);
        double c = 1.0, s = 0.0;
        if (p < n && q < n) {
          const double apq = As[sym_idx(p, q)];
          const double app = As[sym_idx(p, p)], aqq = As[sym_idx(q, q)];
          if (jacobi_rotates(apq, app, aqq, rotFloor)) {
            const double th = (aqq - app) / (2.0 * apq);
            const double t = copysign(1.0, th) / (fabs(th) + sqrt(th * th + 1.0));
            c = 1.0 / sqrt(t * t + 1.0);
            s = t * c;
            atomicAdd(&nrot, 1);
          }
        }
        rp[k] = p;
        rq[k] = q;
        rc[k] = c;
        rs[k] = s;
      }
      lds_barrier();
      // A <- J^T A J over the unordered 2 x 2 blocks (pairs k1 <= k2)
      for (int u = tid; u < nunit; u += NT) {
        int k1, k2;
        unit_pairs(u, k1, k2);
        const double s1 = rs[k1], s2 = rs[k2];
        if (s1 == 0.0 && s2 == 0.0) continue;
        const double c1 = rc[k1], c2 = rc[k2];
        const int row[2] = {rp[k1], rq[k1]}, col[2] = {rp[k2], rq[k2]};
        double x[4];
        int o[4];
        bool v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int ri = row[e & 1], ci = col[e >> 1];
          v[e] = ri < n && ci < n;
          o[e] = v[e] ? sym_idx(ri, ci) : 0;
          x[e] = v[e] ? As[o[e]] : 0.0;
        }
        // e = 0 (p1, p2), 1 (q1, p2), 2 (p1, q2), 3 (q1, q2); columns first
        const double y0 = c2 * x[0] - s2 * x[2];
        const double y1 = c2 * x[1] - s2 * x[3];
        const double y2 = s2 * x[0] + c2 * x[2];
        const double y3 = s2 * x[1] + c2 * x[3];
        const double z[4] = {c1 * y0 - s1 * y1, s1 * y0 + c1 * y1, c1 * y2 - s1 * y3,
                             s1 * y2 + c1 * y3};
        if (k1 == k2) {
          // (p, p), (q, q) and the shared off-diagonal element
          if (v[0]) As[o[0]] = z[0];
          if (v[3]) As[o[3]] = z[3];
          if (v[2]) As[o[2]] = z[2];
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (v[e]) As[o[e]] = z[e];
        }
      }
      rotate_columns<8>(Cs, n, np, rp, rq, rc, rs);
      lds_barrier();
    }
    const int nr = nrot;
    lds_barrier();   // every thread has read nrot before the next sweep clears it
    if (nr == 0) {
      done = true;
      break;
    }
  }
  __syncthreads();   // every column of C written before other threads read it
  double* wm = w + L.orb0[m];
  for (int i = tid; i < n; i += NT) {
    const double di = As[sym_idx(i, i)];
    int rank = 0;
    for (int j = 0; j < n; ++j) {
      const double dj = As[sym_idx(j, j)];
      rank += (dj < di || (dj == di && j < i)) ? 1 : 0;
    }
    perm[rank] = i;
    wm[rank] = di;
  }
  __syncthreads();
  double* Cm = C + base;
  for (long e = tid; e < nn; e += NT) {
    const int i = (int)(e % n), c = (int)(e / n);
    Cm[e] = Cs[i + perm[c] * n];
    Cw[e] = Cs[e];   // the next warm call starts from the rotated C
  }
  // a molecule whose last allowed sweep still rotated is reported (info > 0), not taken as
  // converged
  if (tid == 0) info[m] = done ? 0 : kBatchEigenNoConv;
}

// ------------------------------------------------------------------------------------------
// Direct eigensolver for the other molecules of up to kWgBatchMax orbitals: L^-1 once per
// geometry (panels of 64 columns, every launch for all molecules that reach its panel; one
// workgroup per molecule in HBM took 2.1 ms for 190 orbitals), then per call A = L^-1 H L^-T
// (batched MFMA GEMMs), tridiagonalisation with the matrix in the registers of one workgroup
// (sytrd_resident.hip), divide and conquer of all molecules together (stedc.hip), the reflectors
// applied to strips of eigenvectors, and C = L^-T (Q Z). A parallel cyclic Jacobi with A and C in
// LDS ran here before, n dependent rounds per sweep and 7 to 10 sweeps. From
// set-up to forces, 32 molecules of 13 to 190 orbitals, eight iterations: 138 ms before, 14.6 ms
// now; 1000 molecules, five iterations: 249 ms before, 43.6 ms now. Bound by the column chain of
// the reduction (0.38 ms per iteration for 190 orbitals, 0.12 for 112), then by the solve's own
// latencies.
// ------------------------------------------------------------------------------------------
// Start of the factorisation: B0 = S, the place of L^-1 zero, info 0
__global__ void batch_factor_init_kernel(BatchLayout L, const int* list, const double* S,
                                         double* work, int* info) {
  const int m = list[blockIdx.y];
  const long n = L.orb0[m + 1] - L.orb0[m], nn = n * n;
  double* B0 = work + 3 * L.dOff[m];
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < nn;
       e += (long)gridDim.x * blockDim.x) {
    B0[e] = S[L.dOff[m] + e];
    B0[2 * nn + e] = 0.0;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) info[m] = 0;
}

// The products of a call, empty for molecules that are not active (or whose overlap failed)
__global__ void batch_desc_kernel(BatchLayout L, const int* list, int count, const double* H,
                                  double* work, double* C, const int* info, const int* active,
                                  BatchDescs g) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= count) return;
  const int m = list[t];
  const bool on = (!active || active[m]) && info[m] == 0;
  const int n = on ? (int)(L.orb0[m + 1] - L.orb0[m]) : 0;
  const long nn = L.dOff[m + 1] - L.dOff[m], ld = L.orb0[m + 1] - L.orb0[m];
  double* B0 = work + 3 * L.dOff[m];
  double* B1 = B0 + nn;
  const double* Li = B1 + nn;
  g.hc[t] = {n, n, n, H + L.dOff[m], ld, Li, ld, B1, ld};      // B1 = H L^-T
  g.chc[t] = {n, n, n, Li, ld, B1, ld, B0, ld};                // B0 = L^-1 B1
  g.back[t] = {n, n, n, Li, ld, B1, ld, C + L.dOff[m], ld};    // C = L^-T (Q Z)
  g.solve[m] = on;
}

// Z <- Q Z for the reflectors in A (below the subdiagonal of its columns): eight lanes per column
// of Z, lane g rows g + 8 r, all rows in registers, a wave eight columns; the reflectors are
// applied one after the other without any barrier, the next one's rows loaded meanwhile (without
// conditions: the rows above it are set to zero at their use). Bound by the chain of a reflector
// (dot product, sum over eight lanes, update): 103 us for 190 orbitals; 273 us with one
// accumulator and the row ranges tested per load.
// reflectors c1 down to c0, which leave the rows below 8 R0 as they are
template <int RQ, int R0>
__device__ __forceinline__ void apply_reflectors(int n, const double* A, const double* tm, int g,
                                                 int c1, int c0, double (&z)[RQ]) {
  if (c1 < c0) return;
  constexpr int K = RQ - R0;
  double v[K];
  auto load = [&](int c) {
#pragma unroll
    for (int r = 0; r < K; ++r) v[r] = A[min(g + 8 * (R0 + r), n - 1) + c * n];
  };
  load(c1);
  double t = tm[c1];
  for (int c = c1; c >= c0; --c) {
    double u[K];
#pragma unroll
    for (int r = 0; r < K; ++r) {
      const int i = g + 8 * (R0 + r);
      u[r] = i > c + 1 && i < n ? v[r] : (i == c + 1 ? 1.0 : 0.0);
    }
    const double tc = t;
    const int cn = max(c - 1, 0);
    load(cn);
    t = tm[cn];
    double p0 = 0.0, p1 = 0.0, p2 = 0.0, p3 = 0.0;
#pragma unroll
    for (int r = 0; r < K; ++r) {
      double& p = (r & 3) == 0 ? p0 : (r & 3) == 1 ? p1 : (r & 3) == 2 ? p2 : p3;
      p = fma(u[r], z[R0 + r], p);
    }
    const double dot = -tc * octet_sum((p0 + p1) + (p2 + p3));
#pragma unroll
    for (int r = 0; r < K; ++r) z[R0 + r] = fma(dot, u[r], z[R0 + r]);
  }
}

template <int RQ>
__global__ __launch_bounds__(256) void batch_apply_q_kernel(BatchLayout L, const int* list,
                                                            const int* solve, double* work,
                                                            const double* tau) {
  const int m = list[blockIdx.y];
  if (!solve[m]) return;
  const int n = (int)(L.orb0[m + 1] - L.orb0[m]);
  const int lane = threadIdx.x & 63, g = lane & 7;
  const int col = blockIdx.x * 32 + (threadIdx.x >> 6) * 8 + (lane >> 3);
  if (blockIdx.x * 32 + (threadIdx.x >> 6) * 8 >= n || n > 8 * RQ) return;   // whole waves
  const double* A = work + 3 * L.dOff[m];
  double* Z = work + 3 * L.dOff[m] + (long)n * n + (long)min(col, n - 1) * n;
  const double* tm = tau + L.orb0[m];
  double z[RQ];
#pragma unroll
  for (int r = 0; r < RQ; ++r) z[r] = g + 8 * r < n ? Z[g + 8 * r] : 0.0;
  // reflector c has rows from c + 1 on: four ranges of c, each with the rows it can reach
  constexpr int S1 = RQ / 4, S2 = RQ / 2, S3 = 3 * RQ / 4;
  apply_reflectors<RQ, S3>(n, A, tm, g, n - 2, 8 * S3 - 1, z);
  apply_reflectors<RQ, S2>(n, A, tm, g, min(n - 2, 8 * S3 - 2), 8 * S2 - 1, z);
  apply_reflectors<RQ, S1>(n, A, tm, g, min(n - 2, 8 * S2 - 2), 8 * S1 - 1, z);
  apply_reflectors<RQ, 0>(n, A, tm, g, min(n - 2, 8 * S1 - 2), 0, z);
  if (col < n)
#pragma unroll
    for (int r = 0; r < RQ; ++r)
      if (g + 8 * r < n) Z[g + 8 * r] = z[r];
}

// info of a molecule from its divide and conquer
__global__ void batch_info_kernel(const int* list, int count, const int* dc, int* info) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < count && dc[t] > 0) info[list[t]] = kBatchEigenNoConv;
}

// B1 = C diag(f) over the first nocc columns and the product P = B1 C^T
__global__ void batch_scale_kernel(BatchLayout L, const int* list, const double* C, const double* f,
                                   const int* nocc, double* P, const int* active, double* work,
                                   GemmDesc<double>* desc) {
  const int t = blockIdx.y, m = list[t];
  const long base = L.dOff[m];
  const int n = (int)(L.orb0[m + 1] - L.orb0[m]);
  const bool on = !active || active[m];
  double* B1 = work + 3 * base + (long)n * n;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    const int nd = on ? n : 0;
    desc[t] = {nd, nd, nocc[m], B1, (long)n, C + base, (long)n, P + base, (long)n};
  }
  if (!on) return;
  const long len = (long)n * nocc[m];
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < len;
       e += (long)gridDim.x * blockDim.x)
    B1[e] = C[base + e] * f[L.orb0[m] + e / n];
}

// gamma_m: 1/r off the diagonal minus the short-range expGamma part within its cutoff (on the
// diagonal the r -> 0 limit), the same sum the single-system path builds from the half list
__global__ __launch_bounds__(256) void batch_gamma_kernel(BatchLayout L, const double* coords,
                                                          const int* species,
                                                          const double* hubbu,
                                                          const double* gcut, int nsp,
                                                          double* g) {
  const int m = blockIdx.x;
  const int a0 = L.atom0[m];
  const int na = L.atom0[m + 1] - a0;
  double* gm = g + L.gOff[m];
  for (int e = threadIdx.x; e < na * na; e += 256) {
    const int i = e % na, j = e / na;
    const int ai = a0 + i, aj = a0 + j;
    const double dx = coords[3 * ai] - coords[3 * aj], dy = coords[3 * ai + 1] - coords[3 * aj + 1],
                 dz = coords[3 * ai + 2] - coords[3 * aj + 2];
    const double r = sqrt(dx * dx + dy * dy + dz * dz);
    double v = (i != j) ? 1.0 / r : 0.0;
    const int hi = ai > aj ? ai : aj, lo = ai > aj ? aj : ai;
    const int sh = species[hi], sl = species[lo];
    if (i == j || r <= gcut[sh * nsp + sl]) v += -expgamma(r, hubbu[sh], hubbu[sl]);
    gm[e] = v;
  }
}

// v_a = sum_b gamma(b, a) dq_b within the molecule of a
__global__ void batch_gemv_kernel(BatchLayout L, int nat, const double* g, const double* dq,
                                  double* v) {
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= nat) return;
  const int m = L.atomMol[a];
  const int a0 = L.atom0[m];
  const int na = L.atom0[m + 1] - a0;
  const double* col = g + L.gOff[m] + (long)(a - a0) * na;
  double acc = 0.0;
  for (int b = 0; b < na; ++b) acc += col[b] * dq[a0 + b];
  v[a] = acc;
}

// cluster 1/R gradient within each molecule
__global__ void batch_invr_grad_kernel(BatchLayout L, int nat, const double* coords,
                                       const double* dq, double* grad) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nat) return;
  const int m = L.atomMol[i];
  const int a0 = L.atom0[m], a1 = L.atom0[m + 1];
  double g0 = 0.0, g1 = 0.0, g2 = 0.0;
  for (int j = a0; j < a1; ++j) {
    if (j == i) continue;
    const double d0 = coords[3 * i] - coords[3 * j], d1 = coords[3 * i + 1] - coords[3 * j + 1],
                 d2 = coords[3 * i + 2] - coords[3 * j + 2];
    const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
    const double f = -dq[i] * dq[j] / (r2 * sqrt(r2));
    g0 += f * d0;
    g1 += f * d1;
    g2 += f * d2;
  }
  grad[3 * i] += g0;
  grad[3 * i + 1] += g1;
  grad[3 * i + 2] += g2;
}

int launch_batch_unpack(hipStream_t s, const PairsDev& pr, const int* norb,
                        const long* iAtomStart, const BatchLayout& L, const double* x,
                        double* dense, long denseSize) {
  DH_TRY(fill<double>(s, dense, denseSize, 0.0));
  if (pr.nblk == 0) return 0;
  hipLaunchKernelGGL(batch_unpack_kernel, dim3(cdiv((long)pr.nblk * kBatchBlkLanes, 256)),
                     dim3(256), 0, s, pr, norb,
                     iAtomStart, L, x, dense);
  DH_LAUNCH_CHECK();
  return 0;
}

int launch_batch_pack(hipStream_t s, const PairsDev& pr, const int* norb, const long* iAtomStart,
                      const BatchLayout& L, const double* dense, double* x) {
  if (pr.nblk == 0) return 0;
  hipLaunchKernelGGL(batch_pack_kernel, dim3(cdiv((long)pr.nblk * kBatchBlkLanes, 256)),
                     dim3(256), 0, s, pr, norb,
                     iAtomStart, L, dense, x);
  DH_LAUNCH_CHECK();
  return 0;
}

int BatchEigen::prepare(hipStream_t s, const BatchLayout& L, const std::vector<int>& order,
                        const std::vector<long>& orb0, const std::vector<long>& dOff,
                        double* matrices, double* C) {
  first[0] = 0;
  for (int c = 0; c < kBatchClasses; ++c) {
    first[c + 1] = first[c] + L.ncls[c];
    maxn[c] = L.ncls[c] > 0
                  ? (int)(orb0[order[first[c]] + 1] - orb0[order[first[c]]])   // largest first
                  : 0;
  }
  DH_CHECK(first[kBatchClasses] == L.nmol, "batch_sygv: size classes do not cover the batch");
  direct = first[kBatchJacobi] - first[1];
  DH_TRY(desc.alloc(4 * (size_t)std::max(L.nmol, 1)));
  if (direct == 0) return 0;
  const int end = first[kBatchJacobi];
  std::vector<DcBlock> blocks;
  for (int t = first[1]; t < end; ++t) {
    const int m = order[t];
    const int n = (int)(orb0[m + 1] - orb0[m]);
    // z goes to B1 of the molecule's work area
    blocks.push_back({n, orb0[m], dOff[m], 3 * dOff[m] + (long)n * n, n, m});
  }
  if (!dc) dc.reset(stedc_ws_new(), stedc_ws_delete);
  size_t dcWork = 0;
  DH_TRY(stedc_many_prepare(s, blocks, dc.get(), &dcWork));
  DH_TRY(work.alloc(dcWork));
  DH_TRY(solve.alloc(L.nmol));
  const size_t norb = orb0.back();
  DH_TRY(vec.alloc(3 * norb));
  d = vec.p;
  e = d + norb;
  tau = e + norb;
  // the products of the factorisation; the list is sorted, so the molecules that reach a panel or
  // a level are its first ones
  std::vector<GemmDesc<double>> h;
  steps.clear();
  auto size = [&](int t) { return orb0[order[t] + 1] - orb0[order[t]]; };
  const int big = (int)size(first[1]);
  for (int j = 0; j + kFactorNB < big; j += kFactorNB)
    for (int q = 0; q < 2; ++q) {
      FactorStep st{j, 0, 0, 0, (long)h.size()};
      for (int t = first[1]; t < end && size(t) > j + kFactorNB; ++t) {
        const long n = size(t), nn = n * n, r = j + kFactorNB;
        const int m = (int)(n - r);
        double* A = matrices + 3 * dOff[order[t]];
        // L21 = A21 L11^-T into B1, then A22 -= L21 L21^T
        if (q == 0) h.push_back({m, kFactorNB, kFactorNB, A + r + j * n, n, A + 2 * nn + j + j * n, n,
                                 A + nn + r + j * n, n});
        else h.push_back({m, m, kFactorNB, A + nn + r + j * n, n, A + nn + r + j * n, n,
                          A + r + r * n, n});
        ++st.count;
        st.m = std::max(st.m, m);
        st.n = std::max(st.n, q == 0 ? kFactorNB : m);
      }
      steps.push_back(st);
    }
  // pairs of diagonal blocks joined: T = L21 X11 (in C's place), X21 = -X22 T
  for (int p = kFactorNB; p < big; p *= 2)
    for (int q = 0; q < 2; ++q) {
      FactorStep st{-1, 0, 0, 0, (long)h.size()};
      for (int t = first[1]; t < end && size(t) > p; ++t) {
        const long n = size(t), nn = n * n;
        double* A = matrices + 3 * dOff[order[t]];
        double* T = C + dOff[order[t]];
        for (int r1 = 0; r1 + p < n; r1 += 2 * p) {
          const long r2 = r1 + p;
          const int n2 = (int)(std::min(r2 + p, n) - r2);
          double* X = A + 2 * nn;
          if (q == 0) h.push_back({n2, p, p, A + nn + r2 + r1 * n, n, X + r1 + r1 * n, n, T, n2});
          else h.push_back({n2, p, n2, X + r2 + r2 * n, n, T, n2, X + r2 + r1 * n, n});
          T += (long)n2 * p;
          ++st.count;
          st.m = std::max(st.m, n2);
          st.n = p;
        }
      }
      steps.push_back(st);
    }
  if (h.empty()) return 0;
  DH_TRY(factorDesc.upload(h.data(), h.size(), s));
  DH_HIP(hipStreamSynchronize(s));   // the descriptors' host copy
  return 0;
}

int launch_batch_sygv(hipStream_t s, const hipStream_t* st, BatchEigen& E, const BatchLayout& L,
                      const double* S, const double* H, double* work, double* w, double* C,
                      int* info, const int* active, bool warm, hipEvent_t* done) {
  if (L.ncls[0] > 0) {
    hipLaunchKernelGGL(batch_sygv_kernel, dim3(L.ncls[0]), dim3(kSygvThreads), 0, st[0], L,
                       L.order, S, H, work, w, C, info, active, warm ? 1 : 0);
    DH_LAUNCH_CHECK();
  }
  if (L.ncls[kBatchJacobi] > 0) {
    hipLaunchKernelGGL(batch_sygv_small_kernel, dim3(L.ncls[kBatchJacobi]), dim3(kSygvThreads), 0,
                       st[kBatchJacobi], L, L.order + E.first[kBatchJacobi], S, H, work, w, C,
                       info, active, warm ? 1 : 0);
    DH_LAUNCH_CHECK();
  }
  if (E.direct == 0) return 0;
  const int* list = L.order + E.first[1];
  const int nd = E.direct;
  GemmDesc<double>* g = E.desc.p;
  const BatchDescs ds{g, g + L.nmol, g + 2 * (size_t)L.nmol, E.solve.p};
  if (!warm) {
    for (int p = 0; p < nd; p += 32768) {
      hipLaunchKernelGGL(batch_factor_init_kernel, dim3(8, std::min(32768, nd - p)), dim3(256), 0, s,
                         L, list + p, S, work, info);
      DH_LAUNCH_CHECK();
    }
    int done = 0;   // panels whose diagonal block has been factored
    auto diagonals = [&](int upTo) -> int {
      for (; done <= upTo; done += kFactorNB)
        DH_TRY(launch_potrf_diag_list(s, nd, list, L.dOff, L.orb0, work, done, info));
      return 0;
    };
    bool second = false;
    for (const FactorStep& st : E.steps) {
      DH_TRY(diagonals(st.panel >= 0 ? st.panel : E.maxDirect() - 1));
      const GemmDesc<double>* d = E.factorDesc.p + st.first;
      if (st.panel >= 0)
        DH_TRY(gemm_batched<double>(s, false, true, d, st.count, st.m, st.n, second ? -1.0 : 1.0,
                                    second ? 1.0 : 0.0));
      else
        DH_TRY(gemm_batched<double>(s, false, false, d, st.count, st.m, st.n,
                                    second ? -1.0 : 1.0, 0.0));
      second = !second;
    }
    DH_TRY(diagonals(E.maxDirect() - 1));
  }
  hipLaunchKernelGGL(batch_desc_kernel, dim3(cdiv(nd, 256)), dim3(256), 0, s, L, list, nd, H, work,
                     C, info, active, ds);
  DH_LAUNCH_CHECK();
  auto each = [&](auto&& f) -> int {
    for (int c = 1; c < kBatchJacobi; ++c)
      if (L.ncls[c] > 0) DH_TRY(f(c, E.first[c] - E.first[1], L.ncls[c], E.maxn[c]));
    return 0;
  };
  // the classes' reductions side by side: a large molecule's chain of columns is long, and its
  // class has few workgroups
  DH_HIP(hipEventRecord(done[0], s));
  DH_TRY(each([&](int c, int o, int cnt, int mx) -> int {
    hipStream_t sc = st[c];
    if (sc != s) DH_HIP(hipStreamWaitEvent(sc, done[0], 0));
    DH_TRY(gemm_batched<double>(sc, false, true, ds.hc + o, cnt, mx, mx, 1.0, 0.0));
    DH_TRY(gemm_batched<double>(sc, false, false, ds.chc + o, cnt, mx, mx, 1.0, 0.0));
    WgBatch bt;
    bt.list = list + o;
    bt.active = E.solve.p;
    bt.aOff = L.dOff;
    bt.aMul = 3;
    bt.vOff = L.orb0;
    DH_TRY(sytrd_wg_batch(sc, work, cnt, mx, bt, E.d, E.e, E.tau));
    if (sc != s) {
      DH_HIP(hipEventRecord(done[c], sc));
      DH_HIP(hipStreamWaitEvent(s, done[c], 0));
    }
    return 0;
  }));
  DH_TRY(stedc_many(s, E.d, E.e, w, work, E.work.p, E.solve.p, E.dc.get()));
  hipLaunchKernelGGL(batch_info_kernel, dim3(cdiv(nd, 256)), dim3(256), 0, s, list, nd,
                     stedc_info(E.dc.get()), info);
  DH_LAUNCH_CHECK();
  return each([&](int c, int o, int cnt, int mx) -> int {
    for (int p = 0; p < cnt; p += 32768) {
      const dim3 grid(cdiv(mx, 32), std::min(32768, cnt - p));
#define DH_APPLY(RQ_)                                                                           \
  hipLaunchKernelGGL((batch_apply_q_kernel<RQ_>), grid, dim3(256), 0, s, L, list + o + p, E.solve.p, \
                     work, E.tau)
      if (mx <= 32) DH_APPLY(4);
      else if (mx <= 64) DH_APPLY(8);
      else if (mx <= 128) DH_APPLY(16);
      else if (mx <= 192) DH_APPLY(24);
      else DH_APPLY(28);
#undef DH_APPLY
      DH_LAUNCH_CHECK();
    }
    return gemm_batched<double>(s, true, false, ds.back + o, cnt, mx, mx, 1.0, 0.0);
  });
}

int launch_batch_density(hipStream_t s, BatchEigen& E, const BatchLayout& L, const double* C,
                         const double* f, const int* nocc, double* P, const int* active,
                         double* work) {
  GemmDesc<double>* g = E.desc.p + 3 * (size_t)L.nmol;
  for (int c = 0; c < kBatchClasses; ++c) {
    const int mx = E.maxn[c];
    for (int p = 0; p < L.ncls[c]; p += 32768) {
      const int cnt = std::min(32768, L.ncls[c] - p), o = E.first[c] + p;
      hipLaunchKernelGGL(batch_scale_kernel, dim3(cdiv((long)mx * mx, 2048), cnt), dim3(256), 0, s,
                         L, L.order + o, C, f, nocc, P, active, work, g + o);
      DH_LAUNCH_CHECK();
      DH_TRY(gemm_batched<double>(s, false, true, g + o, cnt, mx, mx, 1.0, 0.0));
    }
  }
  return 0;
}

int launch_batch_gamma(hipStream_t s, const BatchLayout& L, const double* coords,
                       const int* species, const double* hubbu, const double* gcut, int nsp,
                       double* g) {
  if (L.nmol == 0) return 0;
  hipLaunchKernelGGL(batch_gamma_kernel, dim3(L.nmol), dim3(256), 0, s, L, coords, species, hubbu,
                     gcut, nsp, g);
  DH_LAUNCH_CHECK();
  return 0;
}

int launch_batch_gemv(hipStream_t s, const BatchLayout& L, int nat, const double* g,
                      const double* dq, double* v) {
  if (nat == 0) return 0;
  hipLaunchKernelGGL(batch_gemv_kernel, dim3(cdiv(nat, 256)), dim3(256), 0, s, L, nat, g, dq, v);
  DH_LAUNCH_CHECK();
  return 0;
}

int launch_batch_invr_grad(hipStream_t s, const BatchLayout& L, int nat, const double* coords,
                           const double* dq, double* grad) {
  if (nat == 0) return 0;
  hipLaunchKernelGGL(batch_invr_grad_kernel, dim3(cdiv(nat, 256)), dim3(256), 0, s, L, nat,
                     coords, dq, grad);
  DH_LAUNCH_CHECK();
  return 0;
}

}  // namespace dftbhip
