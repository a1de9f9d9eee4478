// Symmetric tridiagonal eigensolver by divide and conquer (Cuppen's tearing with Gu-Eisenstat
// eigenvectors), producing all eigenvalues and eigenvectors of one tridiagonal or of many
// independent ones at once. Everything runs on the device: the launches of a solve depend on
// the sizes only, and the host neither reads nor decides anything in between.
//
//  * A tridiagonal is torn recursively into halves down to <= 16 rows; each tear subtracts |e|
//    from the two neighbouring diagonal entries and is undone by a rank-one merge
//    D + rho z z^T, rho = 2|e| after normalising z.
//  * Leaves: implicit QL with eigenvector accumulation, one wave per leaf.
//  * Merges, all merges of one height at once (a merge of height h joins blocks of height h - 1,
//    so problems of different depth share the launches):
//      - deflation (small |z| or close eigenvalues, LAPACK dlaed2 rules), one workgroup per merge:
//        ranks by binary search, prefix sums for the lists; only runs of close eigenvalues are
//        followed one by one, because a rotation changes the next test;
//      - secular roots, 16 lanes per root, by the fixed-weight rational iteration of Li ("the
//        middle way": two poles matched in value and slope) inside a bracket, bisection over
//        the IEEE bit patterns where a step leaves it; lambda is kept as pole + tau with the
//        origin at the pole nearer to the root, so d_i - lambda has no cancellation;
//      - z-hat from the roots (Loewner formula), eigenvectors u_j = zhat / (d - lambda_j);
//      - Q_new = Q_old(:, nondeflated) * U as two batched MFMA GEMMs (top rows use the columns
//        living in the first child plus the mixed ones, bottom rows the second child's).
//
// Bound by the latency of about eight launches per height. Measured, all of a solve: 2.3 ms at 573
// rows and 1.1 ms at 72 with the deflation on the host (two round trips and ten small copies per
// height), 64-step bisection for every root and leaves of 64; 0.52 ms and 0.25 ms in this form.
// Leaves of 32 instead of 16 took 130 instead of 44 us, a height costs about 45 us.
#include <algorithm>
#include <cmath>
#include <memory>

#include "common.h"
#include "stedc.h"

namespace dftbhip {

constexpr int kLeaf = 16;

struct LeafDev {
  int s, m;        // first array element and rows
  int c0, n;       // first row within the problem, rows of the problem
  int prob, pad;
  long q;          // offset of the block's first element in Q
  long ld;
};

struct MergeDev {
  // fixed by the sizes
  int s, n1, n2;   // first array element, rows of the children
  int prob;
  long q;          // offset of the block's first element (row and column s) in Q
  long ld;
  long qgOff;      // offset of the gathered columns (n x k) and of U (k x k)
  // set by the deflation
  int k, k1, k2, k3, nrot, ndefl;
  double rho;
};

struct ProblemDev {
  int s, n, parity;   // parity: which of the two Q buffers holds the eigenvectors
  int id;
  long q, z, ldz;     // offsets in Q and in the output
};

// Device buffers and the size-dependent tables of a solve, kept by the caller between calls:
// they only grow, so repeated solves of one size allocate and copy nothing.
struct StedcWs {
  std::vector<DcBlock> blocks;            // what the tables are for
  std::vector<LeafDev> leaves;
  std::vector<MergeDev> merges;           // by height
  std::vector<ProblemDev> problems;
  std::vector<int> first;                 // first merge of height h (h = 1 ...), and the end
  std::vector<int> maxn;                  // largest block of height h
  int maxProblem = 0;
  long total = 0, totalSq = 0;
  std::vector<char> staging;              // the tables as uploaded
  DevBuf<char> tables, arrays;
  const LeafDev* dleaf = nullptr;         // in tables
  MergeDev* dmerge = nullptr;
  const ProblemDev* dproblem = nullptr;
  GemmDesc<double>* ddesc = nullptr;      // in arrays
  double* darr = nullptr;                 // double arrays of length `total`, then the scales
  int* iarr = nullptr;                    // int arrays of length `total`, then the info words
  DevBuf<double> dd, de;                  // uploads of the host interface
  int* info = nullptr;
};

StedcWs* stedc_ws_new() { return new StedcWs(); }
void stedc_ws_delete(StedcWs* w) { delete w; }

// arrays indexed by element (s .. s + n of a block); columns are named by their array element
struct DcArrays {
  double *D, *z, *DL, *W, *tau, *lam, *zhat, *dval, *rc, *rs;
  int *ord, *idx, *cand, *flag, *type, *org, *row, *gcol, *dcol, *rp, *rn;
  int* info;   // per problem: not 0 when it failed; its merges and output are then skipped
  double* scale;   // per problem: the power of two its elements are multiplied by
};
constexpr int kDcDoubles = 10, kDcInts = 11;

// ------------------------------------------------------------------------------------------
// Leaves: implicit QL (tql2 scheme) with eigenvectors. Every lane runs the scalar recurrence
// (same operands, no broadcast), lane t applies each rotation to row t of the eigenvector matrix
// as soon as it is known; the recurrence is the bound, about 20 dependent operations a rotation.
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ void rotation_of(double f, double g, double& r, double& c, double& s) {
  const double q = fma(f, f, g * g);
  // every lane holds the same q: a scalar branch
  if (__ballot(q > 1e-280 && q < 1e280) == ~0ull) {
    double y = __builtin_amdgcn_rsq(q);
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const double hy = 0.5 * y;
      y = fma(hy, fma(-q * y, y, 1.0), y);
    }
    r = q * y;
    s = f * y;
    c = g * y;
    return;
  }
  r = hypot(f, g);
  s = r != 0.0 ? f / r : 0.0;
  c = r != 0.0 ? g / r : 0.0;
}

__global__ __launch_bounds__(64) void leaf_kernel(const double* dIn, const double* eIn,
                                                  const LeafDev* leaves, double* Q, DcArrays A) {
  __shared__ double z[kLeaf][kLeaf + 1];   // z[col][row]
  __shared__ double d[kLeaf + 1], e[kLeaf + 1];
  const LeafDev L = leaves[blockIdx.x];
  const int m = L.m, t = threadIdx.x;
  if (A.info[L.prob] < 0) return;
  const double sc = A.scale[L.prob];
  if (t < m) {
    double v = sc * dIn[L.s + t];
    // the tears on both sides of the leaf
    if (t == 0 && L.c0 > 0) v -= fabs(sc * eIn[L.s - 1]);
    if (t == m - 1 && L.c0 + m < L.n) v -= fabs(sc * eIn[L.s + m - 1]);
    d[t] = v;
    e[t] = t < m - 1 ? sc * eIn[L.s + t] : 0.0;
  }
  const int row = min(t, kLeaf - 1);       // lanes past the leaf repeat a row nobody reads
  if (t < kLeaf)
    for (int c = 0; c < m; ++c) z[c][t] = c == t ? 1.0 : 0.0;
  __syncthreads();
  const double eps = 2.220446049250313e-16;
  // values that are no numbers would leave the lists of the merges incomplete
  const bool finite = t >= m || (fabs(d[t]) < HUGE_VAL && fabs(e[t]) < HUGE_VAL);
  int fail = __ballot(!finite) != 0;
  for (int l = 0; l < m && !fail; ++l) {
    for (int iter = 0;; ++iter) {
      // first negligible off-diagonal element from l on
      bool small = false;
      if (t < m - 1 && t >= l) small = fabs(e[t]) <= eps * (fabs(d[t]) + fabs(d[t + 1]));
      const unsigned long long b = __ballot(small);
      const int mm = b ? __ffsll((long long)b) - 1 : m - 1;
      if (mm == l) break;
      if (iter == 60) {
        fail = 1;
        break;
      }
      const double el = e[l], dl = d[l];
      double g = (d[l + 1] - dl) / (2.0 * el);
      double r = hypot(g, 1.0);
      g = d[mm] - dl + el / (g + copysign(r, g));
      double sn = 1.0, cs = 1.0, p = 0.0;
      double zf = z[mm][row];
      double ei = e[mm - 1], di = d[mm - 1], di1 = d[mm];
      bool under = false;
      for (int i = mm - 1; i >= l; --i) {
        const double zi = z[i][row];
        const double en = i > l ? e[i - 1] : 0.0, dn = i > l ? d[i - 1] : 0.0;
        const double f = sn * ei, bb = cs * ei;
        rotation_of(f, g, r, cs, sn);
        if (t == 0) e[i + 1] = r;
        if (r == 0.0) {
          if (t == 0) {
            d[i + 1] = di1 - p;
            e[mm] = 0.0;
          }
          z[i + 1][row] = zf;
          under = true;
          break;
        }
        g = di1 - p;
        r = (di - g) * sn + 2.0 * cs * bb;
        p = sn * r;
        if (t == 0) d[i + 1] = g + p;
        g = cs * r - bb;
        if (t < kLeaf) z[i + 1][row] = fma(sn, zi, cs * zf);
        zf = fma(cs, zi, -sn * zf);
        ei = en;
        di1 = di;
        di = dn;
      }
      if (!under) {
        if (t < kLeaf) z[l][row] = zf;
        if (t == 0) {
          d[l] = dl - p;
          e[l] = g;
          e[mm] = 0.0;
        }
      }
      __syncthreads();
    }
  }
  if (t == 0 && fail) atomicMax(&A.info[L.prob], L.c0 + 1);
  __syncthreads();
  if (t < m) {
    const double v = d[t];
    A.D[L.s + t] = v;
    int rank = 0;
    for (int c = 0; c < m; ++c) rank += d[c] < v || (d[c] == v && c < t);
    A.ord[L.s + rank] = L.s + t;
    for (int c = 0; c < m; ++c) Q[L.q + t + (long)c * L.ld] = z[c][t];
  }
}

// ------------------------------------------------------------------------------------------
// Deflation: one workgroup per merge
// ------------------------------------------------------------------------------------------
constexpr int kDefT = 256;

// exclusive prefix sum over the workgroup of one value per thread; total to all
__device__ __forceinline__ u64 block_scan(u64 v, u64* part, u64& total) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  u64 x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const u64 y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  __syncthreads();   // the last use of part
  if (lane == 63) part[wv] = x;
  __syncthreads();
  u64 base = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < kDefT / 64; ++w) {
    if (w < wv) base += part[w];
    total += part[w];
  }
  return base + x - v;
}

// number of elements of the ascending list (column names in ord[0 .. n-1]) below v (or, with
// `equal`, not above it)
__device__ __forceinline__ int count_below(const int* ord, int n, const double* D, double v,
                                           bool equal) {
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    const double x = D[ord[mid]];
    if (x < v || (equal && x == v)) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

__global__ __launch_bounds__(kDefT) void deflate_kernel(MergeDev* md, const double* eIn,
                                                        const double* Q, double* Qn, double* Qg,
                                                        double* U, GemmDesc<double>* desc,
                                                        DcArrays A) {
  __shared__ u64 part[kDefT / 64];
  __shared__ double red[2][kDefT / 64];
  __shared__ int sRot;
  MergeDev& m = md[blockIdx.x];
  const int s = m.s, n1 = m.n1, nb = m.n1 + m.n2;
  const int t = threadIdx.x;
  if (A.info[m.prob] != 0) {   // the same for every thread: written by earlier launches only
    if (t == 0) {
      m.k = m.k1 = m.k2 = m.k3 = m.nrot = m.ndefl = 0;
      desc[2 * blockIdx.x] = desc[2 * blockIdx.x + 1] = {0, 0, 0, Q, 1, Q, 1, Qn, 1};
    }
    return;
  }
  const double b = A.scale[m.prob] * eIn[s + n1 - 1];
  const double rho = 2.0 * fabs(b), sigma = b >= 0.0 ? 1.0 : -1.0;
  const double isq2 = 0.70710678118654752440;
  const double eps = 2.220446049250313e-16;
  // z: last row of child 1, sigma * first row of child 2
  double zmax = 0.0, dmax = 0.0;
  for (int c = t; c < nb; c += kDefT) {
    const double q = Q[m.q + (c < n1 ? n1 - 1 : n1) + (long)c * m.ld];
    const double z = (c < n1 ? q : sigma * q) * isq2;
    A.z[s + c] = z;
    A.type[s + c] = c < n1 ? 1 : 3;
    zmax = fmax(zmax, fabs(z));
    dmax = fmax(dmax, fabs(A.D[s + c]));
  }
  for (int o = 32; o > 0; o >>= 1) {
    zmax = fmax(zmax, __shfl_xor(zmax, o, 64));
    dmax = fmax(dmax, __shfl_xor(dmax, o, 64));
  }
  if ((t & 63) == 0) {
    red[0][t >> 6] = zmax;
    red[1][t >> 6] = dmax;
  }
  // ascending order of the block from its children's
  for (int c = t; c < nb; c += kDefT) {
    const int col = A.ord[s + c];
    const double v = A.D[col];
    const int r = c < n1 ? c + count_below(A.ord + s + n1, nb - n1, A.D, v, false)
                         : c - n1 + count_below(A.ord + s, n1, A.D, v, true);
    A.idx[s + r] = col;
  }
  __syncthreads();
  zmax = dmax = 0.0;
  for (int w = 0; w < kDefT / 64; ++w) {
    zmax = fmax(zmax, red[0][w]);
    dmax = fmax(dmax, red[1][w]);
  }
  const double tol = 8.0 * eps * fmax(dmax, zmax);
  // each thread a chunk of positions, so that lists keep their order
  const int ch = (nb + kDefT - 1) / kDefT;
  const int c0 = min(nb, t * ch), c1 = min(nb, c0 + ch);
  // small |z|: deflated; the others are candidates
  u64 cnt = 0, tot;
  for (int c = c0; c < c1; ++c) cnt += !(rho * fabs(A.z[A.idx[s + c]]) <= tol);
  u64 at = block_scan(cnt, part, tot);
  const int nc = (int)tot;
  for (int c = c0; c < c1; ++c) {
    const int col = A.idx[s + c];
    if (rho * fabs(A.z[col]) <= tol) {
      const int d = s + c - (int)at;   // positions before c that are not candidates
      A.dcol[d] = col;
      A.dval[d] = A.D[col];
    } else {
      A.cand[s + (int)at++] = col;
    }
  }
  __syncthreads();
  // candidates too close to the one before them, judged before any rotation
  auto close = [&](double zp, double zn, double dp, double dn, double& c, double& sn, double& r) {
    r = hypot(zn, zp);
    c = zn / r;
    sn = -zp / r;
    return fabs((dn - dp) * c * sn) <= tol;
  };
  const int q0 = min(nc, t * ch), q1 = min(nc, q0 + ch);
  cnt = 0;
  for (int q = q0; q < q1; ++q) {
    bool f = false;
    if (q > 0) {
      const int pj = A.cand[s + q - 1], nj = A.cand[s + q];
      double c, sn, r;
      f = close(A.z[pj], A.z[nj], A.D[pj], A.D[nj], c, sn, r);
    }
    A.org[s + q] = f;   // scratch until the roots are found
    cnt += f;
  }
  at = block_scan(cnt, part, tot);
  const int nf = (int)tot;
  for (int q = q0; q < q1; ++q) {
    const bool f = A.org[s + q] != 0;
    A.org[s + q] = 0;               // from here on: deflated by a rotation
    if (f) A.flag[s + (int)at++] = q;
  }
  __syncthreads();
  if (t == 0) {
    int nrot = 0, next = 0;
    for (int u = 0; u < nf; ++u) {
      int q = A.flag[s + u];
      if (q < next) continue;       // its pair was judged with rotated values
      while (q < nc) {
        const int pj = A.cand[s + q - 1], nj = A.cand[s + q];
        const double dp = A.D[pj], dn = A.D[nj];
        double c, sn, r;
        if (!close(A.z[pj], A.z[nj], dp, dn, c, sn, r)) break;
        A.z[nj] = r;
        A.z[pj] = 0.0;
        if (A.type[nj] != A.type[pj]) A.type[nj] = 2;
        A.type[pj] = 4;
        A.rp[s + nrot] = pj;
        A.rn[s + nrot] = nj;
        A.rc[s + nrot] = c;
        A.rs[s + nrot] = sn;
        ++nrot;
        A.D[nj] = dp * sn * sn + dn * c * c;
        A.D[pj] = dp * c * c + dn * sn * sn;
        A.org[s + q - 1] = 1;
        ++q;
      }
      next = q + 1;
    }
    sRot = nrot;
  }
  __syncthreads();
  const int nrot = sRot;
  const int nsmall = nb - nc, k = nc - nrot;
  // the remaining candidates in ascending order, grouped by type: 1 (child-1 rows only), 2
  // (both), 3 (child-2 rows only); counts of the three packed into one word
  u64 packed = 0;
  for (int q = q0; q < q1; ++q)
    if (!A.org[s + q]) packed += 1ull << (21 * (A.type[A.cand[s + q]] - 1));
  u64 before = block_scan(packed, part, tot);
  constexpr u64 kMask = (1ull << 21) - 1;
  const int k1 = (int)(tot & kMask), k2 = (int)((tot >> 21) & kMask), k3 = (int)(tot >> 42);
  for (int q = q0; q < q1; ++q) {
    const int col = A.cand[s + q];
    const int b1 = (int)(before & kMask), b2 = (int)((before >> 21) & kMask),
              b3 = (int)(before >> 42);
    if (A.org[s + q]) {
      const int d = s + nsmall + q - (b1 + b2 + b3);
      A.dcol[d] = col;
      A.dval[d] = A.D[col];
      continue;
    }
    const int ty = A.type[col];
    const int i = b1 + b2 + b3;
    const int pos = ty == 1 ? b1 : (ty == 2 ? k1 + b2 : k1 + k2 + b3);
    before += 1ull << (21 * (ty - 1));
    A.DL[s + i] = A.D[col];
    A.W[s + i] = A.z[col];
    A.row[s + i] = pos;
    A.gcol[s + pos] = col;
  }
  if (t == 0) {
    m.rho = rho;
    m.k = k;
    m.k1 = k1;
    m.k2 = k2;
    m.k3 = k3;
    m.nrot = nrot;
    m.ndefl = nsmall + nrot;
    const double* qg = Qg + m.qgOff;
    const double* u = U + m.qgOff;
    double* qn = Qn + m.q;
    GemmDesc<double>* g = desc + 2 * blockIdx.x;
    g[0] = {n1, k, k1 + k2, qg, (long)nb, u, (long)k, qn, m.ld};
    g[1] = {m.n2, k, k2 + k3, qg + n1 + (long)k1 * nb, (long)nb, u + k1, (long)k, qn + n1, m.ld};
  }
}

// Deflation rotations (in order) on the full rows of the merged block: one thread per row.
__global__ void rotate_kernel(const MergeDev* md, double* Q, DcArrays A) {
  const MergeDev m = md[blockIdx.y];
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= m.n1 + m.n2) return;
  for (int q = 0; q < m.nrot; ++q) {
    const int o = m.s + q;
    const double c = A.rc[o], s = A.rs[o];
    double* x = Q + m.q + r + (long)(A.rp[o] - m.s) * m.ld;
    double* y = Q + m.q + r + (long)(A.rn[o] - m.s) * m.ld;
    const double xv = *x, yv = *y;
    *x = c * xv + s * yv;
    *y = c * yv - s * xv;
  }
}

// Sums over the k terms of a merge are split over a group of kSecG lanes (lane sub takes
// i = sub, sub + kSecG, ...) and combined by an xor butterfly, which leaves the same total in
// every lane of the group (IEEE addition is commutative), so the group's decisions agree.
constexpr int kSecG = 16;

__device__ __forceinline__ double group_sum(double v) {
#pragma unroll
  for (int s = kSecG / 2; s >= 1; s >>= 1) v += __shfl_xor(v, s, 64);
  return v;
}
__device__ __forceinline__ double group_prod(double v) {
#pragma unroll
  for (int s = kSecG / 2; s >= 1; s >>= 1) v *= __shfl_xor(v, s, 64);
  return v;
}
// 1 / x to a unit in the last place for x in the normal range (poles differ by more than that)
__device__ __forceinline__ double recip(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(r, fma(-x, r, 1.0), r);
  return fma(r, fma(-x, r, 1.0), r);
}

// f(tau) = 1 + psi + phi, psi over the poles up to j, phi over those above, and their slopes
struct Secular {
  double psi, dpsi, phi, dphi;
};
__device__ __forceinline__ Secular secular_at(const double* DL, const double* W, int k, int j,
                                              double rho, double dorg, double tau, int sub) {
  Secular f{0.0, 0.0, 0.0, 0.0};
  for (int i = sub; i < k; i += kSecG) {
    const double den = (DL[i] - dorg) - tau, w = W[i];
    const double x = fabs(den) > 1e-290 ? w * recip(den) : w / den;
    if (i <= j) {
      f.psi = fma(w, x, f.psi);
      f.dpsi = fma(x, x, f.dpsi);
    } else {
      f.phi = fma(w, x, f.phi);
      f.dphi = fma(x, x, f.dphi);
    }
  }
  f.psi = rho * group_sum(f.psi);
  f.dpsi = rho * group_sum(f.dpsi);
  f.phi = rho * group_sum(f.phi);
  f.dphi = rho * group_sum(f.dphi);
  return f;
}

// Roots of 1 + rho sum_i W_i^2 / (DL_i - lambda) = 0, one lane group per root.
__global__ void secular_kernel(const MergeDev* md, DcArrays A) {
  const MergeDev& m = md[blockIdx.y];
  const int gid = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = gid / kSecG, sub = gid % kSecG;
  const int k = m.k;
  if (j >= k) return;   // the whole group: j is the same in its lanes
  const double* DL = A.DL + m.s;
  const double* W = A.W + m.s;
  const double rho = m.rho;
  const double eps = 2.220446049250313e-16;
  const bool last = j == k - 1;
  int org = j;
  double lo = 0.0, hi;   // bracket of tau: f < 0 at lo, f > 0 at hi (poles or evaluated points)
  double tau;
  Secular f;
  if (!last) {
    const double gap = DL[j + 1] - DL[j];
    tau = 0.5 * gap;
    f = secular_at(DL, W, k, j, rho, DL[j], tau, sub);
    if (1.0 + f.psi + f.phi >= 0.0) {
      hi = tau;
    } else {
      org = j + 1;
      tau -= gap;
      lo = tau;
      hi = 0.0;
    }
  } else {
    double nz = 0.0;
    for (int i = sub; i < k; i += kSecG) nz += W[i] * W[i];
    hi = rho * group_sum(nz);
    tau = hi;
    f = secular_at(DL, W, k, j, rho, DL[j], tau, sub);
  }
  const double dorg = DL[org];
  const double poleL = DL[j] - dorg, poleR = last ? 0.0 : DL[j + 1] - dorg;
  // f is known to eps times its terms and a factor that grows with the length of the sums, tau to
  // eps of itself
  const double noise = eps * (4.0 + 0.25 * sqrt((double)k));
  for (int it = 0; it < 80; ++it) {
    const double w = 1.0 + f.psi + f.phi;
    const double tol = noise * (1.0 + fabs(f.psi) + fabs(f.phi)) +
                       2.0 * eps * fabs(tau) * (f.dpsi + f.dphi);
    // closer than about 1e-154 to a pole, where the halving may take tau, the slopes overflow
    if (fabs(w) <= tol && tol < HUGE_VAL) break;
    if (w < 0.0) lo = tau;
    else hi = tau;
    // neighbours in the floating-point numbers: nothing lies between
    const long long bl = __double_as_longlong(fabs(lo)), bh = __double_as_longlong(fabs(hi));
    if (llabs(bh - bl) <= 1) break;
    // rational step: psi and phi each as a constant and their nearest pole, matched in value and
    // slope at tau
    const double dl = poleL - tau, dr = poleR - tau;
    double eta;
    if (last) {
      const double sres = f.dpsi * dl * dl, c = w - f.dpsi * dl;   // c + sres / (poleL - x) = 0
      eta = poleL + sres / c - tau;
    } else {
      const double c = w - dl * f.dpsi - dr * f.dphi;
      const double a = (dl + dr) * w - dl * dr * (f.dpsi + f.dphi);
      const double bb = dl * dr * w;
      const double disc = sqrt(fabs(a * a - 4.0 * bb * c));
      eta = c == 0.0 ? bb / a : (a <= 0.0 ? (a - disc) / (2.0 * c) : 2.0 * bb / (a + disc));
    }
    double next = tau + eta;
    // The step lost its sign or left the bracket: the root is then next to the origin's pole, many
    // orders of magnitude below tau, and comes from that pole with the rest of f as a constant.
    // (A Newton step or a bisection there took up to 55 more evaluations, and a launch lasts as
    // long as its slowest root: 576 instead of 30 us at 573 rows.)
    if (!(w * eta < 0.0 && next > lo && next < hi)) {
      const double pw = rho * W[org] * W[org];
      next = pw / (w + pw / tau);
    }
    // halve the bit patterns (tau keeps its sign)
    if (!(next > lo && next < hi) || it >= 16) {
      const long long mid = bl + (bh - bl) / 2;
      next = __longlong_as_double(mid);
      if (lo < 0.0 || hi <= 0.0) next = -next;
      if (!(next > lo && next < hi)) break;
    }
    tau = next;
    f = secular_at(DL, W, k, j, rho, dorg, tau, sub);
  }
  if (sub == 0) {
    A.org[m.s + j] = org;
    A.tau[m.s + j] = tau;
    A.lam[m.s + j] = dorg + tau;
  }
}

// zhat_i = sign(W_i) sqrt( -(DL_i - lam_i)/rho * prod_{j != i} (DL_i - lam_j)/(DL_i - DL_j) ),
// one lane group per i; by interlacing every factor below i is in (0, 1) and their product stays
// above the smallest gap over the spread, and those above i likewise from above, so the lanes'
// partial products stay in range.
__global__ void zhat_kernel(const MergeDev* md, DcArrays A) {
  const MergeDev& m = md[blockIdx.y];
  const int gid = blockIdx.x * blockDim.x + threadIdx.x;
  const int i = gid / kSecG, sub = gid % kSecG;
  if (i >= m.k) return;
  const double* DL = A.DL + m.s;
  const int* org = A.org + m.s;
  const double* tau = A.tau + m.s;
  const double di = DL[i];
  double prod = 1.0;
  for (int j = sub; j < m.k; j += kSecG) {
    const double num = (di - DL[org[j]]) - tau[j];
    prod *= j == i ? -num / m.rho : num / (di - DL[j]);
  }
  prod = group_prod(prod);
  if (sub == 0) {
    const double a = sqrt(fmax(prod, 0.0));
    A.zhat[m.s + i] = A.W[m.s + i] >= 0.0 ? a : -a;
  }
}

// Column j of U, rows in column-group order: U(row(i), j) = zhat_i / (DL_i - lam_j), normalised;
// one wave per column. Then the gathered columns Qg(:, q) = Q(block rows, gcol[q]), the same
// grid: a wave per column.
__global__ void buildu_kernel(const MergeDev* md, const double* Q, double* U, double* Qg,
                              DcArrays A) {
  const MergeDev& m = md[blockIdx.y];
  const int j = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, lane = threadIdx.x & 63;
  const int k = m.k, s = m.s, nb = m.n1 + m.n2;
  if (j >= k) return;
  const double* DL = A.DL + s;
  const double dorg = DL[A.org[s + j]], tj = A.tau[s + j];
  double acc = 0.0;
  for (int i = lane; i < k; i += 64) {
    const double v = A.zhat[s + i] / ((DL[i] - dorg) - tj);
    acc = fma(v, v, acc);
  }
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  const double inv = 1.0 / sqrt(acc);
  double* u = U + m.qgOff + (long)j * k;
  for (int i = lane; i < k; i += 64)
    u[A.row[s + i]] = A.zhat[s + i] / ((DL[i] - dorg) - tj) * inv;
  const double* q = Q + m.q + (long)(A.gcol[s + j] - s) * m.ld;
  double* g = Qg + m.qgOff + (long)j * nb;
  for (int r = lane; r < nb; r += 64) g[r] = q[r];
}

// New layout of a merged block: the k roots, then the deflated columns (copied to Qn, a wave per
// column); its eigenvalues and their ascending order.
__global__ void finish_kernel(const MergeDev* md, const double* Qold, double* Qn, DcArrays A) {
  const MergeDev& m = md[blockIdx.y];
  const int c = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, lane = threadIdx.x & 63;
  const int s = m.s, k = m.k, nb = m.n1 + m.n2;
  if (c >= nb || A.info[m.prob] != 0) return;
  const bool root = c < k;
  const double v = root ? A.lam[s + c] : A.dval[s + c - k];
  // deflated values before this one (a root comes before an equal deflated value)
  int below = 0;
  for (int q = lane; q < m.ndefl; q += 64) {
    const double x = A.dval[s + q];
    below += x < v || (!root && x == v && q < c - k);
  }
  for (int o = 32; o > 0; o >>= 1) below += __shfl_xor(below, o, 64);
  if (lane == 0) {
    int rank = below;
    if (root) {
      rank += c;
    } else {
      int lo = 0, hi = k;   // roots ascend
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (A.lam[s + mid] <= v) lo = mid + 1;
        else hi = mid;
      }
      rank += lo;
    }
    A.ord[s + rank] = s + c;
    A.D[s + c] = v;
  }
  if (!root) {
    const double* src = Qold + m.q + (long)(A.dcol[s + c - k] - s) * m.ld;
    double* dst = Qn + m.q + (long)c * m.ld;
    for (int r = lane; r < nb; r += 64) dst[r] = src[r];
  }
}

// eigenvalues ascending and the ordered eigenvectors
__global__ void collect_kernel(const ProblemDev* pr, const double* Qa, const double* Qb, double* w,
                               double* z, DcArrays A) {
  const ProblemDev p = pr[blockIdx.y];
  const int c = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, lane = threadIdx.x & 63;
  if (c >= p.n || A.info[blockIdx.y] != 0) return;
  const int col = A.ord[p.s + c];
  if (lane == 0) w[p.s + c] = A.D[col] / A.scale[blockIdx.y];   // a power of two
  const double* src = (p.parity ? Qb : Qa) + p.q + (long)(col - p.s) * p.n;
  double* dst = z + p.z + (long)c * p.ldz;
  for (int r = lane; r < p.n; r += 64) dst[r] = src[r];
}

// Zeros, and for each problem its state, to be solved or (-1) left as it is, and its scale. The
// deflation is to eps times the larger of the levels and z, so a matrix is scaled to a norm of at
// least 1/2 (LAPACK: to 1), and so that its squares stay in range.
constexpr int kZeroT = 256;
__global__ __launch_bounds__(kZeroT) void stedc_zero_kernel(double* q, size_t n,
                                                            const ProblemDev* pr,
                                                            const int* active, const double* d,
                                                            const double* e, int nprob,
                                                            int* info, double* scale) {
  __shared__ double part[kZeroT / 64];
  for (int k = blockIdx.x; k < nprob; k += gridDim.x) {
    const ProblemDev p = pr[k];
    double v = 0.0;
    for (int c = threadIdx.x; c < p.n; c += kZeroT) {
      v = fmax(v, fabs(d[p.s + c]));
      if (c + 1 < p.n) v = fmax(v, fabs(e[p.s + c]));
    }
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    __syncthreads();   // the last use of part
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 0; w < kZeroT / 64; ++w) v = fmax(v, part[w]);
      const bool asIs = v == 0.0 || (v >= 0.5 && v < 1e100) || !(v < HUGE_VAL);
      scale[k] = asIs ? 1.0 : ldexp(1.0, max(-1000, min(1000, -ilogb(v))));
      info[k] = active && !active[p.id] ? -1 : 0;
    }
  }
  const size_t stride = (size_t)gridDim.x * kZeroT;
  for (size_t i = (size_t)blockIdx.x * kZeroT + threadIdx.x; i < n; i += stride) q[i] = 0.0;
}

// ------------------------------------------------------------------------------------------
namespace {
struct Node {
  int s, n1, n2, height;
};
// Halves down to blocks of at most kLeaf rows, every branch to the same depth
void build_tree(int s, int n, int height, std::vector<Node>& merges,
                std::vector<std::pair<int, int>>& leaves) {
  if (height == 0) {
    leaves.push_back({s, n});
    return;
  }
  const int n1 = n / 2;
  build_tree(s, n1, height - 1, merges, leaves);
  build_tree(s + n1, n - n1, height - 1, merges, leaves);
  merges.push_back({s, n1, n - n1, height});
}
}  // namespace

static int dc_tables(hipStream_t s, StedcWs& W, const std::vector<DcBlock>& blocks) {
  if (W.blocks == blocks) return 0;
  W.blocks.clear();
  W.leaves.clear();
  W.merges.clear();
  W.problems.clear();
  W.maxProblem = 0;
  long off = 0, q = 0;   // ends of the arrays and of Q
  std::vector<std::vector<MergeDev>> byHeight;
  for (size_t p = 0; p < blocks.size(); ++p) {
    const DcBlock& bl = blocks[p];
    const int n = bl.n;
    DH_CHECK(n > 0 && n < (1 << 21), "stedc: problem size");   // packed counts of the deflation
    int h = 0;
    while (((n + (1 << h) - 1) >> h) > kLeaf) ++h;
    std::vector<Node> nodes;
    std::vector<std::pair<int, int>> lv;
    build_tree(0, n, h, nodes, lv);
    for (const auto& l : lv)
      W.leaves.push_back({(int)bl.off + l.first, l.second, l.first, n, (int)p, 0,
                          bl.q + l.first + (long)l.first * n, n});
    if ((int)byHeight.size() < h + 1) byHeight.resize(h + 1);
    for (const Node& x : nodes) {
      MergeDev m{};
      m.s = (int)bl.off + x.s;
      m.n1 = x.n1;
      m.n2 = x.n2;
      m.prob = (int)p;
      m.q = bl.q + x.s + (long)x.s * n;
      m.ld = n;
      byHeight[x.height].push_back(m);
    }
    W.problems.push_back({(int)bl.off, n, h & 1, bl.id, bl.q, bl.z, bl.ldz});
    W.maxProblem = std::max(W.maxProblem, n);
    off = std::max(off, bl.off + n);
    q = std::max(q, bl.q + (long)n * n);
  }
  DH_CHECK(off < (1L << 31), "stedc: too many rows");
  W.total = off;
  W.totalSq = q;
  W.first.assign(1, 0);
  W.maxn.assign(1, 0);
  for (size_t h = 1; h < byHeight.size(); ++h) {
    long o = 0;
    int mx = 0;
    W.first.push_back((int)W.merges.size());
    for (MergeDev& m : byHeight[h]) {
      const long nb = m.n1 + m.n2;
      m.qgOff = o;
      o += nb * nb;
      mx = std::max(mx, (int)nb);
      W.merges.push_back(m);
    }
    W.maxn.push_back(mx);
  }
  W.first.push_back((int)W.merges.size());
  // one buffer each for the tables and the arrays: a new batch or size makes all of them anew
  auto up = [](size_t bytes) { return (bytes + 255) / 256 * 256; };
  const size_t bl = up(W.leaves.size() * sizeof(LeafDev)),
               bm = up(W.merges.size() * sizeof(MergeDev)),
               bp = up(W.problems.size() * sizeof(ProblemDev));
  W.staging.resize(bl + bm + bp);
  std::copy_n(reinterpret_cast<const char*>(W.leaves.data()), W.leaves.size() * sizeof(LeafDev),
              W.staging.begin());
  std::copy_n(reinterpret_cast<const char*>(W.merges.data()), W.merges.size() * sizeof(MergeDev),
              W.staging.begin() + bl);
  std::copy_n(reinterpret_cast<const char*>(W.problems.data()),
              W.problems.size() * sizeof(ProblemDev), W.staging.begin() + bl + bm);
  DH_TRY(W.tables.upload(W.staging.data(), W.staging.size(), s));
  W.dleaf = reinterpret_cast<const LeafDev*>(W.tables.p);
  W.dmerge = reinterpret_cast<MergeDev*>(W.tables.p + bl);
  W.dproblem = reinterpret_cast<const ProblemDev*>(W.tables.p + bl + bm);
  const size_t bd = up(2 * W.merges.size() * sizeof(GemmDesc<double>)),
               ba = up(((size_t)kDcDoubles * W.total + blocks.size()) * sizeof(double)),
               bi = ((size_t)kDcInts * W.total + blocks.size()) * sizeof(int);
  DH_TRY(W.arrays.alloc(bd + ba + bi));
  W.ddesc = reinterpret_cast<GemmDesc<double>*>(W.arrays.p);
  W.darr = reinterpret_cast<double*>(W.arrays.p + bd);
  W.iarr = reinterpret_cast<int*>(W.arrays.p + bd + ba);
  W.info = W.iarr + (size_t)kDcInts * W.total;
  W.blocks = blocks;
  return 0;
}

// The launches of a solve on the tables in W. work: 4 totalSq doubles.
static int dc_launch(hipStream_t s, StedcWs& W, const double* d, const double* e, double* w,
                     double* z, double* work, const int* active) {
  constexpr int kRows = 32768;   // merges or problems in the y dimension of a launch
  DcArrays A;
  {
    double** dp[kDcDoubles] = {&A.D, &A.z, &A.DL, &A.W, &A.tau, &A.lam, &A.zhat, &A.dval,
                               &A.rc, &A.rs};
    int** ip[kDcInts] = {&A.ord, &A.idx, &A.cand, &A.flag, &A.type, &A.org, &A.row, &A.gcol,
                         &A.dcol, &A.rp, &A.rn};
    for (int i = 0; i < kDcDoubles; ++i) *dp[i] = W.darr + (size_t)i * W.total;
    for (int i = 0; i < kDcInts; ++i) *ip[i] = W.iarr + (size_t)i * W.total;
    A.info = W.info;
    A.scale = W.darr + (size_t)kDcDoubles * W.total;
  }
  const size_t sq = W.totalSq;
  double* Q[2] = {work, work + sq};
  double* Qg = work + 2 * sq;
  double* U = work + 3 * sq;
  // zeros outside the blocks of the leaves; the second buffer's blocks are written whole, its
  // zeros outside them are read by the next height
  hipLaunchKernelGGL(stedc_zero_kernel, dim3((unsigned)std::min<size_t>(cdiv(2 * sq, 1024), 2048)),
                     dim3(kZeroT), 0, s, work, 2 * sq, W.dproblem, active, d, e,
                     (int)W.problems.size(), A.info, A.scale);
  DH_LAUNCH_CHECK();
  hipLaunchKernelGGL(leaf_kernel, dim3((unsigned)W.leaves.size()), dim3(64), 0, s, d, e, W.dleaf,
                     Q[0], A);
  DH_LAUNCH_CHECK();
  for (size_t h = 1; h + 1 < W.first.size(); ++h) {
    const int mx = W.maxn[h];
    double* Qo = Q[(h - 1) & 1];
    double* Qn = Q[h & 1];
    for (int f = W.first[h]; f < W.first[h + 1]; f += kRows) {
      const int nm = std::min(kRows, W.first[h + 1] - f);
      MergeDev* md = W.dmerge + f;
      GemmDesc<double>* gd = W.ddesc + 2 * (size_t)f;
      hipLaunchKernelGGL(deflate_kernel, dim3(nm), dim3(kDefT), 0, s, md, e, Qo, Qn, Qg, U, gd, A);
      DH_LAUNCH_CHECK();
      hipLaunchKernelGGL(rotate_kernel, dim3(cdiv(mx, 64), nm), dim3(64), 0, s, md, Qo, A);
      DH_LAUNCH_CHECK();
      const dim3 gg(cdiv((long)mx * kSecG, 64), nm), gw(cdiv((long)mx * 64, 256), nm);
      hipLaunchKernelGGL(secular_kernel, gg, dim3(64), 0, s, md, A);
      DH_LAUNCH_CHECK();
      hipLaunchKernelGGL(zhat_kernel, gg, dim3(64), 0, s, md, A);
      DH_LAUNCH_CHECK();
      hipLaunchKernelGGL(buildu_kernel, gw, dim3(256), 0, s, md, Qo, U, Qg, A);
      DH_LAUNCH_CHECK();
      DH_TRY(gemm_batched<double>(s, false, false, gd, 2 * nm, (mx + 1) / 2, mx, 1.0, 0.0));
      hipLaunchKernelGGL(finish_kernel, gw, dim3(256), 0, s, md, Qo, Qn, A);
      DH_LAUNCH_CHECK();
    }
  }
  for (size_t p = 0; p < W.problems.size(); p += kRows) {
    DcArrays Ap = A;
    Ap.info += p;
    Ap.scale += p;
    hipLaunchKernelGGL(collect_kernel, dim3(cdiv((long)W.maxProblem * 64, 256),
                                            (unsigned)std::min<size_t>(kRows, W.problems.size() - p)),
                       dim3(256), 0, s, W.dproblem + p, Q[0], Q[1], w, z, Ap);
    DH_LAUNCH_CHECK();
  }
  return 0;
}

size_t stedc_work_size(int n) {
  // two Q buffers, gathered columns and U: 4 n^2
  return 4 * (size_t)n * n + 64;
}

int stedc_device(hipStream_t s, int n, const double* d, const double* e, double* w, double* z,
                 long ldz, double* work, size_t workSize, StedcWs* ws) {
  DH_CHECK(n > 0 && ws, "stedc: bad arguments");
  DH_CHECK(workSize >= stedc_work_size(n), "stedc: workspace too small");
  DH_TRY(dc_tables(s, *ws, {DcBlock{n, 0, 0, 0, ldz, 0}}));
  return dc_launch(s, *ws, d, e, w, z, work, nullptr);
}

int stedc_many_prepare(hipStream_t s, const std::vector<DcBlock>& blocks, StedcWs* ws,
                       size_t* workSize) {
  DH_TRY(dc_tables(s, *ws, blocks));
  *workSize = 4 * (size_t)ws->totalSq;
  return 0;
}

int stedc_many(hipStream_t s, const double* d, const double* e, double* w, double* z,
               double* work, const int* active, StedcWs* ws) {
  return ws->blocks.empty() ? 0 : dc_launch(s, *ws, d, e, w, z, work, active);
}

const int* stedc_info(const StedcWs* ws) { return ws->info; }

int stedc_fetch(hipStream_t s, int n, const double* w, double* wHost, StedcWs* ws, int* info) {
  DH_HIP(hipMemcpyAsync(wHost, w, n * sizeof(double), hipMemcpyDeviceToHost, s));
  DH_HIP(hipMemcpyAsync(info, ws->info, sizeof(int), hipMemcpyDeviceToHost, s));
  DH_HIP(hipStreamSynchronize(s));
  if (*info != 0) set_error("stedc: QL iteration did not converge in a leaf");
  return 0;
}

int stedc(hipStream_t s, int n, const double* dHost, const double* eHost, double* w, double* z,
          long ldz, double* work, size_t workSize, int* info, StedcWs* ws) {
  *info = 0;
  if (n <= 0) return 0;
  std::unique_ptr<StedcWs> own;
  if (!ws) {
    own.reset(new StedcWs());
    ws = own.get();
  }
  DH_TRY(ws->dd.upload(dHost, n, s));
  DH_TRY(ws->de.alloc(std::max(n - 1, 1)));
  if (n > 1) DH_TRY(ws->de.upload(eHost, n - 1, s));
  DH_TRY(stedc_device(s, n, ws->dd.p, ws->de.p, w, z, ldz, work, workSize, ws));
  DH_HIP(hipMemcpyAsync(info, ws->info, sizeof(int), hipMemcpyDeviceToHost, s));
  DH_HIP(hipStreamSynchronize(s));
  if (*info != 0) set_error("stedc: QL iteration did not converge in a leaf");
  return 0;
}

}  // namespace dftbhip
