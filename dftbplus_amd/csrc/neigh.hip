// Neighbour list and sparse block descriptor on the device: the half list of
// updateNeighbourList (src/dftbp/dftb/periodic.F90:446-696) and the block offsets of
// getSparseDescriptor (src/dftbp/dftb/sparse2dense.F90:3617-3662), in the order the host
// builder and the reference produce.
//
//   candidate images (translation t, atom a) -> index t * nat + a, binned on a grid of cells of
//   one cutoff over the atoms' bounding box grown by the cutoff (counting sort, positions
//   stored in cell order);
//   one workgroup per central atom counts the candidates of the 27 surrounding cells with
//   a >= atom and d^2 <= cutoff^2, then a second pass collects them in LDS and sorts them by
//   (d^2, index): the index order is (translation, atom);
//   images in use get numbers after the central atoms by a scan over the candidate index;
//   pairs within the SK cutoff and their block sizes are scanned into the block list.
// Bound by latency (a few MB of candidates); 150 atoms of 341 neighbours each: 0.3 ms, from
// 3.4 ms with a thread per atom, the scans in one workgroup and a host copy between the steps.
//
// Squared distances are formed as the host builder forms them (differences, then a sum of
// squares from x to z, no fused multiply-add), so the sort keys and cutoff tests agree bit
// for bit.
#include <climits>
#include <cmath>

#include "neigh.h"

namespace dftbhip {

constexpr int kNlSortMax = 4096;    // neighbours of one atom sorted in LDS
constexpr int kNlThreads = 512;     // threads of an atom's workgroup
// up to this many neighbours each one's rank is counted (n^2 comparisons, no barriers: 150 atoms
// of 341 take 46 us, collecting them included); more are sorted bitonically (log^2 n barriers,
// 51 us for the same atoms without collecting, but n log^2 n comparisons)
constexpr int kNlRankMax = 1024;
constexpr double kNlMinDist2 = 1.0e-4;   // (0.01 bohr)^2: atoms closer are an input error

void cell_translations(const double* lat, double cutoff, std::vector<double>& tr) {
  tr.assign(3, 0.0);
  if (!lat) return;
  // reciprocal vectors / 2 pi: rows of inv(lat)^T
  const double* a = lat;
  const double det = a[0] * (a[4] * a[8] - a[5] * a[7]) - a[1] * (a[3] * a[8] - a[5] * a[6]) +
                     a[2] * (a[3] * a[7] - a[4] * a[6]);
  double inv[9];
  inv[0] = (a[4] * a[8] - a[5] * a[7]) / det;
  inv[1] = -(a[1] * a[8] - a[2] * a[7]) / det;
  inv[2] = (a[1] * a[5] - a[2] * a[4]) / det;
  inv[3] = -(a[3] * a[8] - a[5] * a[6]) / det;
  inv[4] = (a[0] * a[8] - a[2] * a[6]) / det;
  inv[5] = -(a[0] * a[5] - a[2] * a[3]) / det;
  inv[6] = (a[3] * a[7] - a[4] * a[6]) / det;
  inv[7] = -(a[0] * a[7] - a[1] * a[6]) / det;
  inv[8] = (a[0] * a[4] - a[1] * a[3]) / det;
  int nmax[3];
  for (int i = 0; i < 3; ++i) {
    // row i of inv^T = column i of inv
    const double nr = std::sqrt(inv[i] * inv[i] + inv[3 + i] * inv[3 + i] + inv[6 + i] * inv[6 + i]);
    nmax[i] = (int)std::ceil(cutoff * nr) + 1;
  }
  for (int x = -nmax[0]; x <= nmax[0]; ++x)
    for (int y = -nmax[1]; y <= nmax[1]; ++y)
      for (int z = -nmax[2]; z <= nmax[2]; ++z) {
        if (x == 0 && y == 0 && z == 0) continue;
        for (int c = 0; c < 3; ++c) tr.push_back(x * lat[c] + y * lat[3 + c] + z * lat[6 + c]);
      }
}

struct NlGrid {
  double lo[3], hi[3];
  double cutoff;
  int nbin[3];
};

__device__ __forceinline__ double dist2_xyz(const double* x, const double* y) {
#pragma clang fp contract(off)
  double d2 = 0.0;
  for (int c = 0; c < 3; ++c) {
    const double d = x[c] - y[c];
    d2 += d * d;
  }
  return d2;
}

__device__ __forceinline__ void bin_of(const NlGrid& g, const double* x, int* b) {
  for (int c = 0; c < 3; ++c) {
    const int v = (int)floor((x[c] - (g.lo[c] - g.cutoff)) / g.cutoff);
    b[c] = min(max(v, 0), g.nbin[c] - 1);
  }
}

// Exclusive scan over the threads of a workgroup of NT; total: the sum over all of them
template <int NT>
__device__ __forceinline__ long block_scan(long v, long* total) {
  __shared__ long wsum[NT / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  long x = v;
  for (int o = 1; o < 64; o <<= 1) {
    const long y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  __syncthreads();   // wsum of the scan before
  if (lane == 63) wsum[w] = x;
  __syncthreads();
  long pre = 0, all = 0;
#pragma unroll
  for (int q = 0; q < NT / 64; ++q) {
    if (q < w) pre += wsum[q];
    all += wsum[q];
  }
  *total = all;
  return pre + x - v;
}

// Exclusive scan of f.value(i) (a pair of sums) over n elements in two launches: the sums of
// kScanBlocks tiles at most, then each workgroup adds up the tiles before its own, scans its tile
// and hands f.emit every element's offsets; the last tile writes the totals. One workgroup
// looping over everything took 0.64 ms for the 350000 candidates of 2744 atoms.
constexpr int kScanBlocks = 1024, kScanThreads = 256, kScanEach = 8;
struct Sum2 {
  long a = 0, b = 0;
};

template <typename F>
__global__ __launch_bounds__(kScanThreads) void scan_sums_kernel(F f, long n, long tile,
                                                                 Sum2* sums) {
  Sum2 v;
  const long i1 = min(n, (blockIdx.x + 1) * tile);
  for (long i = blockIdx.x * tile + threadIdx.x; i < i1; i += kScanThreads) {
    const Sum2 x = f.value(i);
    v.a += x.a;
    v.b += x.b;
  }
  Sum2 t;
  block_scan<kScanThreads>(v.a, &t.a);
  block_scan<kScanThreads>(v.b, &t.b);
  if (threadIdx.x == 0) sums[blockIdx.x] = t;
}

template <typename F>
__global__ __launch_bounds__(kScanThreads) void scan_apply_kernel(F f, long n, long tile,
                                                                  const Sum2* sums, long* totA,
                                                                  long* totB) {
  Sum2 v, carry;
  for (int q = threadIdx.x; q < (int)blockIdx.x; q += kScanThreads) {
    v.a += sums[q].a;
    v.b += sums[q].b;
  }
  block_scan<kScanThreads>(v.a, &carry.a);
  block_scan<kScanThreads>(v.b, &carry.b);
  const long i1 = min(n, (blockIdx.x + 1) * tile);
  for (long base = blockIdx.x * tile; base < i1; base += kScanThreads * kScanEach) {
    Sum2 x[kScanEach], mine;
    const long i0 = base + (long)threadIdx.x * kScanEach;
#pragma unroll
    for (int j = 0; j < kScanEach; ++j) {
      if (i0 + j < i1) x[j] = f.value(i0 + j);
      mine.a += x[j].a;
      mine.b += x[j].b;
    }
    Sum2 tot, pre;
    pre.a = carry.a + block_scan<kScanThreads>(mine.a, &tot.a);
    pre.b = carry.b + block_scan<kScanThreads>(mine.b, &tot.b);
#pragma unroll
    for (int j = 0; j < kScanEach; ++j) {
      if (i0 + j < i1) f.emit(i0 + j, x[j], pre);
      pre.a += x[j].a;
      pre.b += x[j].b;
    }
    carry.a += tot.a;
    carry.b += tot.b;
  }
  if (threadIdx.x == 0 && blockIdx.x == gridDim.x - 1) {
    *totA = carry.a;
    *totB = carry.b;
  }
}

template <typename F>
static int scan(hipStream_t s, const F& f, long n, DevBuf<long>& sums, long* totA, long* totB) {
  const long chunk = kScanThreads * kScanEach;
  const long tile = chunk * std::max(1L, (n + chunk * kScanBlocks - 1) / (chunk * kScanBlocks));
  const int nb = (int)std::max(1L, (n + tile - 1) / tile);
  DH_TRY(sums.alloc(2 * kScanBlocks));
  Sum2* q = reinterpret_cast<Sum2*>(sums.p);
  hipLaunchKernelGGL(scan_sums_kernel<F>, dim3(nb), dim3(kScanThreads), 0, s, f, n, tile, q);
  DH_LAUNCH_CHECK();
  hipLaunchKernelGGL(scan_apply_kernel<F>, dim3(nb), dim3(kScanThreads), 0, s, f, n, tile, q,
                     totA, totB);
  DH_LAUNCH_CHECK();
  return 0;
}

// first candidate of each grid cell
struct BinScan {
  const int* count;
  int* start;
  __device__ Sum2 value(long i) const { return {count[i], 0}; }
  __device__ void emit(long i, const Sum2&, const Sum2& pre) const { start[i] = (int)pre.a; }
};

// first neighbour of each atom
struct AtomScan {
  const int* cnt;
  long* start;
  __device__ Sum2 value(long i) const { return {cnt[i], 0}; }
  __device__ void emit(long i, const Sum2&, const Sum2& pre) const { start[i] = pre.a; }
};

// numbers, positions and central atoms of the images in use
struct ImageScan {
  int nat;
  const double *coords, *px;
  const int* used;
  int* rank;
  double* coordsAll;
  int* img2cent;
  __device__ Sum2 value(long i) const { return {used[i], 0}; }
  __device__ void emit(long i, const Sum2& v, const Sum2& pre) const {
    if (i >= nat && !v.a) return;
    const long img = i < nat ? i : nat + pre.a;
    const double* x = i < nat ? coords + 3 * i : px + 3 * i;
    if (i >= nat) rank[i] = (int)pre.a;
    for (int c = 0; c < 3; ++c) coordsAll[3 * img + c] = x[c];
    img2cent[img] = (int)(i % nat);
  }
};

// pairs within the SK cutoff and the sizes of their blocks
struct BlockScan {
  const double* d2;
  const int *at1, *img2, *at2, *norb;
  double sk2;
  int *bAt1, *bImg2, *bAt2;
  long* bStart;
  __device__ Sum2 value(long q) const {
    if (!(d2[q] <= sk2)) return {};
    return {1, (long)norb[at1[q]] * norb[at2[q]]};
  }
  __device__ void emit(long q, const Sum2& v, const Sum2& pre) const {
    if (!v.a) return;
    bAt1[pre.a] = at1[q];
    bImg2[pre.a] = img2[q];
    bAt2[pre.a] = at2[q];
    bStart[pre.a] = pre.b;
  }
};

__global__ void nl_points_kernel(int nat, long P, const double* coords, const double* tr,
                                 NlGrid g, double* px, int* pbin, int* prank, int* binCount) {
  const long pi = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (pi >= P) return;
  const int t = (int)(pi / nat), a = (int)(pi - (long)t * nat);
  double x[3];
  bool in = true;
  for (int c = 0; c < 3; ++c) {
    x[c] = coords[3 * a + c] + tr[3 * t + c];
    if (x[c] < g.lo[c] - g.cutoff || x[c] > g.hi[c] + g.cutoff) in = false;
    px[3 * pi + c] = x[c];
  }
  int bin = -1;
  if (in) {
    int b[3];
    bin_of(g, x, b);
    bin = (b[0] * g.nbin[1] + b[1]) * g.nbin[2] + b[2];
    prank[pi] = atomicAdd(&binCount[bin], 1);
  }
  pbin[pi] = bin;
}

__global__ void nl_scatter_kernel(long P, const int* pbin, const int* prank,
                                  const double* px, const int* binStart, int* binItems,
                                  double* binX) {
  const long pi = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (pi >= P) return;
  const int b = pbin[pi];
  if (b < 0) return;
  const long q = binStart[b] + prank[pi];
  binItems[q] = (int)pi;
  for (int c = 0; c < 3; ++c) binX[3 * q + c] = px[3 * pi + c];
}

// hit(d^2, candidate) for this thread's share of the candidates of central atom a2 within the
// cutoff, close(a) for atoms too close to it. The cells of one (x, y) are neighbours in the cell
// order, so the 27 cells are nine runs of candidates.
template <typename Hit, typename Close>
__device__ __forceinline__ void nl_visit(int a2, int nat, const NlGrid& g, const double* coords,
                                         const int* binStart, const int* binCount,
                                         const int* binItems, const double* binX, double cut2,
                                         Hit hit, Close close) {
  double c2[3];
  for (int c = 0; c < 3; ++c) c2[c] = coords[3 * a2 + c];
  int b[3];
  bin_of(g, c2, b);
  int start[9], pre[10];
  pre[0] = 0;
#pragma unroll
  for (int r = 0; r < 9; ++r) {
    const int bx = b[0] + r / 3 - 1, by = b[1] + r % 3 - 1;
    start[r] = 0;
    int len = 0;
    if (bx >= 0 && by >= 0 && bx < g.nbin[0] && by < g.nbin[1]) {
      const int row = (bx * g.nbin[1] + by) * g.nbin[2];
      const int z0 = max(b[2] - 1, 0), z1 = min(b[2] + 1, g.nbin[2] - 1);
      start[r] = binStart[row + z0];
      len = binStart[row + z1] + binCount[row + z1] - start[r];
    }
    pre[r + 1] = pre[r] + len;
  }
  for (int u = threadIdx.x; u < pre[9]; u += kNlThreads) {
    int q = start[0] + u;
#pragma unroll
    for (int r = 1; r < 9; ++r)
      if (u >= pre[r]) q = start[r] + u - pre[r];
    const int pi = binItems[q];
    const double d2 = dist2_xyz(binX + 3 * (long)q, c2);
    if (!(d2 <= cut2)) continue;   // nor has one that is no number
    const int t = pi / nat, a = pi - t * nat;
    if (a < a2) continue;
    if (d2 < kNlMinDist2) {
      if (t != 0 || a != a2) close(a);
      continue;
    }
    hit(d2, pi);
  }
}

// candidates of each central atom, one workgroup each; err: a pair of atoms too close
__global__ __launch_bounds__(kNlThreads) void nl_count_kernel(int nat, NlGrid g,
                                                              const double* coords,
                                                              const int* binStart,
                                                              const int* binCount,
                                                              const int* binItems,
                                                              const double* binX, double cut2,
                                                              int* cnt, int* err) {
  __shared__ int total;
  const int a2 = blockIdx.x;
  if (threadIdx.x == 0) total = 0;
  __syncthreads();
  int k = 0;
  nl_visit(
      a2, nat, g, coords, binStart, binCount, binItems, binX, cut2, [&](double, int) { ++k; },
      [&](int a) {
        if (atomicCAS(&err[0], 0, 1) == 0) {
          err[1] = a + 1;
          err[2] = a2 + 1;
        }
      });
  if (k) atomicAdd(&total, k);
  __syncthreads();
  if (threadIdx.x == 0) {
    cnt[a2] = total;
    atomicMax(&err[3], total);
  }
}

// one workgroup per central atom: its candidates sorted by (d^2, candidate index) in LDS;
// candidates of other cells (index >= nat) are marked used
__global__ __launch_bounds__(kNlThreads) void nl_sort_kernel(int nat, NlGrid g,
                                                             const double* coords,
                                                             const int* binStart,
                                                             const int* binCount,
                                                             const int* binItems,
                                                             const double* binX, double cut2,
                                                             const long* fStart, double* fD2,
                                                             int* fPi, int* used) {
  __shared__ double kd[kNlSortMax];
  __shared__ int kp[kNlSortMax];
  __shared__ int total;
  const int a2 = blockIdx.x;
  if (threadIdx.x == 0) total = 0;
  __syncthreads();
  nl_visit(
      a2, nat, g, coords, binStart, binCount, binItems, binX, cut2,
      [&](double d2, int pi) {
        const int k = atomicAdd(&total, 1);
        if (k < kNlSortMax) {   // more are refused by the host before this launch
          kd[k] = d2;
          kp[k] = pi;
        }
      },
      [](int) {});
  __syncthreads();
  const int n = min(total, kNlSortMax);
  const long o = fStart[a2];
  if (n <= kNlRankMax) {
    for (int i = threadIdx.x; i < n; i += kNlThreads) {
      const double d = kd[i];
      const int p = kp[i];
      int rank = 0;
#pragma unroll 8
      for (int j = 0; j < n; ++j) {   // no branches: all lanes read the same element
        const double dj = kd[j];
        const int pj = kp[j];
        rank += (int)(dj < d) | ((int)(dj == d) & (int)(pj < p));
      }
      fD2[o + rank] = d;
      fPi[o + rank] = p;
      if (p >= nat) used[p] = 1;
    }
    return;
  }
  int N2 = 1;
  while (N2 < n) N2 <<= 1;
  for (int i = n + threadIdx.x; i < N2; i += kNlThreads) {
    kd[i] = INFINITY;
    kp[i] = INT_MAX;
  }
  __syncthreads();
  for (int k = 2; k <= N2; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = threadIdx.x; i < N2; i += kNlThreads) {
        const int l = i ^ j;
        if (l > i) {
          const bool gt = kd[i] > kd[l] || (kd[i] == kd[l] && kp[i] > kp[l]);
          if (gt == ((i & k) == 0)) {
            const double td = kd[i];
            kd[i] = kd[l];
            kd[l] = td;
            const int tp = kp[i];
            kp[i] = kp[l];
            kp[l] = tp;
          }
        }
      }
      __syncthreads();
    }
  for (int i = threadIdx.x; i < n; i += kNlThreads) {
    fD2[o + i] = kd[i];
    fPi[o + i] = kp[i];
    if (kp[i] >= nat) used[kp[i]] = 1;
  }
}

__global__ void nl_pairs_kernel(int nat, const int* cnt, const long* fStart, const double* fD2,
                                const int* fPi, const int* imgRank, int* pAt1, int* pImg2,
                                int* pAt2, double* pD2, int* pCount, long* pStart) {
  const int a2 = blockIdx.x;
  const long o = fStart[a2], base = o + a2;
  const int n = cnt[a2];
  if (threadIdx.x == 0) {
    pAt1[base] = a2;
    pImg2[base] = a2;
    pAt2[base] = a2;
    pD2[base] = 0.0;
    pCount[a2] = n;
    pStart[a2] = base;
    if (a2 == nat - 1) pStart[nat] = base + 1 + n;
  }
  for (int j = threadIdx.x; j < n; j += blockDim.x) {
    const int pi = fPi[o + j];
    const int t = pi / nat, a = pi - t * nat;
    const long q = base + 1 + j;
    pAt1[q] = a2;
    pImg2[q] = t == 0 ? a : nat + imgRank[pi];
    pAt2[q] = a;
    pD2[q] = fD2[o + j];
  }
}

struct Inv9 {
  double v[9];
};

// integer cell translation of each block's image: rint((r_img - r_centre) L^-1)
__global__ void nl_block_translations_kernel(int nBlk, const int* img2, const int* at2,
                                             const double* coordsAll, const double* coords,
                                             Inv9 inv, double* T) {
#pragma clang fp contract(off)
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nBlk) return;
  const int img = img2[k], jc = at2[k];
  double d[3];
  for (int q = 0; q < 3; ++q) d[q] = coordsAll[3 * (long)img + q] - coords[3 * (long)jc + q];
  for (int q = 0; q < 3; ++q)
    T[3 * (long)k + q] = rint(d[0] * inv.v[q] + d[1] * inv.v[3 + q] + d[2] * inv.v[6 + q]);
}

int block_translations(hipStream_t s, int nBlk, const int* img2, const int* at2,
                       const double* coordsAll, const double* coords, const double* inv,
                       double* T) {
  if (nBlk <= 0) return 0;
  Inv9 iv;
  for (int q = 0; q < 9; ++q) iv.v[q] = inv[q];
  hipLaunchKernelGGL(nl_block_translations_kernel, dim3(cdiv(nBlk, 256)), dim3(256), 0, s, nBlk,
                     img2, at2, coordsAll, coords, iv, T);
  DH_LAUNCH_CHECK();
  return 0;
}

int device_neighbours(hipStream_t s, int nat, const double* coords, const double* lat,
                      double cutoff, double skcut, const int* norb, DevNeighbourList& nl) {
  DH_CHECK(nat >= 1 && coords && norb && cutoff > 0.0 && skcut <= cutoff,
           "neighbour list: bad arguments");
  // a distance that is no number has no place in the sorted lists
  for (int k = 0; k < 3 * nat; ++k)
    if (!std::isfinite(coords[k])) {
      set_error("neighbour list: coordinates of atom " + std::to_string(k / 3 + 1) +
                " are not finite");
      return kErrArg;
    }
  for (int k = 0; lat && k < 9; ++k)
    DH_CHECK(std::isfinite(lat[k]), "neighbour list: lattice vectors are not finite");
  std::vector<double> tr;
  cell_translations(lat, cutoff, tr);
  for (double x : tr)
    DH_CHECK(std::isfinite(x), "neighbour list: lattice vectors out of range");
  const long ntr = (long)tr.size() / 3;
  const long P = ntr * nat;
  DH_CHECK(P < INT_MAX / 2, "neighbour list: too many candidate images");
  NlGrid g;
  g.cutoff = cutoff;
  for (int c = 0; c < 3; ++c) {
    g.lo[c] = 1e300;
    g.hi[c] = -1e300;
  }
  for (int a = 0; a < nat; ++a)
    for (int c = 0; c < 3; ++c) {
      g.lo[c] = std::min(g.lo[c], coords[3 * a + c]);
      g.hi[c] = std::max(g.hi[c], coords[3 * a + c]);
    }
  long nbins = 1;
  for (int c = 0; c < 3; ++c) {
    g.nbin[c] = std::max(1, (int)std::floor((g.hi[c] - g.lo[c] + 2 * cutoff) / cutoff));
    nbins *= g.nbin[c];
  }
  DH_CHECK(nbins < INT_MAX / 2, "neighbour list: too many grid cells");
  nl.nat = nat;
  DH_TRY(nl.coordsD.upload(coords, 3 * (size_t)nat, s));
  DH_TRY(nl.trD.upload(tr.data(), tr.size(), s));
  DH_TRY(nl.norbD.upload(norb, nat, s));
  DH_TRY(nl.px.alloc(3 * (size_t)P));
  DH_TRY(nl.binX.alloc(3 * (size_t)P));
  DH_TRY(nl.pbin.alloc(P));
  DH_TRY(nl.binItems.alloc(P));
  DH_TRY(nl.binCount.alloc(nbins));
  DH_TRY(nl.binStart.alloc(nbins));
  DH_TRY(nl.prank.alloc(P));
  DH_TRY(nl.err.alloc(4));
  DH_TRY(nl.scal.alloc(6));
  DH_TRY(nl.cnt.alloc(nat));
  DH_TRY(nl.fStart.alloc(nat));
  DH_TRY(nl.used.alloc(P));
  DH_TRY(nl.imgRank.alloc(P));
  DH_TRY(fill<int>(s, nl.binCount.p, nbins, 0));
  DH_TRY(fill<int>(s, nl.err.p, 4, 0));
  DH_TRY(fill<int>(s, nl.used.p, P, 0));
  long* sc = nl.scal.p;   // totals of the scans
  // candidates into grid cells
  hipLaunchKernelGGL(nl_points_kernel, dim3(cdiv(P, 256)), dim3(256), 0, s, nat, P, nl.coordsD.p,
                     nl.trD.p, g, nl.px.p, nl.pbin.p, nl.prank.p, nl.binCount.p);
  DH_LAUNCH_CHECK();
  DH_TRY(scan(s, BinScan{nl.binCount.p, nl.binStart.p}, nbins, nl.sums, sc, sc + 5));
  hipLaunchKernelGGL(nl_scatter_kernel, dim3(cdiv(P, 256)), dim3(256), 0, s, P, nl.pbin.p,
                     nl.prank.p, nl.px.p, nl.binStart.p, nl.binItems.p, nl.binX.p);
  DH_LAUNCH_CHECK();
  // neighbours per central atom, their offsets
  const double cut2 = cutoff * cutoff;
  hipLaunchKernelGGL(nl_count_kernel, dim3(nat), dim3(kNlThreads), 0, s, nat, g, nl.coordsD.p,
                     nl.binStart.p, nl.binCount.p, nl.binItems.p, nl.binX.p, cut2, nl.cnt.p,
                     nl.err.p);
  DH_LAUNCH_CHECK();
  DH_TRY(scan(s, AtomScan{nl.cnt.p, nl.fStart.p}, nat, nl.sums, sc + 1, sc + 5));
  long F = 0;
  {
    int err[4];
    DH_HIP(hipMemcpyAsync(&F, sc + 1, sizeof(F), hipMemcpyDeviceToHost, s));
    DH_HIP(hipMemcpyAsync(err, nl.err.p, sizeof(err), hipMemcpyDeviceToHost, s));
    DH_HIP(hipStreamSynchronize(s));
    if (err[0]) {
      set_error("Atoms " + std::to_string(err[1]) + " and " + std::to_string(err[2]) +
                " too close together");
      return kErrArg;
    }
    nl.maxNeighbour = err[3];
    if (nl.maxNeighbour > kNlSortMax) {
      set_error("neighbour list: an atom has " + std::to_string(nl.maxNeighbour) +
                " neighbours, more than " + std::to_string(kNlSortMax));
      return kErrArg;
    }
  }
  DH_TRY(nl.fD2.alloc(std::max<long>(F, 1)));
  DH_TRY(nl.fPi.alloc(std::max<long>(F, 1)));
  hipLaunchKernelGGL(nl_sort_kernel, dim3(nat), dim3(kNlThreads), 0, s, nat, g, nl.coordsD.p,
                     nl.binStart.p, nl.binCount.p, nl.binItems.p, nl.binX.p, cut2, nl.fStart.p,
                     nl.fD2.p, nl.fPi.p, nl.used.p);
  DH_LAUNCH_CHECK();
  // images: at most one per neighbour and per candidate
  const long maxAll = nat + std::min(F, P - nat);
  DH_TRY(nl.coordsAll.alloc(3 * (size_t)maxAll));
  DH_TRY(nl.img2cent.alloc(maxAll));
  DH_TRY(scan(s, ImageScan{nat, nl.coordsD.p, nl.px.p, nl.used.p, nl.imgRank.p, nl.coordsAll.p,
                           nl.img2cent.p},
              P, nl.sums, sc + 2, sc + 5));
  // pairs, self first per atom
  nl.nPairs = (int)(F + nat);
  DH_TRY(nl.pAt1.alloc(nl.nPairs));
  DH_TRY(nl.pImg2.alloc(nl.nPairs));
  DH_TRY(nl.pAt2.alloc(nl.nPairs));
  DH_TRY(nl.pD2.alloc(nl.nPairs));
  DH_TRY(nl.pCount.alloc(nat));
  DH_TRY(nl.pStart.alloc(nat + 1));
  hipLaunchKernelGGL(nl_pairs_kernel, dim3(nat), dim3(256), 0, s, nat, nl.cnt.p,
                     nl.fStart.p, nl.fD2.p, nl.fPi.p, nl.imgRank.p, nl.pAt1.p, nl.pImg2.p,
                     nl.pAt2.p, nl.pD2.p, nl.pCount.p, nl.pStart.p);
  DH_LAUNCH_CHECK();
  // blocks within the SK cutoff and their offsets
  DH_TRY(nl.bAt1.alloc(nl.nPairs));
  DH_TRY(nl.bImg2.alloc(nl.nPairs));
  DH_TRY(nl.bAt2.alloc(nl.nPairs));
  DH_TRY(nl.bStart.alloc(nl.nPairs));
  DH_TRY(scan(s, BlockScan{nl.pD2.p, nl.pAt1.p, nl.pImg2.p, nl.pAt2.p, nl.norbD.p, skcut * skcut,
                           nl.bAt1.p, nl.bImg2.p, nl.bAt2.p, nl.bStart.p},
              nl.nPairs, nl.sums, sc + 3, sc + 4));
  long tot[3];
  DH_HIP(hipMemcpyAsync(tot, sc + 2, sizeof(tot), hipMemcpyDeviceToHost, s));
  DH_HIP(hipStreamSynchronize(s));
  nl.nAll = nat + (int)tot[0];
  nl.nBlk = (int)tot[1];
  nl.nnz = tot[2];
  return 0;
}

}  // namespace dftbhip
