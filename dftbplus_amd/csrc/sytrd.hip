// Householder tridiagonalisation of a real symmetric matrix (lower storage) and the
// back-transformation of eigenvectors, one-stage blocked form:
//
//   for each panel of kNB columns:
//     for each column c: update column c with the panel's V W^T + W V^T;
//                        form the reflector (alpha, ||x||) -> (beta, tau, 1/(alpha-beta));
//                        w = tau * (A22 v - V (W^T v) - W (V^T v)),  w += -tau/2 (w.v) v;
//     trailing update A22 -= [V W] [W V]^T on the MFMA GEMM (lower tiles).
//
// The symmetric product A22 v reads only the lower triangle: each workgroup takes an equal run of
// its 64 x 64 tiles; row-block partial sums and transposed-tile partial sums go to workspaces that
// the next kernel reduces (no atomics on the vector). This product is the HBM-bound part of the
// eigensolver (it streams the trailing matrix once per column).
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "symv_table.h"
#include "tri_inverse.h"

namespace dftbhip {

constexpr int kNB = 64;      // panel width
// Panel products t1 = W^T v, t2 = V^T v of the column being reduced: one 128-byte line per entry
// (the SYMV's workgroups add into them atomically; entries sharing a line would serialize those
// atomics) and two columns in a ring, the next column's entries cleared by col_update.
constexpr int kT12Pad = 16;
__host__ __device__ inline long t12_at(int c, int p) {
  return ((long)(c & 1) * 2 * kNB + p) * kT12Pad;
}
constexpr long kT12Size = 2L * 2 * kNB * kT12Pad;

// Optional per-launch timing of the symmetric product kernel (HIP events on the launch stream):
// launches, summed duration and the algorithmic bytes (lower triangle of the trailing matrix).
struct SymvProfile {
  bool on = false;
  std::vector<hipEvent_t> ev;
  std::vector<double> bytes;
  std::vector<int> size;   // trailing size m of each recorded launch
  size_t used = 0;
  double launches = 0, seconds = 0, algBytes = 0;
  std::vector<std::pair<int, float>>* sink = nullptr;   // (m, ms) per launch, when set
};
static SymvProfile g_symvProf;

void symv_profiling(bool on) {
  g_symvProf.on = on;
  g_symvProf.launches = g_symvProf.seconds = g_symvProf.algBytes = 0;
}

void symv_profile_stats(double* out) {
  out[0] = g_symvProf.launches;
  out[1] = g_symvProf.seconds;
  out[2] = g_symvProf.algBytes;
}

static int symv_prof_collect(hipStream_t s) {
  SymvProfile& p = g_symvProf;
  if (!p.on || p.used == 0) return 0;
  DH_HIP(hipStreamSynchronize(s));
  for (size_t i = 0; i < p.used; ++i) {
    float ms = 0.f;
    DH_HIP(hipEventElapsedTime(&ms, p.ev[2 * i], p.ev[2 * i + 1]));
    p.seconds += ms * 1e-3;
    p.algBytes += p.bytes[i];
    if (p.sink) p.sink->push_back({p.size[i], ms});
    p.launches += 1;
  }
  p.used = 0;
  return 0;
}
constexpr int kTB = 64;      // SYMV tile
constexpr int kCHMin = 2;    // fewest tiles per SYMV workgroup (sizes the slot array)
// SYMV workgroups that are resident together (two on each of 256 compute units): the tiles of
// all problems are shared out to as many, so that there is one round and no last, half empty one
constexpr int kSymvSlots = 512;
// tiles per SYMV workgroup (2, 4, 8 or 16; 0: the tiles shared out evenly), set through
// set_symv_tiles
static int g_symvTiles = 0;
// bumped whenever the tile choice changes: captured launch sequences (below) are only replayed
// while it is unchanged
static unsigned g_tileGen = 0;

int set_symv_tiles(int tiles) {
  DH_CHECK(tiles == 0 || tiles == 2 || tiles == 4 || tiles == 8 || tiles == 16,
           "symv tiles must be 0 (by size), 2, 4, 8 or 16");
  g_symvTiles = tiles;
  ++g_tileGen;
  return 0;
}

// Tile choice by trailing size from the autotuner (symv_autotune), per arithmetic type
// ([0] FP64, [1] FP32): rows (first trailing size, tiles) in ascending size; empty, or 0 tiles:
// shared out evenly.
static TileTable g_tileTable[2];

int clear_symv_tables() {
  g_tileTable[0].clear();
  g_tileTable[1].clear();
  ++g_tileGen;
  return 0;
}

// Tiles per SYMV workgroup for K problems of trailing size m
template <typename T>
static int symv_tiles(int m, int K) {
  if (g_symvTiles != 0) return g_symvTiles;
  const auto& t = g_tileTable[std::is_same<T, float>::value ? 1 : 0];
  if (!t.empty()) {
    const int mk = (int)std::min<long>((long)m * K, 1L << 30);
    int v = t.front().second;
    for (const auto& r : t)
      if (mk >= r.first) v = r.second;
    if (v > 0) return v;
  }
  const long nRB = (m + kTB - 1) / kTB, all = nRB * (nRB + 1) / 2 * K;
  return (int)std::max<long>(kCHMin, (all + kSymvSlots - 1) / kSymvSlots);
}

// The lower tiles of nRB row blocks in the order of their columns: column J's start at
// symv_first(J); a workgroup takes q tiles in a row, so column J is worked out in
// symv_pieces(J) pieces.
__host__ __device__ inline int symv_first(int nRB, int J) { return J * nRB - J * (J - 1) / 2; }
__device__ inline int symv_pieces(int nRB, int J, int q) {
  const int t = symv_first(nRB, J);
  return (t + nRB - J - 1) / q - t / q + 1;
}

template <typename T>
struct SytrdWs {
  T* W;            // n x kNB
  T* Y;            // nSlot x n   partial sums of A22 v, slot-major: Y(row, slot) at slot n + row
  T* vbuf;         // n
  double* nrm2;    // n   ||x||^2 per column
  double* dot;     // n   w.v per column (before the rank-one correction of w)
  double* t12;     // panel products, see t12_at
  double* scal;    // n
  T* P;            // n x 2kNB
  T* Q;            // n x 2kNB
  int nSlot;
};

static int sytrd_slots(int n) {
  const int nRB = (n + kTB - 1) / kTB;
  // a column of tiles is worked out in at most half as many pieces, rounded up
  return nRB + (nRB + kCHMin - 1) / kCHMin;
}

// byte layout of the workspace (each array 256-byte aligned)
template <typename T>
static size_t sytrd_layout(int n, SytrdWs<T>* ws, char* base) {
  size_t off = 0;
  auto take = [&](auto** p, size_t bytes) {
    if (ws) *p = reinterpret_cast<std::remove_reference_t<decltype(**p)>*>(base + off);
    off += (bytes + 255) / 256 * 256;
  };
  SytrdWs<T> dummy;
  SytrdWs<T>* w = ws ? ws : &dummy;
  w->nSlot = sytrd_slots(n);
  take(&w->W, sizeof(T) * n * kNB);
  take(&w->Y, sizeof(T) * n * w->nSlot);
  take(&w->vbuf, sizeof(T) * n);
  take(&w->nrm2, sizeof(double) * n);
  take(&w->dot, sizeof(double) * n);
  take(&w->t12, sizeof(double) * kT12Size);
  take(&w->scal, sizeof(double) * n);
  take(&w->P, sizeof(T) * n * 2 * kNB);
  take(&w->Q, sizeof(T) * n * 2 * kNB);
  return off;
}

// workspace bytes
size_t sytrd_work_bytes(int n, int elemSize) {
  return elemSize == 8 ? sytrd_layout<double>(n, nullptr, nullptr)
                       : sytrd_layout<float>(n, nullptr, nullptr);
}
size_t sytrd_work_size(int n) { return (sytrd_work_bytes(n, 8) + 7) / 8; }

// Several problems of one size in one launch: problem blockIdx.z finds its matrix, workspace
// block and vectors at these strides from those of problem 0 (all zero for a single problem).
struct ProblemStrides {
  long a;    // matrix elements
  long ws;   // workspace bytes
  long v;    // elements of d, e, tau
};

template <typename P>
__device__ __forceinline__ P* ws_of(P* p, long bytes) {
  return (P*)((const char*)p + (long)blockIdx.z * bytes);
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}

// Reflector constants of column c from alpha = A(c+1,c) and ||x||^2 (LAPACK dlarfg without the
// rescaling loop): beta = -sign(alpha) sqrt(alpha^2 + ||x||^2), tau = (beta - alpha)/beta,
// x scale = 1/(alpha - beta).
__device__ __forceinline__ void reflector(double alpha, double xn2, double& beta, double& tau,
                                          double& scal) {
  if (xn2 == 0.0) {
    beta = alpha;
    tau = 0.0;
    scal = 0.0;
    return;
  }
  const double nrm = sqrt(alpha * alpha + xn2);
  beta = alpha >= 0.0 ? -nrm : nrm;
  tau = (beta - alpha) / beta;
  scal = 1.0 / (alpha - beta);
}

// W stores w before its rank-one correction: the true column p of the panel is
// W(:,p) + alpha_p V(:,p) with alpha_p = -tau_p (w_p . v_p) / 2, applied by every reader.
template <typename T>
__device__ __forceinline__ double wcorr(int cp, const T* tau, const double* dot) {
  return -0.5 * (double)tau[cp] * dot[cp];
}

// A(r,c) -= sum_p V(r,p) W(c,p) + W(r,p) V(c,p), rows r >= c; accumulate ||A(c+2:n,c)||^2.
// A block handles 64 rows (the lanes); wave g takes the reflectors p = 16 g .. 16 g + 15 with
// all their loads in one batch, and the four partial sums meet in LDS.
template <typename T>
__global__ __launch_bounds__(256) void col_update_kernel(T* a, long lda, int n, int c, int j0,
                                                         const T* W, long ldw, const T* tau,
                                                         const double* dot, double* nrm2,
                                                         double* t12, ProblemStrides ps) {
  __shared__ double vc[kNB], wc[kNB], al[kNB], part[4][64];
  a += (long)blockIdx.z * ps.a;
  tau += (long)blockIdx.z * ps.v;
  W = ws_of(W, ps.ws);
  dot = ws_of(dot, ps.ws);
  nrm2 = ws_of(nrm2, ps.ws);
  t12 = ws_of(t12, ps.ws);
  const int i = c - j0;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (threadIdx.x < i) {
    const int p = threadIdx.x;
    al[p] = wcorr(j0 + p, tau, dot);
    vc[p] = a[c + (long)(j0 + p) * lda];
    wc[p] = W[c + (long)p * ldw] + al[p] * vc[p];
  }
  // the panel products of column c + 1 start from zero (their ring entry was column c - 1's,
  // whose readers have finished)
  if (blockIdx.x == 0)
    for (int e = threadIdx.x; e < 2 * kNB; e += blockDim.x) t12[t12_at(c + 1, e)] = 0.0;
  __syncthreads();
  const int r = c + blockIdx.x * 64 + lane;
  double d = 0.0;
  const int p0 = 16 * wv;
  if (r < n && p0 < i) {
    double vr[16], wr[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      vr[q] = 0.0;
      wr[q] = 0.0;
      if (p0 + q < i) {
        vr[q] = a[r + (long)(j0 + p0 + q) * lda];
        wr[q] = W[r + (long)(p0 + q) * ldw];
      }
    }
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int p = p0 + q;
      if (p < i) d += vr[q] * wc[p] + (wr[q] + al[p] * vr[q]) * vc[p];
    }
  }
  part[wv][lane] = d;
  __syncthreads();
  if (wv == 0) {
    double sq = 0.0;
    if (r < n) {
      double v = a[r + (long)c * lda] - ((part[0][lane] + part[1][lane]) +
                                         (part[2][lane] + part[3][lane]));
      a[r + (long)c * lda] = (T)v;
      v = (double)(T)v;
      if (r >= c + 2) sq = v * v;
    }
    const double tot = wave_sum(sq);
    if (lane == 0 && tot != 0.0) atomicAdd(&nrm2[c], tot);
  }
}

// Sum of each z[0..15] over the wave, in 17 exchanges instead of 96: every step adds the halves of
// the array that two lanes exchange. Lane l returns the sum of z[l & 15].
template <int H, typename T>
__device__ __forceinline__ void fold_halves(T (&z)[16], int lane) {
  const bool up = lane & H;
#pragma unroll
  for (int e = 0; e < H; ++e) {
    const T send = up ? z[e] : z[e + H], keep = up ? z[e + H] : z[e];
    z[e] = keep + __shfl_xor(send, H, 64);
  }
}
template <typename T>
__device__ __forceinline__ T wave_sum16(T (&z)[16], int lane) {
  fold_halves<8>(z, lane);
  fold_halves<4>(z, lane);
  fold_halves<2>(z, lane);
  fold_halves<1>(z, lane);
  T v = z[0];
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}

// Partial sums of y = A22 v (A22 = a(c+1:n, c+1:n), lower triangle read once).
// The first nRB workgroups take a row block each: they publish v and add up the panel products
// t1, t2. Workgroup nRB + w takes the tiles w q .. w q + q - 1 of the lower triangle, column by
// column, the next two tiles on the way while one is worked on; the first two are requested
// before the reflector of the column is formed.
//   y partial of tile (I, J)       -> Y(row, J)          (reduced over 4 waves)
//   transposed sums (A^T v)_J      -> Y(col, nRB + piece) (in registers over the column's tiles)
// Thread (ii = tid % 64, cg = tid / 64) holds rows ii of 16 columns cg*16 .. cg*16+15.
// Bound by the stream of the trailing triangle: 22 us on average over trailing sizes 2560 to 6656
// (4.1 TB/s), 29 us with fixed chunks of a column per workgroup, whose last round was partly
// empty, and the panel products ahead of the first tile of some of them.
template <typename T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void symv_kernel(
    const T* a, long lda, int n, int c, int j0, const T* W, long ldw, const double* nrm2,
    const T* tauA, const double* dotA, T* Y, T* vbuf, double* t12, double* scalOut, T* eOut,
    T* tauOut, int q, ProblemStrides ps) {
  __shared__ T vJs[kTB];
  __shared__ T red[4][4][kTB];
  a += (long)blockIdx.z * ps.a;
  tauA += (long)blockIdx.z * ps.v;
  eOut += (long)blockIdx.z * ps.v;
  tauOut += (long)blockIdx.z * ps.v;
  W = ws_of(W, ps.ws);
  nrm2 = ws_of(nrm2, ps.ws);
  dotA = ws_of(dotA, ps.ws);
  Y = ws_of(Y, ps.ws);
  vbuf = ws_of(vbuf, ps.ws);
  t12 = ws_of(t12, ps.ws);
  scalOut = ws_of(scalOut, ps.ws);
  const int m = n - c - 1;
  const int nRB = (m + kTB - 1) / kTB;
  const int tid = threadIdx.x;
  const int ii = tid & 63, cg = __builtin_amdgcn_readfirstlane(tid >> 6);
  const T* const col = a + (c + 1) + (long)c * lda;   // the column's elements below the diagonal
  const double alpha = col[0], xn2 = nrm2[c];
  double beta, tau, scal;
  if ((int)blockIdx.x < nRB) {
    reflector(alpha, xn2, beta, tau, scal);
    if (blockIdx.x == 0 && tid == 0) {
      scalOut[c] = scal;
      eOut[c] = (T)beta;
      tauOut[c] = (T)tau;
    }
    const int k = blockIdx.x * kTB + ii, r = c + 1 + k;
    const bool rowOk = k < m;
    const T v = !rowOk ? T(0) : (k == 0 ? T(1) : (T)((double)col[k] * scal));
    if (cg == 0 && rowOk) vbuf[r] = v;
    // panel products over this block's rows: t12[p] += W(:, p)^T v, t12[i + p] += V(:, p)^T v
    // for p < i (wave cg takes p = cg + 4 e). All loads are issued before the reductions and
    // atomics, which would otherwise order every load behind the previous atomic.
    const int i = c - j0;
    const double vv = (double)v;
    double pw[kNB / 4], pv[kNB / 4];
    static_assert(kNB / 4 == 16, "wave_sum16");
#pragma unroll
    for (int e = 0; e < kNB / 4; ++e) {
      const int p = cg + 4 * e;
      pw[e] = 0.0;
      pv[e] = 0.0;
      if (p < i && rowOk) {
        const double vr = a[r + (long)(j0 + p) * lda];
        pv[e] = vr * vv;
        pw[e] = ((double)W[r + (long)p * ldw] + wcorr(j0 + p, tauA, dotA) * vr) * vv;
      }
    }
    const double sw = wave_sum16(pw, ii), sv = wave_sum16(pv, ii);
    const int p = cg + 4 * (ii & 15);
    if (ii < 16 && p < i) {
      if (sw != 0.0) atomicAdd(&t12[t12_at(c, p)], sw);
      if (sv != 0.0) atomicAdd(&t12[t12_at(c, i + p)], sv);
    }
    return;
  }
  const int w = blockIdx.x - nRB;
  const int t0 = w * q, t1 = min(t0 + q, nRB * (nRB + 1) / 2);
  if (t0 >= t1) return;
  // column of the first tile
  int J = (int)(0.5 * (2 * nRB + 1 - sqrt((double)(2 * nRB + 1) * (2 * nRB + 1) - 8.0 * t0)));
  J = min(max(J, 0), nRB - 1);
  while (symv_first(nRB, J) > t0) --J;
  while (J + 1 < nRB && symv_first(nRB, J + 1) <= t0) ++J;
  int I = J + t0 - symv_first(nRB, J);
  int lI = I, lJ = J, left = t1 - t0;   // next tile to request
  T b0[16], b1[16], b2[16], zacc[16];
  T v0 = T(0), v1 = T(0), v2 = T(0), u0 = T(0), u1 = T(0), u2 = T(0);
#pragma unroll
  for (int e = 0; e < 16; ++e) zacc[e] = T(0);
  // rows ii of the tile's 16 columns, v of row ii and of column ii & 15 (raw column-c elements,
  // scaled at use so that the request is not waited on). Rows and columns past the end and the
  // upper triangle of a diagonal tile are read at the nearest place that exists and masked at
  // their use.
  auto load = [&](T(&dst)[16], T& vdst, T& udst) __attribute__((always_inline)) {
    const int gr = min(lI * kTB + ii, m - 1), gc0 = lJ * kTB + cg * 16;
#pragma unroll
    for (int e = 0; e < 16; ++e) dst[e] = (col + (long)(1 + min(gc0 + e, m - 1)) * lda)[gr];
    vdst = col[gr];
    udst = col[min(gc0 + (ii & 15), m - 1)];
    // past the run's last tile the requests repeat it (in the caches) instead of branching
    if (--left > 0) {
      const bool next = lI + 1 == nRB;
      lJ += next;
      lI = next ? lJ : lI + 1;
    }
  };
  load(b0, v0, u0);
  load(b1, v1, u1);
  reflector(alpha, xn2, beta, tau, scal);
  T* vj = vJs + cg * 16;   // v of this wave's 16 columns
  bool fresh = true;       // the next tile is the first of its column here
  // barrier for the LDS row sums only: __syncthreads would also wait for the prefetched global
  // loads of the next tiles (its workgroup fence waits on every outstanding memory operation)
  auto lds_barrier = [&]() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0); vmcnt, expcnt untouched (gfx9 encoding)
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  };
  int k = 0, pI = 0, pJ = 0;   // tiles done; the tile before
  // one tile: row partials (reduced over the 4 waves through LDS) and transposed sums
  auto tile = [&](const T(&t)[16], T vraw, T uraw) __attribute__((always_inline)) {
    const int gr = I * kTB + ii;
    const T vi = (gr >= m) ? T(0) : (gr == 0 ? T(1) : (T)((double)vraw * scal));
    if (fresh) {
      const int gc = J * kTB + cg * 16 + (ii & 15);
      if (ii < 16) vj[ii] = gc == 0 ? T(1) : (gc < m ? (T)((double)uraw * scal) : T(0));
      __builtin_amdgcn_wave_barrier();
      fresh = false;
    }
    T yp = T(0);
    if (I > J) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        yp += t[e] * vj[e];
        zacc[e] += t[e] * vi;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const T x = ii >= cg * 16 + e && gr < m ? t[e] : T(0);
        yp += x * vj[e];
        if (ii > cg * 16 + e) zacc[e] += x * vi;
      }
    }
    red[k & 3][cg][ii] = yp;
    // every second tile (and the last): one barrier, then the rows of the last two tiles are
    // summed over the waves (wave 0 and wave 1 take one tile each). A buffer is written again
    // four tiles later, after at least one more barrier.
    const bool last = t0 + k + 1 == t1;
    if ((k & 1) || last) {
      lds_barrier();
      if (cg == 0 || (cg == 1 && (k & 1))) {
        const int b = (k - cg) & 3, row = (cg == 0 ? I : pI) * kTB + ii;
        if (row < m)
          Y[(long)(cg == 0 ? J : pJ) * n + row] =
              red[b][0][ii] + red[b][1][ii] + red[b][2][ii] + red[b][3][ii];
      }
    }
    pI = I;
    pJ = J;
    ++k;
    if (++I == nRB || last) {   // the column's end here
      const T z = wave_sum16(zacc, ii);
      const int kc = J * kTB + cg * 16 + ii;
      if (ii < 16 && kc < m) Y[(long)(nRB + w - symv_first(nRB, J) / q) * n + kc] = z;
#pragma unroll
      for (int e = 0; e < 16; ++e) zacc[e] = T(0);
      I = ++J;
      fresh = true;
    }
  };
  for (int t = t0; t < t1; t += 3) {
    load(b2, v2, u2);
    tile(b0, v0, u0);
    if (t + 1 >= t1) break;
    load(b0, v0, u0);
    tile(b1, v1, u1);
    if (t + 2 >= t1) break;
    load(b1, v1, u1);
    tile(b2, v2, u2);
  }
}

// y(r) from its slots, w = tau * (y - V t1 - W t2); store v into column c and accumulate w.v.
// Slots are stored slot-major (Y(row, slot) at slot * n + row): a block handles 64 rows (the
// lanes) and its kFinW waves split the slots and the panel correction between them (many
// waves per row block keep enough loads in flight: there are only m / 64 blocks).
constexpr int kFinW = 16;
template <typename T>
__global__ __launch_bounds__(64 * kFinW) void finalize_w_kernel(T* a, long lda, int n, int c,
                                                                int j0, T* W, long ldw, const T* Y,
                                                                int nSlot, const T* vbuf,
                                                                const double* t12, const T* tauA,
                                                                double* dot, int tiles,
                                                                ProblemStrides ps) {
  __shared__ double red[kFinW][64];
  a += (long)blockIdx.z * ps.a;
  tauA += (long)blockIdx.z * ps.v;
  W = ws_of(W, ps.ws);
  Y = ws_of(Y, ps.ws);
  vbuf = ws_of(vbuf, ps.ws);
  t12 = ws_of(t12, ps.ws);
  dot = ws_of(dot, ps.ws);
  const int m = n - c - 1;
  const int nRB = (m + kTB - 1) / kTB;
  const int i = c - j0;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int k = blockIdx.x * 64 + lane;
  const int r = c + 1 + k;
  double acc = 0.0;
  if (k < m) {
    const int Ir = k / kTB;
    const int nch = symv_pieces(nRB, Ir, tiles);
    // this wave's slots (sl = wv, wv + kFinW, ...) with four independent sums
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    int sl = wv;
    for (; sl + 3 * kFinW <= Ir; sl += 4 * kFinW) {
      s0 += Y[(long)sl * n + k];
      s1 += Y[(long)(sl + kFinW) * n + k];
      s2 += Y[(long)(sl + 2 * kFinW) * n + k];
      s3 += Y[(long)(sl + 3 * kFinW) * n + k];
    }
    for (; sl <= Ir; sl += kFinW) s0 += Y[(long)sl * n + k];
    const T* Yc = Y + (long)nRB * n;
    sl = wv;
    for (; sl + 3 * kFinW < nch; sl += 4 * kFinW) {
      s1 += Yc[(long)sl * n + k];
      s2 += Yc[(long)(sl + kFinW) * n + k];
      s3 += Yc[(long)(sl + 2 * kFinW) * n + k];
      s0 += Yc[(long)(sl + 3 * kFinW) * n + k];
    }
    for (; sl < nch; sl += kFinW) s1 += Yc[(long)sl * n + k];
    acc = (s0 + s1) + (s2 + s3);
    // panel correction of this wave's p = wv + kFinW q, loads ahead of the products
    double vr[kNB / kFinW], wr[kNB / kFinW];
#pragma unroll
    for (int q = 0; q < kNB / kFinW; ++q) {
      const int p = wv + kFinW * q;
      vr[q] = 0.0;
      wr[q] = 0.0;
      if (p < i) {
        vr[q] = a[r + (long)(j0 + p) * lda];
        wr[q] = W[r + (long)p * ldw];
      }
    }
#pragma unroll
    for (int q = 0; q < kNB / kFinW; ++q) {
      const int p = wv + kFinW * q;
      if (p < i) {
        const double w = wr[q] + wcorr(j0 + p, tauA, dot) * vr[q];
        acc -= vr[q] * t12[t12_at(c, p)] + w * t12[t12_at(c, i + p)];
      }
    }
  }
  red[wv][lane] = acc;
  __syncthreads();
  if (wv == 0) {
    double prod = 0.0;
    if (k < m) {
      double y = 0.0;
#pragma unroll
      for (int q = 0; q < kFinW; ++q) y += red[q][lane];
      const T w = (T)((double)tauA[c] * y);
      W[r + (long)i * ldw] = w;
      const T v = vbuf[r];
      a[r + (long)c * lda] = v;
      prod = (double)w * (double)v;
    }
    prod = wave_sum(prod);
    if (lane == 0 && prod != 0.0) atomicAdd(&dot[c], prod);
  }
}

// P = [V W], Q = [W V] for the trailing update, rows r0..n-1 (W with its rank-one correction).
template <typename T>
__global__ void panel_pack_kernel(const T* a, long lda, int n, int r0, int j0, int pw,
                                  const T* W, long ldw, const T* tau, const double* dot, T* P,
                                  T* Q, long ldp) {
  const int p = blockIdx.y;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int r = r0 + k;
  if (r >= n) return;
  const T v = a[r + (long)(j0 + p) * lda];
  const T w = (T)((double)W[r + (long)p * ldw] + wcorr(j0 + p, tau, dot) * (double)v);
  P[k + (long)p * ldp] = v;
  P[k + (long)(p + pw) * ldp] = w;
  Q[k + (long)p * ldp] = w;
  Q[k + (long)(p + pw) * ldp] = v;
}

template <typename T>
__global__ void panel_restore_kernel(T* a, long lda, int n, int j0, int pw, T* d, const T* e) {
  const int p = threadIdx.x;
  if (p >= pw) return;
  const int c = j0 + p;
  d[c] = a[c + (long)c * lda];
  if (c + 1 < n) a[(c + 1) + (long)c * lda] = e[c];
}

// K problems of size n at once: problem k's matrix at a + k sA, d, e, tau at + k sV and its
// workspace block at work + k wsStride bytes (wsStride >= sytrd_layout(n)). The column kernels
// run all problems in one launch each; the panel products and trailing updates run per problem.
// Panels from .. to - 1 (multiples of kNB, or to = n); the panels before `from` have been run.
template <typename T>
static int sytrd_launches(hipStream_t s, T* a, long lda, long sA, int n, T* d, T* e, T* tau,
                          long sV, void* work, size_t wsStride, int K, int from, int to) {
  std::vector<SytrdWs<T>> wk(K);
  for (int k = 0; k < K; ++k) {
    sytrd_layout<T>(n, &wk[k], static_cast<char*>(work) + (size_t)k * wsStride);
    if (from > 0) continue;
    DH_TRY(fill<double>(s, wk[k].nrm2, n, 0.0));
    DH_TRY(fill<double>(s, wk[k].dot, n, 0.0));
    DH_TRY(fill<double>(s, wk[k].t12, (size_t)kT12Size, 0.0));
    DH_TRY(fill<T>(s, e + k * sV, std::max(n - 1, 1), T(0)));
    DH_TRY(fill<T>(s, tau + k * sV, std::max(n, 1), T(0)));
  }
  const SytrdWs<T>& ws = wk[0];
  const ProblemStrides ps{K > 1 ? sA : 0, K > 1 ? (long)wsStride : 0, K > 1 ? sV : 0};
  const long ldw = n;
  for (int j0 = from; j0 < to; j0 += kNB) {
    const int pw = std::min(kNB, n - j0);
    for (int i = 0; i < pw; ++i) {
      const int c = j0 + i;
      hipLaunchKernelGGL(col_update_kernel<T>, dim3(cdiv(n - c, 64), 1, K), dim3(256), 0, s, a,
                         lda, n, c, j0, ws.W, ldw, tau, ws.dot, ws.nrm2, ws.t12, ps);
      DH_LAUNCH_CHECK();
      const int m = n - c - 1;
      if (m <= 0) continue;
      const int nRB = (m + kTB - 1) / kTB;
      const int tiles = symv_tiles<T>(m, K);
      const int nWg = (nRB * (nRB + 1) / 2 + tiles - 1) / tiles;
      SymvProfile& pf = g_symvProf;
      if (pf.on) {
        if (pf.ev.size() < 2 * (pf.used + 1)) {
          const size_t old = pf.ev.size();
          pf.ev.resize(2 * (pf.used + 1) + 2 * 1024);
          for (size_t q = old; q < pf.ev.size(); ++q) DH_HIP(hipEventCreate(&pf.ev[q]));
          pf.bytes.resize(pf.ev.size() / 2);
          pf.size.resize(pf.ev.size() / 2);
        }
        DH_HIP(hipEventRecord(pf.ev[2 * pf.used], s));
      }
      hipLaunchKernelGGL(symv_kernel<T>, dim3(nRB + nWg, 1, K), dim3(256), 0, s, a, lda, n, c, j0,
                         ws.W, ldw, ws.nrm2, tau, ws.dot, ws.Y, ws.vbuf, ws.t12, ws.scal, e, tau,
                         tiles, ps);
      DH_LAUNCH_CHECK();
      if (pf.on) {
        DH_HIP(hipEventRecord(pf.ev[2 * pf.used + 1], s));
        // lower triangle of the m x m trailing matrix plus v in and the partial sums out, for
        // each problem
        pf.bytes[pf.used] = (double)K * sizeof(T) * ((double)m * (m + 1) / 2 + 2.0 * m);
        pf.size[pf.used] = m;
        ++pf.used;
      }
      hipLaunchKernelGGL(finalize_w_kernel<T>, dim3(cdiv(m, 64), 1, K), dim3(64 * kFinW), 0, s,
                         a, lda, n, c, j0, ws.W, ldw, ws.Y, ws.nSlot, ws.vbuf, ws.t12, tau,
                         ws.dot, tiles, ps);
      DH_LAUNCH_CHECK();
    }
    const int r0 = j0 + pw;
    for (int k = 0; k < K; ++k) {
      T* ak = a + k * sA;
      const T* tk = tau + k * sV;
      if (r0 < n) {
        const int mt = n - r0;
        hipLaunchKernelGGL(panel_pack_kernel<T>, dim3(cdiv(mt, 256), pw), dim3(256), 0, s, ak,
                           lda, n, r0, j0, pw, wk[k].W, ldw, tk, wk[k].dot, wk[k].P, wk[k].Q,
                           (long)mt);
        DH_LAUNCH_CHECK();
        T* a22 = ak + r0 + (long)r0 * lda;
        DH_TRY(gemm<T>(s, false, true, mt, mt, 2 * pw, T(-1), wk[k].P, mt, wk[k].Q, mt, T(1),
                       a22, lda, true));
      }
      hipLaunchKernelGGL(panel_restore_kernel<T>, dim3(1), dim3(64), 0, s, ak, lda, n, j0, pw,
                         d + k * sV, e + k * sV);
      DH_LAUNCH_CHECK();
    }
  }
  return 0;
}

// The launch sequence of one tridiagonalisation (3 launches per column and the panel updates, up
// to the size from which the resident kernels take over) depends only on the sizes, the buffers
// and the tile choice, and holds no host synchronisation: it is captured once into a HIP graph
// and replayed for every later call with the same arguments (an SCC cycle calls it once per iteration on
// the same buffers), which removes the host launch cost between the short column kernels
// (when switched on: set_sytrd_graphs).
// Cleared memory inside the sequence is written by fill kernels (no memset nodes). A few
// sequences are kept, the oldest replaced; not while the per-launch SYMV timing is on.
struct SytrdGraphKey {
  const void* a;
  long lda, sA, sV;
  int n, K, prec;
  const void *d, *e, *tau, *work;
  size_t wsStride;
  unsigned gen;
  bool operator==(const SytrdGraphKey& o) const {
    return a == o.a && lda == o.lda && sA == o.sA && sV == o.sV && n == o.n && K == o.K &&
           prec == o.prec && d == o.d && e == o.e && tau == o.tau && work == o.work &&
           wsStride == o.wsStride && gen == o.gen;
  }
};
struct SytrdGraph {
  SytrdGraphKey key;
  hipGraphExec_t exec = nullptr;
  unsigned long use = 0;
};
static std::vector<SytrdGraph> g_sytrdGraphs;
static std::mutex g_sytrdGraphMutex;
static unsigned long g_sytrdGraphUse = 0;
// off by default: the replay saves about 2 % of an FP32 iteration, and rocprofv3's kernel
// tracing takes the process down on the capture (a host fault inside the tool)
static bool g_sytrdGraphOn = false;
constexpr size_t kSytrdGraphsKept = 4;

int set_sytrd_graphs(bool on) {
  g_sytrdGraphOn = on;
  return 0;
}

void release_sytrd_graphs() {
  std::lock_guard<std::mutex> lock(g_sytrdGraphMutex);
  for (auto& g : g_sytrdGraphs)
    if (g.exec) (void)hipGraphExecDestroy(g.exec);
  g_sytrdGraphs.clear();
}

// the panels up to column `to`: launched one by one, or replayed
template <typename T>
static int sytrd_panels(hipStream_t s, T* a, long lda, long sA, int n, T* d, T* e, T* tau,
                        long sV, void* work, size_t wsStride, int K, int to) {
  if (!g_sytrdGraphOn || g_symvProf.on || n < 2)
    return sytrd_launches<T>(s, a, lda, sA, n, d, e, tau, sV, work, wsStride, K, 0, to);
  std::lock_guard<std::mutex> lock(g_sytrdGraphMutex);
  const SytrdGraphKey key{a, lda, sA, sV, n, K, (int)sizeof(T), d, e, tau, work, wsStride,
                          g_tileGen};
  for (auto& g : g_sytrdGraphs)
    if (g.key == key) {
      g.use = ++g_sytrdGraphUse;
      DH_HIP(hipGraphLaunch(g.exec, s));
      return 0;
    }
  DH_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
  const int rc = sytrd_launches<T>(s, a, lda, sA, n, d, e, tau, sV, work, wsStride, K, 0, to);
  hipGraph_t graph = nullptr;
  const hipError_t ec = hipStreamEndCapture(s, &graph);
  if (rc != 0) {
    if (graph) (void)hipGraphDestroy(graph);
    return rc;
  }
  if (ec != hipSuccess) {
    if (graph) (void)hipGraphDestroy(graph);
    DH_HIP(ec);
  }
  hipGraphExec_t exec = nullptr;
  const hipError_t ei = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  DH_HIP(ei);
  if (g_sytrdGraphs.size() >= kSytrdGraphsKept) {
    auto old = std::min_element(g_sytrdGraphs.begin(), g_sytrdGraphs.end(),
                                [](const SytrdGraph& x, const SytrdGraph& y) {
                                  return x.use < y.use;
                                });
    (void)hipGraphExecDestroy(old->exec);
    g_sytrdGraphs.erase(old);
  }
  g_sytrdGraphs.push_back(SytrdGraph{key, exec, ++g_sytrdGraphUse});
  DH_HIP(hipGraphLaunch(exec, s));
  return 0;
}

// allColumns: the blocked form to the end (the autotuner times its launches at every size)
template <typename T>
int sytrd_lower_batched_t(hipStream_t s, T* a, long lda, long sA, int n, T* d, T* e, T* tau,
                          long sV, void* work, size_t wsStride, int K, bool allColumns = false) {
  DH_CHECK(K >= 1, "sytrd: no problems");
  DH_CHECK(wsStride >= sytrd_layout<T>(n, nullptr, nullptr), "sytrd: workspace too small");
  DH_CHECK(K == 1 || (sA >= lda * (long)n && sV >= n && wsStride % 256 == 0),
           "sytrd: problems overlap or are misaligned");
  int handOver = n;
  if (!allColumns && n > 1) DH_TRY(sytrd_resident_from(n, K, &handOver));
  if (handOver > 0)
    DH_TRY(sytrd_panels<T>(s, a, lda, sA, n, d, e, tau, sV, work, wsStride, K, handOver));
  if (handOver < n) {
    // the exchange ring lies in P, the flag in Q: both are written at panel ends only
    static_assert(sizeof(T) * 2 * kNB >= 8 * kResidentWords, "ring larger than the panel copy");
    SytrdWs<T> ws;
    sytrd_layout<T>(n, &ws, static_cast<char*>(work));
    bool done = false;
    DH_TRY(sytrd_resident<T>(s, a, lda, K > 1 ? sA : 0, n, handOver, d, e, tau, K > 1 ? sV : 0,
                             reinterpret_cast<unsigned long long*>(ws.P),
                             K > 1 ? (long)(wsStride / 8) : 0, reinterpret_cast<int*>(ws.Q), K,
                             &done));
    if (!done)
      DH_TRY(sytrd_launches<T>(s, a, lda, sA, n, d, e, tau, sV, work, wsStride, K, handOver, n));
  }
  DH_TRY(symv_prof_collect(s));
  return 0;
}

template <typename T>
int sytrd_lower_t(hipStream_t s, T* a, long lda, int n, T* d, T* e, T* tau, void* work,
                  size_t workBytes) {
  return sytrd_lower_batched_t<T>(s, a, lda, 0, n, d, e, tau, 0, work, workBytes, 1);
}

// ---------------------------------------------------------------------------------------------
// Back-transformation Z <- Q Z, Q = H(0) H(1) ... H(n-2), panels applied last to first with the
// compact WY form I - V T V^T (T upper triangular, LAPACK dlarft 'F','C').
// ---------------------------------------------------------------------------------------------
template <typename T>
struct OrmWs {
  T* V;         // n x kOB
  T* G;         // kOB x kOB
  T* Tm;        // kOB x kOB
  T* W1;        // kOB x ncols
  T* W2;        // kOB x ncols
};

constexpr int kOB = 256;    // reflectors per block of the back-transformation
constexpr int kOBH = 128;   // half block: the compact-WY T of a half is formed in LDS

template <typename T>
static size_t ormtr_layout(int n, int ncols, OrmWs<T>* ws, char* base) {
  size_t off = 0;
  OrmWs<T> dummy;
  OrmWs<T>* w = ws ? ws : &dummy;
  auto take = [&](T** p, size_t cnt) {
    if (ws) *p = reinterpret_cast<T*>(base + off);
    off += (cnt * sizeof(T) + 255) / 256 * 256;
  };
  take(&w->V, (size_t)n * kOB);
  take(&w->G, kOB * kOB);
  take(&w->Tm, kOB * kOB);
  take(&w->W1, (size_t)kOB * std::max(ncols, 1));
  take(&w->W2, (size_t)kOB * std::max(ncols, 1));
  return off;
}

size_t ormtr_work_bytes(int n, int ncols, int elemSize) {
  return elemSize == 8 ? ormtr_layout<double>(n, ncols, nullptr, nullptr)
                       : ormtr_layout<float>(n, ncols, nullptr, nullptr);
}
size_t ormtr_work_size(int n, int ncols) { return (ormtr_work_bytes(n, ncols, 8) + 7) / 8; }

// explicit V (rows j0+shift..n-1) of the block's reflectors; reflector c has its unit element
// at row c + shift and its other elements below it in column c of a
template <typename T>
__global__ void form_v_kernel(const T* a, long lda, int n, int j0, int pw, int shift, T* V,
                              long ldv, long sA = 0, long sW = 0) {
  a += blockIdx.z * sA;
  V += blockIdx.z * sW;
  const int p = blockIdx.y;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int r = j0 + shift + k;
  if (r >= n) return;
  const int c = j0 + p;
  T v;
  if (r < c + shift) v = T(0);
  else if (r == c + shift) v = T(1);
  else v = a[r + (long)c * lda];
  V[k + (long)p * ldv] = v;
}

// T of the compact WY form of pw <= kOBH reflectors (LAPACK dlarft 'F','C': T(i,i) = tau_i,
// T(0:i,i) = -tau_i T(0:i,0:i) G(0:i,i), G = V^T V): T = (I + D U)^-1 D with D = diag(tau) and U
// the strict upper triangle of G, the inverse formed by doubling in LDS. Block h of the launch
// takes reflectors j0 + h kOBH .. and the diagonal block h of G and Tout; all of the block of Tout
// is written. One thread per row running the recurrence took 248 us for 128 reflectors; this form
// takes 52 us.
template <typename T>
__global__ __launch_bounds__(256) void larft_kernel(const T* G, long ld, const T* tau, int j0,
                                                    int nref, T* Tout, long sV = 0, long sW = 0) {
  G += blockIdx.y * sW;
  tau += blockIdx.y * sV;
  Tout += blockIdx.y * sW;
  constexpr int kLd = kOBH + 1;
  __shared__ T X[kOBH * kLd];
  __shared__ T tl[kOBH];
  const int o = blockIdx.x * kOBH;
  const int pw = min(kOBH, nref - o);
  const int t = threadIdx.x;
  if (t < kOBH) tl[t] = t < pw ? tau[j0 + o + t] : T(0);
  __syncthreads();
  // row c, column r of X: (D U)(r, c), so that the inverse of X is that of I + D U transposed
  for (int e = t; e < kOBH * kOBH; e += 256) {
    const int r = e % kOBH, c = e / kOBH;
    X[c * kLd + r] = r < c && c < pw ? tl[r] * G[o + r + (long)(o + c) * ld] : (r == c ? T(1) : T(0));
  }
  __syncthreads();
  lower_inverse_lds<T, kOBH, kLd>(X);
  for (int e = t; e < pw * pw; e += 256) {
    const int r = e % pw, c = e / pw;
    Tout[o + r + (long)(o + c) * ld] = r <= c ? X[c * kLd + r] * tl[c] : T(0);
  }
}

template <typename T>
int ormtr_lower_t(hipStream_t s, const T* a, long lda, int n, const T* tau, T* z, long ldz,
                  int ncols, void* work, size_t workBytes, int shift, int nref) {
  DH_CHECK(workBytes >= ormtr_layout<T>(n, ncols, nullptr, nullptr), "ormtr: workspace too small");
  if (nref <= 0 || ncols <= 0) return 0;
  OrmWs<T> ws;
  ormtr_layout<T>(n, ncols, &ws, static_cast<char*>(work));
  const int lastBlock = ((nref - 1) / kOB) * kOB;
  for (int j0 = lastBlock; j0 >= 0; j0 -= kOB) {
    const int pw = std::min(kOB, nref - j0);
    const int m = n - j0 - shift;
    if (m <= 0) continue;
    hipLaunchKernelGGL(form_v_kernel<T>, dim3(cdiv(m, 256), pw), dim3(256), 0, s, a, lda, n, j0,
                       pw, shift, ws.V, (long)m);
    DH_LAUNCH_CHECK();
    const int sk = std::max(1, std::min(64, m / 512));
    DH_TRY(gemm<T>(s, true, false, pw, pw, m, T(1), ws.V, m, ws.V, m, T(0), ws.G, kOB, false,
                   kKFull, nullptr, sk));
    // T of each half in LDS, then the coupling block of H1 H2 = I - [V1 V2] T [V1 V2]^T:
    // T12 = -T11 (V1^T V2) T22 (the product goes through G's unused lower-left block)
    const int p1 = std::min(pw, kOBH), p2 = pw - p1;
    DH_TRY(fill<T>(s, ws.Tm, (size_t)kOB * kOB, T(0)));
    hipLaunchKernelGGL(larft_kernel<T>, dim3(p2 > 0 ? 2 : 1), dim3(256), 0, s, ws.G, (long)kOB,
                       tau, j0, pw, ws.Tm);
    DH_LAUNCH_CHECK();
    if (p2 > 0) {
      T* T22 = ws.Tm + p1 + (long)p1 * kOB;
      T* X = ws.G + p1;
      DH_TRY(gemm<T>(s, false, false, p1, p2, p2, T(1), ws.G + (long)p1 * kOB, kOB, T22, kOB,
                     T(0), X, kOB));
      DH_TRY(gemm<T>(s, false, false, p1, p2, p1, T(-1), ws.Tm, kOB, X, kOB, T(0),
                     ws.Tm + (long)p1 * kOB, kOB));
    }
    T* zr = z + (j0 + shift);
    const int skz = std::max(1, std::min(16, m / 1024));
    DH_TRY(gemm<T>(s, true, false, pw, ncols, m, T(1), ws.V, m, zr, ldz, T(0), ws.W1, kOB, false,
                   kKFull, nullptr, skz));
    DH_TRY(gemm<T>(s, false, false, pw, ncols, pw, T(1), ws.Tm, kOB, ws.W1, kOB, T(0), ws.W2,
                   kOB));
    DH_TRY(gemm<T>(s, false, false, m, ncols, pw, T(-1), ws.V, m, ws.W2, kOB, T(1), zr, ldz));
  }
  return 0;
}

// Z_k <- Q_k Z_k (n x n each) for K problems, kOBH reflectors at a time: six launches a block for
// all problems. desc: room for 4 descriptors per problem and block of reflectors.
static long ormtr_many_stride(int n) { return 3L * kOBH * n + 2L * kOBH * kOBH; }
size_t ormtr_many_work(int n, int K) { return (size_t)K * ormtr_many_stride(n); }

int ormtr_lower_many(hipStream_t s, const double* a, long sA, int n, const double* tau, long sV,
                     double* z, long sZ, int K, double* work, DevBuf<GemmDesc<double>>& desc) {
  const int nref = n - 1;
  if (nref <= 0 || K <= 0) return 0;
  const long sW = ormtr_many_stride(n);
  std::vector<GemmDesc<double>> h;
  for (int j0 = (nref - 1) / kOBH * kOBH; j0 >= 0; j0 -= kOBH) {
    const int pw = std::min(kOBH, nref - j0), m = n - j0 - 1;
    for (int q = 0; q < 4; ++q)
      for (int k = 0; k < K; ++k) {
        double* V = work + k * sW;
        double *W1 = V + (long)kOBH * n, *W2 = W1 + (long)kOBH * n, *G = W2 + (long)kOBH * n,
               *T = G + kOBH * kOBH, *zr = z + k * sZ + j0 + 1;
        if (q == 0) h.push_back({pw, pw, m, V, (long)m, V, (long)m, G, (long)kOBH});
        if (q == 1) h.push_back({pw, n, m, V, (long)m, zr, (long)n, W1, (long)kOBH});
        if (q == 2) h.push_back({pw, n, pw, T, (long)kOBH, W1, (long)kOBH, W2, (long)kOBH});
        if (q == 3) h.push_back({m, n, pw, V, (long)m, W2, (long)kOBH, zr, (long)n});
      }
  }
  DH_TRY(desc.upload(h.data(), h.size(), s));
  const GemmDesc<double>* g = desc.p;
  for (int j0 = (nref - 1) / kOBH * kOBH; j0 >= 0; j0 -= kOBH, g += 4 * (size_t)K) {
    const int pw = std::min(kOBH, nref - j0), m = n - j0 - 1;
    double *G = work + 3L * kOBH * n, *T = G + kOBH * kOBH;
    hipLaunchKernelGGL(form_v_kernel<double>, dim3(cdiv(m, 256), pw, K), dim3(256), 0, s, a,
                       (long)n, n, j0, pw, 1, work, (long)m, sA, sW);
    DH_LAUNCH_CHECK();
    DH_TRY(gemm_batched<double>(s, true, false, g, K, pw, pw, 1.0, 0.0));
    hipLaunchKernelGGL(larft_kernel<double>, dim3(1, K), dim3(256), 0, s, G, (long)kOBH, tau, j0,
                       pw, T, sV, sW);
    DH_LAUNCH_CHECK();
    DH_TRY(gemm_batched<double>(s, true, false, g + K, K, pw, n, 1.0, 0.0));
    DH_TRY(gemm_batched<double>(s, false, false, g + 2 * K, K, pw, n, 1.0, 0.0));
    DH_TRY(gemm_batched<double>(s, false, false, g + 3 * K, K, m, n, -1.0, 1.0));
  }
  DH_HIP(hipStreamSynchronize(s));   // the descriptors' host copy
  return 0;
}

int sytrd_lower(hipStream_t s, double* a, long lda, int n, double* d, double* e, double* tau,
                double* work, size_t workSize) {
  return sytrd_lower_t<double>(s, a, lda, n, d, e, tau, work, workSize * sizeof(double));
}
int sytrd_lower_batched(hipStream_t s, double* a, long lda, long sA, int n, double* d, double* e,
                        double* tau, long sV, void* work, size_t wsStride, int K) {
  return sytrd_lower_batched_t<double>(s, a, lda, sA, n, d, e, tau, sV, work, wsStride, K);
}
int sytrd_lower_f32(hipStream_t s, float* a, long lda, int n, float* d, float* e, float* tau,
                    void* work, size_t workBytes) {
  return sytrd_lower_t<float>(s, a, lda, n, d, e, tau, work, workBytes);
}
// ---------------------------------------------------------------------------------------------
// Autotuner of the SYMV tile count: the tridiagonalisation of a synthetic symmetric n x n matrix
// is run once per fixed tile count and once with the tiles shared out evenly, with every SYMV
// launch timed by HIP events; launches are grouped by trailing size in buckets of kTuneBucket rows
// and symv_choose picks from the summed times. Its table is installed for the arithmetic type.
// 15769 rows, FP64, SYMV of one tridiagonalisation: even share 1.118 s, the fastest fixed count of
// each bucket 1.140 s; 4000 rows: 27.4 and 25.3 ms.
// ---------------------------------------------------------------------------------------------

// lower triangle of a symmetric matrix from a hash of (i, j): values in [-1, 1), diagonal
// shifted by i / n
template <typename T>
__global__ void synth_sym_kernel(T* a, long lda, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
  if (i >= n || i < j) return;
  uint32_t h = (uint32_t)i * 0x9E3779B1u ^ ((uint32_t)j * 0x85EBCA77u + 0x165667B1u);
  h ^= h >> 15;
  h *= 0x2C1B3C6Du;
  h ^= h >> 12;
  h *= 0x297A2D39u;
  h ^= h >> 15;
  double v = (double)(h >> 8) * (1.0 / 8388608.0) - 1.0;
  if (i == j) v += (double)i / n;
  a[i + (long)j * lda] = (T)v;
}

template <typename T>
static int symv_autotune_t(hipStream_t s, int n, TileTable& rows, std::vector<double>* detail) {
  DH_CHECK(n >= kTuneBucket && n <= 65535, "autotune: n must be in [256, 65535]");
  DevBuf<T> a, d, e, tau;
  DevBuf<char> work;
  DH_TRY(a.alloc((size_t)n * n));
  DH_TRY(d.alloc(n));
  DH_TRY(e.alloc(n));
  DH_TRY(tau.alloc(n));
  const size_t wb = sytrd_layout<T>(n, nullptr, nullptr);
  DH_TRY(work.alloc(wb));
  const int nb = (n + kTuneBucket - 1) / kTuneBucket;
  std::vector<double> t((kTuneFixed + 1) * (size_t)nb, 0.0);
  std::vector<std::pair<int, float>> rec;
  SymvProfile& pf = g_symvProf;
  const bool on0 = pf.on;
  const double l0 = pf.launches, s0 = pf.seconds, b0 = pf.algBytes;
  const int tiles0 = g_symvTiles;
  int rc = 0;
  TileTable& table = g_tileTable[std::is_same<T, float>::value ? 1 : 0];
  TileTable before;
  before.swap(table);
  for (int o = 0; o <= kTuneFixed && rc == 0; ++o) {
    g_symvTiles = o < kTuneFixed ? kTuneOptions[o] : 0;
    ++g_tileGen;
    // untimed pass on a small matrix first: the option's kernels are loaded before timing
    for (int nn : {kTuneBucket, n}) {
      hipLaunchKernelGGL(synth_sym_kernel<T>, dim3(cdiv(nn, 256), nn), dim3(256), 0, s, a.p,
                         (long)nn, nn);
      rc = hipGetLastError() == hipSuccess ? 0 : kErrDevice;
      if (rc) {
        set_error("autotune: launch of the test matrix kernel failed");
        break;
      }
      pf.on = nn == n;
      pf.sink = nn == n ? &rec : nullptr;
      rec.clear();
      rc = sytrd_lower_batched_t<T>(s, a.p, nn, 0, nn, d.p, e.p, tau.p, 0, work.p, wb, 1, true);
      pf.sink = nullptr;
      if (rc) break;
    }
    for (const auto& r : rec) t[(size_t)o * nb + r.first / kTuneBucket] += 1e-3 * r.second;
  }
  g_symvTiles = tiles0;
  ++g_tileGen;
  pf.on = on0;
  pf.launches = l0;
  pf.seconds = s0;
  pf.algBytes = b0;
  pf.sink = nullptr;
  if (rc) {
    table.swap(before);
    return rc;
  }
  DH_HIP(hipStreamSynchronize(s));
  symv_choose(t, nb, &rows, &table);
  t.resize(kTuneFixed * (size_t)nb);
  if (detail) *detail = t;
  ++g_tileGen;
  return 0;
}

int symv_autotune(hipStream_t s, int n, int precision, std::vector<std::pair<int, int>>& rows,
                  std::vector<double>* detail) {
  DH_CHECK(precision == 0 || precision == 1, "autotune: precision must be 0 (FP64) or 1 (FP32)");
  return precision == 0 ? symv_autotune_t<double>(s, n, rows, detail)
                        : symv_autotune_t<float>(s, n, rows, detail);
}

int ormtr_lower(hipStream_t s, const double* a, long lda, int n, const double* tau, double* z,
                long ldz, int ncols, double* work, size_t workSize) {
  return ormtr_lower_t<double>(s, a, lda, n, tau, z, ldz, ncols, work, workSize * sizeof(double),
                               1, n - 1);
}
int ormtr_lower_f32(hipStream_t s, const float* a, long lda, int n, const float* tau, float* z,
                    long ldz, int ncols, void* work, size_t workBytes) {
  return ormtr_lower_t<float>(s, a, lda, n, tau, z, ldz, ncols, work, workBytes, 1, n - 1);
}
// back-transformation with the reflectors of the band reduction (unit element `shift` rows
// below the column, nref reflectors)
template <typename T>
int ormqr_shift(hipStream_t s, const T* a, long lda, int n, const T* tau, T* z, long ldz,
                int ncols, void* work, size_t workBytes, int shift, int nref) {
  return ormtr_lower_t<T>(s, a, lda, n, tau, z, ldz, ncols, work, workBytes, shift, nref);
}
template int ormqr_shift<double>(hipStream_t, const double*, long, int, const double*, double*,
                                 long, int, void*, size_t, int, int);
template int ormqr_shift<float>(hipStream_t, const float*, long, int, const float*, float*, long,
                                int, void*, size_t, int, int);

}  // namespace dftbhip
