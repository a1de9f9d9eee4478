// Householder tridiagonalisation of a trailing matrix that fits on the chip: the matrix is read
// once into registers, every column is reduced there, and only vectors travel between waves or
// workgroups. It takes over from the blocked form (sytrd.hip) as soon as the trailing matrix is
// small enough; that form needs three launches per column, about 23 us a column however small the
// matrix is. Measured, FP64, whole tridiagonalisations, blocked -> resident: 573 columns 13.1 ->
// 1.5 ms, 1024 columns 23.8 -> 2.8 ms, 1800 columns 42 -> 7.3 ms, 2500 columns 65 -> 10.4 ms.
// What bounds it: one exchange through memory per column (about 1.5 us), then the serial chain
// from the gathered vectors to the next published ones.
//
// Unblocked form with the rank-two update delayed by one column and fused with the product:
//   A <- A - v' w'^T - w' v'^T (the previous column's pair), y = A v, in one pass over registers;
//   w = tau y - (tau^2 / 2) (y.v) v;   next column x = A(:, k+1) - v w_{k+1} - w v_{k+1}.
// Every row of the full symmetric matrix lives in one place, so y needs no sum across
// workgroups, and y together with the (not yet updated) next column is all that the others need:
// one exchange per column. x, v and w are then formed by every wave or workgroup for itself, by
// the same operations in the same order, so all hold the same bits.
//
// Arithmetic is FP64 for both element types; FP32 matrices are rounded where they are stored.
#include <algorithm>
#include <cstring>

#include "common.h"
#include "exchange_ring.h"
#include "lanes.h"

namespace dftbhip {

using u64 = unsigned long long;

namespace {

// Sums of four values per lane over the 64 lanes: lane l returns the total of acc[(l >> 2) & 3].
// Each halving exchanges the pair of values a lane does not keep: three exchanges and four plain
// steps on one value instead of 24. (Sixteen at a time need fewer still, but hold 32 registers.)
__device__ __forceinline__ double rows_total4(const double (&acc)[4], int lane) {
  double pr[2];
  const bool up8 = lane & 8, up4 = lane & 4;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const double keep = up8 ? acc[r + 2] : acc[r], send = up8 ? acc[r] : acc[r + 2];
    pr[r] = keep + dpp<kRor8>(send);
  }
  const double keep = up4 ? pr[1] : pr[0], send = up4 ? pr[0] : pr[1];
  double v = keep + dpp<kHalfMirror>(send);   // lane ^ 7: the other half of eight lanes
  v += dpp<kQuadXor1>(v);
  v += dpp<kQuadXor2>(v);
  v = swap16_add(v, v);
  return swap32_add(v, v);
}

// total of NW (4 or 8) values, lane l holding value l mod NW: the same bits in every lane
template <int NW>
__device__ __forceinline__ double part_total(double v) {
  static_assert(NW == 4 || NW == 8, "part_total: 4 or 8 values");
  if constexpr (NW == 8) v += dpp<kRor4>(v);
  v += dpp<kRor2>(v);
  return v + dpp<kRor1>(v);
}

// element idx of the vector whose element l + 64 q is x[q] of lane l
template <int C>
__device__ __forceinline__ double element(const double (&x)[C], int idx) {
  // lane values first, then a choice between scalars: choosing the register by idx would put x
  // into memory
  double v = lane_value(x[0], idx & 63);
#pragma unroll
  for (int q = 1; q < C; ++q) {
    const double u = lane_value(x[q], idx & 63);
    if (idx >= 64 * q) v = u;
  }
  return v;
}

// Reflector of (alpha, x) as LAPACK dlarfg without the rescaling loop: with s = alpha^2 + |x|^2,
// beta = -sign(alpha) sqrt(s), tau = (beta - alpha) / beta = 1 + |alpha| / sqrt(s), scale
// 1 / (alpha - beta) = sign(alpha) / (|alpha| + sqrt(s)). The column waits for these numbers, so
// the root and both quotients come from one hardware estimate of 1 / sqrt(s) and one of the
// reciprocal, each with two Newton steps (to a few units in the last place; s outside
// [1e-280, 1e280], where the products would leave the range, takes the library functions).
// tau is rounded to T because the back-transformation applies the stored one.
template <typename T>
__device__ __forceinline__ void reflector_of(double alpha, double xn2, double& beta, double& tau,
                                             double& scal) {
  if (xn2 == 0.0) {
    beta = alpha;
    tau = 0.0;
    scal = 0.0;
    return;
  }
  const double s = fma(alpha, alpha, xn2), aa = fabs(alpha);
  if (s > 1e-280 && s < 1e280) {
    double r = __builtin_amdgcn_rsq(s);
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const double hr = 0.5 * r;
      r = fma(hr, fma(-s * r, r, 1.0), r);
    }
    double nrm = s * r;
    nrm = fma(0.5 * r, fma(-nrm, nrm, s), nrm);
    const double den = aa + nrm;
    double q = __builtin_amdgcn_rcp(den);
#pragma unroll
    for (int it = 0; it < 2; ++it) q = fma(q, fma(-den, q, 1.0), q);
    beta = alpha >= 0.0 ? -nrm : nrm;
    tau = (double)(T)fma(aa, r, 1.0);
    scal = alpha >= 0.0 ? q : -q;
    return;
  }
  const double nrm = sqrt(s);
  beta = alpha >= 0.0 ? -nrm : nrm;
  tau = (double)(T)((beta - alpha) / beta);
  scal = 1.0 / (alpha - beta);
}

// barrier for data in LDS only: __syncthreads would also wait for the column's stores to memory,
// about as long as all the rest of a column takes
__device__ __forceinline__ void lds_barrier() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0); vmcnt, expcnt untouched (gfx9 encoding)
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}
// every store of this wave has reached the memory all compute units see
__device__ __forceinline__ void stores_done() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

}  // namespace

// ---------------------------------------------------------------------------------------------
// One workgroup per problem, trailing size m <= min(8 NW S, 8 Q). The 64 lanes of a wave form an
// 8 x 8 grid over the matrix: lane 8 lr + lc of wave w holds rows 8 w + lr + 8 NW s (s < S) and
// columns lc + 8 q (q < Q). A row's product is then summed over eight lanes, and eight rows at a
// time share the loads of v and w. The kernel is bound by instruction issue (one or two waves per
// SIMD, every instruction costs its four cycles), so what counts is their number: with a row per
// wave and step (64 lanes along the columns) the sums over the lanes and the readlanes of v_i, w_i
// outnumbered the products three to one (128 columns: 307 us against 209 us in this form; 64
// columns 110 us against 85 us; the blocked form took 2.6 ms and 1.3 ms).
// Vectors live twice: element l + 64 q in lane l of every wave (x, v, w; same bits everywhere),
// and in LDS, one copy per wave, in the order the grid reads. One barrier per column.
// ---------------------------------------------------------------------------------------------
// sums of S <= 4 values over the eight lanes of a row; lane lc returns value lc >> 1 (S > 2) or
// lc >> 2 (S <= 2)
template <int S>
__device__ __forceinline__ double octet_total(const double (&acc)[S], int lc) {
  double v;
  const bool up4 = lc & 4, up2 = lc & 2;
  if constexpr (S > 2) {
    const double a3 = S > 3 ? acc[S - 1] : 0.0;
    const double k0 = up4 ? acc[2] : acc[0], s0 = up4 ? acc[0] : acc[2];
    const double k1 = up4 ? a3 : acc[1], s1 = up4 ? acc[1] : a3;
    const double p0 = k0 + dpp<kHalfMirror>(s0), p1 = k1 + dpp<kHalfMirror>(s1);
    v = (up2 ? p1 : p0) + dpp<kQuadXor2>(up2 ? p0 : p1);
  } else {
    const double a1 = S > 1 ? acc[S - 1] : 0.0;
    v = (up4 ? a1 : acc[0]) + dpp<kHalfMirror>(up4 ? acc[0] : a1);
    v += dpp<kQuadXor2>(v);
  }
  return v + dpp<kQuadXor1>(v);
}

// row sums of all S rows of a lane group into y, four at a time
template <int S, int S0, int NW>
__device__ __forceinline__ void octet_store(const double (&acc)[S], int lc, int row0, double* y) {
  constexpr int N = S - S0 < 4 ? S - S0 : 4;
  double part[N];
#pragma unroll
  for (int s = 0; s < N; ++s) part[s] = acc[S0 + s];
  const double v = octet_total<N>(part, lc);
  constexpr int sh = N > 2 ? 1 : 2;
  if ((lc & ((1 << sh) - 1)) == 0 && (lc >> sh) < N) y[row0 + 8 * NW * (S0 + (lc >> sh))] = v;
  if constexpr (S0 + 4 < S) octet_store<S, S0 + 4, NW>(acc, lc, row0, y);
}

template <typename T, int NW, int S, int Q>
__global__ __launch_bounds__(64 * NW) void sytrd_wg_kernel(T* a, long lda, long sA, int n, int c0,
                                                           T* d, T* e, T* tauOut, long sV,
                                                           WgBatch bt) {
  constexpr int C = (Q + 7) / 8;        // elements per lane of a vector over the wave
  constexpr int QP = Q + 2;             // padded: the eight lanes of a read meet distinct banks
  constexpr int NV = 8 * QP, QG = 4;
  static_assert(Q % QG == 0, "sytrd_wg: shape");
  __shared__ double sVec[NW][3][NV];    // v of even and odd columns, w
  __shared__ double sY[2][8 * NW * S], sX[2][NV];
  long offA = blockIdx.x * sA, offV = blockIdx.x * sV;
  if (bt.list) {
    const int mol = bt.list[blockIdx.x];
    if (bt.active && !bt.active[mol]) return;
    offA = bt.aMul * bt.aOff[mol];
    offV = bt.vOff[mol];
    n = (int)(bt.vOff[mol + 1] - offV);
    lda = n;
    if (n > 8 * NW * S || n > 8 * Q) return;   // a size the shape does not hold: left alone
  }
  a += offA + c0 + (long)c0 * lda;
  d += offV + c0;
  e += offV + c0;
  tauOut += offV + c0;
  const int m = n - c0;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int lr = lane >> 3, lc = lane & 7;
  const int row0 = 8 * wv + lr;
  auto pos = [](int j) { return (j & 7) * QP + (j >> 3); };
  double A[S][Q], x[C];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int i = row0 + 8 * NW * s;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int j = lc + 8 * q;
      A[s][q] = (i < m && j < m) ? (double)a[max(i, j) + (long)min(i, j) * lda] : 0.0;
    }
  }
#pragma unroll
  for (int q = 0; q < C; ++q) x[q] = lane + 64 * q < m ? (double)a[lane + 64 * q] : 0.0;
  double* const w = sVec[wv][2];
  for (int i = lane; i < NV; i += 64) {
    sVec[wv][1][i] = 0.0;
    w[i] = 0.0;
  }
  for (int k = 0; k + 1 < m; ++k) {
    const int par = k & 1;
    double* const vn = sVec[wv][par];
    const double* const vo = sVec[wv][par ^ 1];
    double ss = 0.0;
#pragma unroll
    for (int q = 0; q < C; ++q)
      if (lane + 64 * q >= k + 2) ss += x[q] * x[q];
    const double xn2 = wave_total(ss);
    double beta, tau, scal;
    reflector_of<T>(element<C>(x, k + 1), xn2, beta, tau, scal);
    const double dk = element<C>(x, k);
    double v[C];
#pragma unroll
    for (int q = 0; q < C; ++q) {
      const int j = lane + 64 * q;
      v[q] = j <= k ? 0.0 : (j == k + 1 ? 1.0 : (double)(T)(x[q] * scal));
      if (j < 8 * Q) vn[pos(j)] = v[q];
    }
    // update of column k - 1's pair and y = A v on this lane's part
    double acc[S], vi[S], wi[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      acc[s] = 0.0;
      const int i = min(row0 + 8 * NW * s, 8 * Q - 1);
      vi[s] = vo[pos(i)];
      wi[s] = w[pos(i)];
    }
#pragma unroll
    for (int q0 = 0; q0 < Q; q0 += QG) {
      if (8 * (q0 + QG) - 1 <= k) continue;   // columns already reduced
      double vj[QG], oj[QG], wj[QG];
#pragma unroll
      for (int u = 0; u < QG; ++u) {
        vj[u] = vn[lc * QP + q0 + u];
        oj[u] = vo[lc * QP + q0 + u];
        wj[u] = w[lc * QP + q0 + u];
      }
#pragma unroll
      for (int s = 0; s < S; ++s) {
        if (8 * wv + 7 + 8 * NW * s <= k) continue;   // rows already reduced
#pragma unroll
        for (int u = 0; u < QG; ++u) {
          A[s][q0 + u] = fma(-wi[s], oj[u], fma(-vi[s], wj[u], A[s][q0 + u]));
          acc[s] = fma(A[s][q0 + u], vj[u], acc[s]);
        }
      }
    }
    // row k + 1 is the next column
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (row0 + 8 * NW * s == k + 1) {
#pragma unroll
        for (int q = 0; q < Q; ++q) sX[par][lc * QP + q] = A[s][q];
      }
    octet_store<S, 0, NW>(acc, lc, row0, sY[par]);
    lds_barrier();
    double y[C], an[C];
    double dt = 0.0;
#pragma unroll
    for (int q = 0; q < C; ++q) {
      const int j = lane + 64 * q, jc = min(j, m - 1);
      const bool on = j > k && j < m;
      y[q] = on ? tau * sY[par][jc] : 0.0;
      an[q] = on ? sX[par][pos(jc)] : 0.0;
      dt += y[q] * v[q];
    }
    const double h = -0.5 * tau * wave_total(dt);
#pragma unroll
    for (int q = 0; q < C; ++q) {
      y[q] += h * v[q];   // now w
      if (lane + 64 * q < 8 * Q) w[pos(lane + 64 * q)] = y[q];
    }
    const double wk = element<C>(y, k + 1);
#pragma unroll
    for (int q = 0; q < C; ++q) x[q] = an[q] - v[q] * wk - y[q];
    // the column goes out after the barrier: every wave has read its part of the matrix by then
    if (wv == (k & (NW - 1))) {
#pragma unroll
      for (int q = 0; q < C; ++q) {
        const int j = lane + 64 * q;
        if (j > k + 1 && j < m) a[j + (long)k * lda] = (T)v[q];
      }
      if (lane == 0) {
        a[k + (long)k * lda] = (T)dk;
        a[k + 1 + (long)k * lda] = (T)beta;
        d[k] = (T)dk;
        e[k] = (T)beta;
        tauOut[k] = (T)tau;
      }
    }
  }
  if (wv == 0) {
    const double dl = element<C>(x, m - 1);
    if (lane == 0) {
      a[m - 1 + (long)(m - 1) * lda] = (T)dl;
      d[m - 1] = (T)dl;
      tauOut[m - 1] = T(0);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// One matrix over P workgroups (blockIdx.y: problems of one size side by side), one workgroup
// per compute unit, all resident (cooperative launch). Workgroup p holds rows p + P s, thread t
// columns t + NT q of each of them.
//
// Exchange of a column: word i of a ring slot is row i's y, word mp + i its next-column element,
// written by the row's owner and polled by everyone (agent-scope 8-byte atomics, relaxed: each
// word carries its own validity, kEmpty until it is written, so no fence and no counter is
// needed). Three slots in turn. The thread that publishes row i sets the row's words of column
// k - 1 back to kEmpty when its workgroup has gathered column k (then every workgroup has read
// column k - 1, see ring_gathers), and waits for those stores before it publishes row i of column
// k + 1; a reader polls row i of column k + 2, in that same slot, only after it has gathered row i
// of column k + 1, so it can no longer meet the old words. A workgroup leaves when it has
// published its last row: rows are not read after their column, so its own words may stay. A wait
// is bounded; when one runs out the flag ends the others as well.
// ---------------------------------------------------------------------------------------------
constexpr u64 kEmpty = 0x7FF4D15EA5E0E5ADull;   // a signalling NaN that no operation returns

__device__ __forceinline__ u64 word_of(double v) {
  const u64 u = (u64)__double_as_longlong(v);
  return u == kEmpty ? 0x7FF8000000000000ull : u;
}
__device__ __forceinline__ void put(u64* p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 get(const u64* p) {
  return __hip_atomic_load(const_cast<u64*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ void ring_init_kernel(u64* ring, long sRing, int words, int* flag) {
  ring += blockIdx.y * sRing;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < words) ring[i] = kEmpty;
  if (i == 0 && blockIdx.y == 0) *flag = 0;
}

template <typename T, int NT, int R, int C>
__global__ __launch_bounds__(NT) void sytrd_grid_kernel(T* a, long lda, long sA, int n, int c0,
                                                        int kEnd, T* d, T* e, T* tauOut, long sV,
                                                        u64* ring, long sRing, int* flag,
                                                        long spinLimit) {
  constexpr int NW = NT / 64, mp = NT * C;   // mp words per vector in the ring
  __shared__ double sN[NW], sD[NW], sPart[NW][R], sv[R], sw[R], sx[R], sB[3];
  __shared__ int sStop;
  const int P = gridDim.x, p = blockIdx.x;
  const unsigned t = threadIdx.x;   // unsigned: addresses are a scalar base plus 8 t
  const int lane = t & 63, wv = t >> 6;
  a += blockIdx.y * sA + c0 + (long)c0 * lda;
  d += blockIdx.y * sV + c0;
  e += blockIdx.y * sV + c0;
  tauOut += blockIdx.y * sV + c0;
  ring += blockIdx.y * sRing;
  const int m = n - c0;
  const int kGather = ring_gathers(ring_last_row(p, P, m), kEnd);
  double A[R][C], x[C], vp[C], wp[C];
  int own[C];   // slot of row j if this workgroup holds it
#pragma unroll
  for (int q = 0; q < C; ++q) {
    const int j = (int)t + NT * q;
    own[q] = j < m && j % P == p ? j / P : -1;
    x[q] = j < m ? (double)(a + NT * q)[t] : 0.0;
    vp[q] = 0.0;
    wp[q] = 0.0;
  }
  // row by row (the fence keeps the addresses of all rows from being formed at once)
#pragma unroll
  for (int s = 0; s < R; ++s) {
    const int i = p + P * s;
#pragma unroll
    for (int q = 0; q < C; ++q) {
      const int j = (int)t + NT * q;
      A[s][q] = 0.0;
      if (i < m && j < m) {
        if (j > i) A[s][q] = (double)(a + (long)i * lda + NT * q)[t];
        else A[s][q] = (double)(a + i)[(long)j * lda];
      }
    }
    asm volatile("" ::: "memory");
  }
  // rows published by this thread: wave w sums and publishes rows 4 g .. 4 g + 3 of the workgroup,
  // g = w, w + NW, ..., lane 16 u row 4 g + u
  constexpr int NG = (R / 4 + NW - 1) / NW;
  int prow[NG];
#pragma unroll
  for (int u = 0; u < NG; ++u) {
    const int ps = 4 * (wv + NW * u) + (lane >> 4);
    prow[u] = ps < R && (lane & 15) == 0 && p + P * ps < m ? p + P * ps : -1;
  }
  if (t < R) {
    sv[t] = 0.0;
    sw[t] = 0.0;
  }
  if (t == 0) sStop = 0;
  double h = 0.0;
  int slot = 0;
  for (int k = 0; k < kEnd; ++k) {
    u64* ry = ring + 2 * slot * mp;
    u64* ra = ry + mp;
    // ---- reflector of column k
    double ss = 0.0;
#pragma unroll
    for (int q = 0; q < C; ++q) {
      const int j = (int)t + NT * q;
      if (j >= k + 2) ss += x[q] * x[q];
      if (j == k + 1) sB[0] = x[q];
      if (j == k) sB[1] = x[q];
    }
    ss = wave_total(ss);
    if (lane == 0) sN[wv] = ss;
    lds_barrier();
    const double xn2 = part_total<NW>(sN[lane & (NW - 1)]);
    double beta, tau, scal;
    reflector_of<T>(sB[0], xn2, beta, tau, scal);
    const double dk = sB[1];
    double v[C];
#pragma unroll
    for (int q = 0; q < C; ++q) {
      const int j = (int)t + NT * q;
      v[q] = j <= k ? 0.0 : (j == k + 1 ? 1.0 : (double)(T)(x[q] * scal));
    }
    // ---- rank-two update of column k - 1 and y = A v
#pragma unroll
    for (int g = 0; g < R; g += 4) {
      double acc[4] = {0.0, 0.0, 0.0, 0.0};
      if (p + P * (g + 3) <= k) continue;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int s = g + u;
        const double vi = sv[s], wi = sw[s] + h * vi;
#pragma unroll
        for (int q = 0; q < C; ++q) {
          A[s][q] = fma(-wi, vp[q], fma(-vi, wp[q], A[s][q]));
          acc[u] = fma(A[s][q], v[q], acc[u]);
        }
      }
      const double yr = rows_total4(acc, lane);
      if ((lane & 3) == 0 && lane < 16) sPart[wv][g + (lane >> 2)] = yr;
    }
#pragma unroll
    for (int q = 0; q < C; ++q)
      if ((int)t + NT * q == k + 1) {
#pragma unroll
        for (int s = 0; s < R; ++s) sx[s] = A[s][q];
      }
    lds_barrier();
    stores_done();   // the words emptied in the last column
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      const int ps = min(4 * (wv + NW * u) + (lane >> 4), R - 1);
      const double y = part_total<NW>(sPart[lane & (NW - 1)][ps]);
      if (ring_published(prow[u], k)) {
        put(ry + prow[u], word_of(y));
        put(ra + prow[u], word_of(sx[ps]));
      }
    }
    const bool leaves = k == kGather;   // its last row is out
    if (!leaves) {
      // ---- gather y and the next column
      u64 uy[C], ua[C];
#pragma unroll
      for (int q = 0; q < C; ++q) {
        const int j = (int)t + NT * q;
        uy[q] = j > k && j < m ? kEmpty : 0;   // 0.0 where there is nothing to gather
        ua[q] = uy[q];
      }
      // Nothing can have arrived yet, and polls slow down the words on their way: at 1024
      // columns 4.6 us per column without this wait, 3.8 with 8 units of 64 clocks, 2.9 with 16
      // to 20, 3.2 with 32.
      __builtin_amdgcn_s_sleep(18);
      for (long spins = 0;; ++spins) {
        // the missing words, all loaded before the first is looked at: one trip to memory, not 2 C
#pragma unroll
        for (int q = 0; q < C; ++q) {
          if (uy[q] == kEmpty) uy[q] = get(ry + NT * q + t);
          if (ua[q] == kEmpty) ua[q] = get(ra + NT * q + t);
        }
        bool ok = true;
#pragma unroll
        for (int q = 0; q < C; ++q) ok = ok && uy[q] != kEmpty && ua[q] != kEmpty;
        if (ok) break;
        if ((spins & 1023) == 1023 || spins > spinLimit) {
          if (spins > spinLimit)
            __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          if (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
            sStop = 1;
            break;
          }
        }
        __builtin_amdgcn_s_sleep(1);
      }
      double y[C], an[C];
#pragma unroll
      for (int q = 0; q < C; ++q) {
        y[q] = __longlong_as_double((long long)uy[q]);
        an[q] = __longlong_as_double((long long)ua[q]);
      }
      // ---- w and the next column
      double dt = 0.0;
#pragma unroll
      for (int q = 0; q < C; ++q) {
        const int j = (int)t + NT * q;
        y[q] *= tau;
        dt += y[q] * v[q];
        if (j == k + 1) sB[2] = y[q];
        if (own[q] >= 0) {
          sv[own[q]] = v[q];
          sw[own[q]] = y[q];
        }
      }
      dt = wave_total(dt);
      if (lane == 0) sD[wv] = dt;
      lds_barrier();
      if (sStop) return;
      h = -0.5 * tau * part_total<NW>(sD[lane & (NW - 1)]);
      const double wk = sB[2] + h;
#pragma unroll
      for (int q = 0; q < C; ++q) {
        vp[q] = v[q];
        wp[q] = y[q] + h * v[q];
        x[q] = (int)t + NT * q > k ? an[q] - v[q] * wk - wp[q] : 0.0;
      }
      // this workgroup has gathered column k, so its words of column k - 1 are no longer needed
      if (k > 0) {
        u64* oy = ring + 2 * (slot == 0 ? kRingSlots - 1 : slot - 1) * mp;
#pragma unroll
        for (int u = 0; u < NG; ++u)
          if (ring_emptied(prow[u], k)) {
            put(oy + prow[u], kEmpty);
            put(oy + mp + prow[u], kEmpty);
          }
      }
    }
    // ---- the column goes out, over what every workgroup has read into registers: it has
    // published column k - 1 (or 0, which no workgroup leaves: it has four rows or more)
    if (p == (k + 1) % P) {
#pragma unroll
      for (int q = 0; q < C; ++q) {
        const int j = (int)t + NT * q;
        if (j > k + 1 && j < m) (a + (long)k * lda + NT * q)[t] = (T)v[q];
      }
      if (t == 0) {
        a[k + (long)k * lda] = (T)dk;
        a[k + 1 + (long)k * lda] = (T)beta;
        d[k] = (T)dk;
        e[k] = (T)beta;
        tauOut[k] = (T)tau;
      }
    }
    if (leaves) return;
    slot = slot == kRingSlots - 1 ? 0 : slot + 1;
  }
  // the trailing matrix goes back (lower triangle) for the one-workgroup kernel
#pragma unroll
  for (int s = 0; s < R; ++s) {
    const int i = p + P * s;
    if (i < kEnd || i >= m) continue;
    const double vi = sv[s], wi = sw[s] + h * vi;
#pragma unroll
    for (int q = 0; q < C; ++q) {
      const int j = (int)t + NT * q;
      if (j >= kEnd && j <= i)
        a[i + (long)j * lda] = (T)fma(-wi, vp[q], fma(-vi, wp[q], A[s][q]));
    }
  }
}

// ---------------------------------------------------------------------------------------------
// launches
// ---------------------------------------------------------------------------------------------
// Largest trailing size of the one-workgroup kernel; the grid hands over there. Per column at 128
// columns the grid takes 2.5 us (two trips to memory and the wait) and one workgroup 1.9 us; an
// eight-wave form for 192 columns took 3.1 us per column above 128.
constexpr int kWgMax = 128;

template <typename T>
static int wg_launch(hipStream_t s, T* a, long lda, long sA, int n, int c0, T* d, T* e, T* tau,
                     long sV, int K) {
  const int m = n - c0;
#define DH_WG(NW_, S_, Q_)                                                                     \
  hipLaunchKernelGGL((sytrd_wg_kernel<T, NW_, S_, Q_>), dim3(K), dim3(64 * NW_), 0, s, a, lda, sA, \
                     n, c0, d, e, tau, sV, WgBatch{})
  if (m <= 32) DH_WG(4, 1, 4);
  else if (m <= 64) DH_WG(4, 2, 8);
  else DH_WG(4, 4, 16);
#undef DH_WG
  DH_LAUNCH_CHECK();
  return 0;
}

// Compiled shapes of the grid kernel: NT threads of C columns hold trailing sizes up to NT C, with
// R rows per workgroup; the first that fits the size and the compute units is taken, few rows
// (many workgroups) first. Per column, one problem: 2.9 us with 4 rows, 3.2 with 8, 3.6 with 16
// at 1024 columns; 4 waves rather than 8 wherever the registers allow it, since every wave repeats
// the vector work. Several problems share the compute units, so they need the shapes of many
// rows. Beyond 2560 columns a thread's share no longer fits 256 registers (12 x 6 elements spilled
// and ran at 11 us per column, no faster than the blocked form there).
struct GridShape {
  int nt, r, c;
  const void* fn;
};
template <typename T>
static const GridShape* grid_shape(int m, int maxP) {
#define DH_SHAPE(NT_, R_, C_) {NT_, R_, C_, (const void*)sytrd_grid_kernel<T, NT_, R_, C_>}
  static const GridShape shapes[] = {
      DH_SHAPE(256, 4, 1), DH_SHAPE(256, 8, 1), DH_SHAPE(256, 16, 1), DH_SHAPE(256, 32, 1),
      DH_SHAPE(256, 4, 2), DH_SHAPE(256, 8, 2), DH_SHAPE(256, 16, 2), DH_SHAPE(256, 32, 2),
      DH_SHAPE(256, 4, 4), DH_SHAPE(256, 8, 4), DH_SHAPE(256, 16, 4), DH_SHAPE(512, 32, 2),
      DH_SHAPE(256, 8, 8), DH_SHAPE(512, 16, 4), DH_SHAPE(512, 12, 5)};
#undef DH_SHAPE
  for (const GridShape& g : shapes)
    if (m <= g.nt * g.c && (m + g.r - 1) / g.r <= maxP) return &g;
  return nullptr;
}

int sytrd_wg_batch(hipStream_t s, double* a, int count, int maxN, const WgBatch& bt, double* d,
                   double* e, double* tau) {
  if (count <= 0) return 0;
  DH_CHECK(bt.list && bt.aOff && bt.vOff && maxN <= kWgBatchMax, "sytrd_wg_batch: bad arguments");
  // 192 columns fit eight waves without spills (379 us for 190); 224 columns leave too few
  // registers either way, and four waves spill least (680 us for 190)
#define DH_WGB(NW_, S_, Q_)                                                                    \
  hipLaunchKernelGGL((sytrd_wg_kernel<double, NW_, S_, Q_>), dim3(count), dim3(64 * NW_), 0, s, \
                     a, 0L, 0L, 0, 0, d, e, tau, 0L, bt)
  if (maxN <= 32) DH_WGB(4, 1, 4);
  else if (maxN <= 64) DH_WGB(4, 2, 8);
  else if (maxN <= 128) DH_WGB(4, 4, 16);
  else if (maxN <= 192) DH_WGB(8, 3, 24);
  else DH_WGB(4, 7, 28);
#undef DH_WGB
  DH_LAUNCH_CHECK();
  return 0;
}

static int cu_count(int* out) {
  int dev = 0;
  DH_HIP(hipGetDevice(&dev));
  DH_HIP(hipDeviceGetAttribute(out, hipDeviceAttributeMultiprocessorCount, dev));
  return 0;
}

int sytrd_resident_from(int n, int K, int* c0) {
  constexpr int kPanel = 64;   // the blocked form stops at panel ends
  int cus = 0;
  DH_TRY(cu_count(&cus));
  *c0 = 0;
  while (*c0 < n && n - *c0 > kWgMax && !grid_shape<double>(n - *c0, cus / K)) *c0 += kPanel;
  *c0 = std::min(*c0, n);
  return 0;
}

template <typename T>
int sytrd_resident(hipStream_t s, T* a, long lda, long sA, int n, int c0, T* d, T* e, T* tau,
                   long sV, u64* ring, long sRing, int* flag, int K, bool* done) {
  *done = false;
  int m = n - c0;
  if (m > kWgMax) {
    int cus = 0;
    DH_TRY(cu_count(&cus));
    const GridShape* g = grid_shape<T>(m, cus / K);
    DH_CHECK(g, "sytrd: trailing matrix too large for the resident kernels");
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    DH_HIP(hipStreamIsCapturing(s, &cap));
    if (cap != hipStreamCaptureStatusNone) return 0;   // no cooperative launch in a graph
    const int P = (m + g->r - 1) / g->r;
    DH_CHECK(6 * g->nt * g->c <= kResidentWords * m, "sytrd: exchange ring too small");
    int kEnd = m - kWgMax;
    long spinLimit = 1L << 24;
    hipLaunchKernelGGL(ring_init_kernel, dim3(cdiv(6L * g->nt * g->c, 256), K), dim3(256), 0, s, ring,
                       sRing, 6 * g->nt * g->c, flag);
    DH_LAUNCH_CHECK();
    void* args[] = {&a, &lda, &sA, &n, &c0, &kEnd, &d, &e, &tau, &sV, &ring, &sRing, &flag, &spinLimit};
    const hipError_t err = hipLaunchCooperativeKernel(g->fn, dim3(P, K), dim3(g->nt), args, 0, s);
    if (err == hipErrorIllegalState || err == hipErrorCooperativeLaunchTooLarge ||
        err == hipErrorNotSupported) {
      (void)hipGetLastError();   // the refused launch ran nothing
      return 0;
    }
    DH_HIP(err);
    int ended = 0;
    DH_HIP(hipMemcpyAsync(&ended, flag, sizeof(int), hipMemcpyDeviceToHost, s));
    DH_HIP(hipStreamSynchronize(s));
    if (ended != 0) {
      set_error("sytrd: a wait between workgroups ran out");
      return kErrDevice;
    }
    c0 += kEnd;
  }
  DH_TRY(wg_launch<T>(s, a, lda, sA, n, c0, d, e, tau, sV, K));
  *done = true;
  return 0;
}
template int sytrd_resident<double>(hipStream_t, double*, long, long, int, int, double*, double*,
                                    double*, long, u64*, long, int*, int, bool*);
template int sytrd_resident<float>(hipStream_t, float*, long, long, int, int, float*, float*,
                                   float*, long, u64*, long, int*, int, bool*);

}  // namespace dftbhip
