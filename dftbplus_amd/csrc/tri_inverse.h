// Inverse of a lower triangular matrix in LDS by one workgroup: 16 x 16 diagonal blocks by
// forward substitution (a thread per column), then pairs of blocks joined by doubling,
//   [A 0; B C]^-1 = [A^-1 0; -C^-1 B A^-1  C^-1],
// so that a matrix of 64 takes 1 + 2 x 2 steps and one of 128 1 + 3 x 2, each using all
// threads, where a column-by-column recurrence takes one step per column.
#pragma once

#include <hip/hip_runtime.h>

namespace dftbhip {

// X (NB x NB, leading dimension LD, X[row * LD + col]) <- inverse of its lower triangle; the
// strict upper triangle is scratch. 256 threads, all of them; ends with a barrier.
template <typename T, int NB, int LD>
__device__ __forceinline__ void lower_inverse_lds(T* X) {
  const int t = threadIdx.x;
  if (t < NB) {
    const int b0 = t & ~15, c = t & 15;
    T x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const T r = T(1) / X[(b0 + i) * LD + b0 + i];
      T acc = T(0);
#pragma unroll
      for (int k = 0; k < i; ++k) acc += X[(b0 + i) * LD + b0 + k] * x[k];
      x[i] = i < c ? T(0) : (i == c ? r : -acc * r);
    }
    // all reads of a block are in this wave and before its writes
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (i >= c) X[(b0 + i) * LD + b0 + c] = x[i];
  }
  __syncthreads();
#pragma unroll
  for (int b = 16; b < NB; b *= 2) {
    // NB / (2 b) pairs, 256 / pairs threads each; a thread forms 4 rows x CB columns
    constexpr int kThreads = 256;
    const int pairs = NB / (2 * b), per = kThreads / pairs;
    const int pr = t / per, u = t % per;
    const int r0 = 2 * b * pr, r1 = r0 + b;      // first rows of A and of C
    const int rb = b / 4;                        // groups of four rows
    const int cb = b * b >= 4 * per ? b * b / per / 4 : 1;   // columns per thread (1, 2 or 4)
    const int i0 = 4 * (u % rb), j0 = cb * (u / rb);
    const bool on = j0 < b;                      // a pair of 16s has work for 64 threads
    T acc[4][4];
    // tmp = B A^-1, kept in the block above the diagonal
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[p][q] = T(0);
    for (int k = on ? j0 : b; k < b; ++k) {
      T l[4], r[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) l[p] = X[(r1 + i0 + p) * LD + r0 + k];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        r[q] = q < cb && k >= j0 + q ? X[(r0 + k) * LD + r0 + j0 + q] : T(0);
#pragma unroll
      for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[p][q] += l[p] * r[q];
    }
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (on && q < cb) X[(r0 + i0 + p) * LD + r1 + j0 + q] = acc[p][q];
    __syncthreads();
    // B <- -C^-1 tmp
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[p][q] = T(0);
    for (int k = on ? 0 : i0 + 4; k < i0 + 4; ++k) {
      T l[4], r[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) l[p] = k <= i0 + p ? X[(r1 + i0 + p) * LD + r1 + k] : T(0);
#pragma unroll
      for (int q = 0; q < 4; ++q) r[q] = q < cb ? X[(r0 + k) * LD + r1 + j0 + q] : T(0);
#pragma unroll
      for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[p][q] += l[p] * r[q];
    }
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (on && q < cb) X[(r1 + i0 + p) * LD + r0 + j0 + q] = -acc[p][q];
    __syncthreads();
  }
}

}  // namespace dftbhip
