// Tridiagonal divide and conquer on the device (stedc.hip): interfaces that need no host data.
#pragma once

#include <vector>

#include "common.h"

namespace dftbhip {

using u64 = unsigned long long;

// Eigenvalues (ascending, w) and eigenvectors (z, n x n, leading dimension ldz) of the device
// tridiagonal (d, e); only launches (tables and buffers are made on the first call of a size).
// work: stedc_work_size(n) doubles. stedc_fetch copies the eigenvalues and the QL failure word
// (0: none) to the host and waits.
int stedc_device(hipStream_t s, int n, const double* d, const double* e, double* w, double* z,
                 long ldz, double* work, size_t workSize, StedcWs* ws);
int stedc_fetch(hipStream_t s, int n, const double* w, double* wHost, StedcWs* ws, int* info);
// Many tridiagonals at once: problem p's d, e, w at the sum of the sizes before it, its z (n x n,
// leading dimension n) at the sum of their squares. work: 4 sum n^2 doubles. stedc_info: a failure
// word per problem (device).
int stedc_many(hipStream_t s, const std::vector<int>& sizes, const double* d, const double* e,
               double* w, double* z, double* work, StedcWs* ws);
const int* stedc_info(const StedcWs* ws);

}  // namespace dftbhip
