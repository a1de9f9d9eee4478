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
// Many tridiagonals at once: block p has n rows, its d, e, w at off, its matrices within the
// work buffers at q and its z (n x n, leading dimension ldz) at z. prepare makes the tables
// (copies to the device, not under stream capture) and says how many doubles of work a solve
// needs; a solve is launches only and leaves the blocks with active[id] == 0 alone (active may be
// null). stedc_info: a failure word per block (device; 0 solved, -1 left alone).
struct DcBlock {
  int n;
  long off, q, z, ldz;
  int id;
  bool operator==(const DcBlock& o) const {
    return n == o.n && off == o.off && q == o.q && z == o.z && ldz == o.ldz && id == o.id;
  }
};
int stedc_many_prepare(hipStream_t s, const std::vector<DcBlock>& blocks, StedcWs* ws,
                       size_t* workSize);
int stedc_many(hipStream_t s, const double* d, const double* e, double* w, double* z,
               double* work, const int* active, StedcWs* ws);
const int* stedc_info(const StedcWs* ws);

}  // namespace dftbhip
