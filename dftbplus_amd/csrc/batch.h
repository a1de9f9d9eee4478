// Per-molecule layout of a molecule batch and the batched kernels (batch.hip).
#pragma once

#include <memory>
#include <vector>

#include "sparse.h"
#include "stedc.h"

namespace dftbhip {

constexpr int kBatchMaxOrb = 512;   // orbitals per molecule in a batch
// size classes of the batched eigensolver, by orbital count (largest first): above kWgBatchMax
// Jacobi with both matrices in HBM, up to it the direct solve, whose reduction has shapes for
// 224, 192, 128, 64 and 32 orbitals. Molecules of up to kBatchSmall orbitals are swept by Jacobi
// in LDS if the batch has none that is solved directly: the sweeps save the direct solve's
// launches, which cost nothing where a larger molecule needs them, and would be one more branch
// beside the classes' reductions (32 molecules of 13 to 190 orbitals: 15.5 ms with the sweeps,
// 13.9 without).
constexpr int kBatchSmall = 16;
constexpr int kBatchJacobi = 6;   // the class of the smallest
constexpr int kBatchClasses = 7;
inline bool batch_direct(long n) { return n > kBatchSmall && n <= kWgBatchMax; }
// anyDirect: batch_direct holds for some molecule of the batch
inline int batch_class(long n, bool anyDirect) {
  return n > kWgBatchMax ? 0 : n > 192 ? 1 : n > 128 ? 2 : n > 64 ? 3 : n > 32 ? 4
         : n > kBatchSmall || anyDirect ? 5 : kBatchJacobi;
}
// info of a molecule whose eigensolver did not converge within its limit (distinct from the
// leading minor of a non-positive-definite overlap)
constexpr int kBatchEigenNoConv = 1 << 24;

struct BatchLayout {
  int nmol;
  const int* atom0;     // nmol + 1: first atom of each molecule
  const long* orb0;     // nmol + 1: first orbital
  const long* dOff;     // nmol + 1: offsets of the packed n_m x n_m dense matrices
  const long* gOff;     // nmol + 1: offsets of the packed nat_m x nat_m gamma matrices
  const int* atomMol;   // molecule of each atom
  const int* order;     // nmol: molecules by decreasing orbital count (launch order)
  int ncls[kBatchClasses];   // molecules per size class, largest class first, in order
};

int launch_batch_unpack(hipStream_t s, const PairsDev& pr, const int* norb,
                        const long* iAtomStart, const BatchLayout& L, const double* x,
                        double* dense, long denseSize);
int launch_batch_pack(hipStream_t s, const PairsDev& pr, const int* norb, const long* iAtomStart,
                      const BatchLayout& L, const double* dense, double* x);
// Buffers and tables of the batched eigensolver for one set of geometries
struct BatchDescs {
  GemmDesc<double>*hc, *chc, *back;
  int* solve;   // per molecule: solved in this call
};
constexpr int kFactorNB = 64;   // panel of the overlap factorisation (potrf_diag's block)
struct FactorStep {
  int panel, count, m, n;   // panel the products belong to (-1: joining of blocks), their extent
  long first;               // first descriptor
};
struct BatchEigen {
  int first[kBatchClasses + 1] = {}, maxn[kBatchClasses] = {}, direct = 0;
  std::shared_ptr<StedcWs> dc;
  DevBuf<double> work, vec;
  double *d = nullptr, *e = nullptr, *tau = nullptr;   // in vec
  DevBuf<GemmDesc<double>> desc, factorDesc;
  std::vector<FactorStep> steps;
  DevBuf<int> solve;
  int prepare(hipStream_t s, const BatchLayout& L, const std::vector<int>& order,
              const std::vector<long>& orb0, const std::vector<long>& dOff, double* matrices,
              double* C);
  int maxDirect() const {
    int n = 0;
    for (int c = 1; c < kBatchJacobi; ++c) n = n > maxn[c] ? n : maxn[c];
    return n;
  }
};
// eigenvalues w (ascending per molecule, at orb0), eigenvectors C (packed), info per molecule
// (0, or j+1 when the leading minor j+1 of S is not positive definite); work 3 x packed size,
// kept between calls. Molecules with active[m] == 0 are skipped (active may be null: all).
// warm: S is the one of the previous call on the same work array (a cold call factors S; the
// Jacobi sweeps of the largest and smallest molecules then start from that call's eigenvectors).
// s: the stream of the call; st[c]: that of class c, s itself or one forked from it by the caller
// and joined afterwards; done[0 .. kBatchClasses-1]: events for the forks in between. Launches
// only, so a call can be captured.
int launch_batch_sygv(hipStream_t s, const hipStream_t* st, BatchEigen& E, const BatchLayout& L,
                      const double* S, const double* H, double* work, double* w, double* C,
                      int* info, const int* active, bool warm, hipEvent_t* done);
// P = C diag(f) C^T over the first nocc columns; work as above (B1 is overwritten)
int launch_batch_density(hipStream_t s, BatchEigen& E, const BatchLayout& L, const double* C,
                         const double* f, const int* nocc, double* P, const int* active,
                         double* work);
int launch_batch_gamma(hipStream_t s, const BatchLayout& L, const double* coords,
                       const int* species, const double* hubbu, const double* gcut, int nsp,
                       double* g);
int launch_batch_gemv(hipStream_t s, const BatchLayout& L, int nat, const double* g,
                      const double* dq, double* v);
int launch_batch_invr_grad(hipStream_t s, const BatchLayout& L, int nat, const double* coords,
                           const double* dq, double* grad);

// Device state of a molecule batch's SCC cycle (batch_scc.hip): per atom (nat) and per molecule
// (nmol) arrays, the Broyden histories (maxHist steps: ww, cc per molecule; aa, B maxHist^2 per
// molecule; dF, uu one vector of all atoms per step) and four counters: iteration, molecules
// still iterating, failure code (1 eigensolver, 2 Fermi level, 3 mixer history) and the lowest
// failing molecule.
struct BatchSccDev {
  int nmol, nat, maxHist;
  const int* atom0;
  const long* orb0;
  const double* q0;
  const double* nel;
  double *qin, *qout, *dq, *tmp;
  int *conv, *active, *iters, *nocc, *mixIt, *counters;
  double *err, *ef, *eband, *ts, *e0, *eNonScc, *eScc;
  double *ww, *aa, *B, *cc, *dF, *uu, *qlast, *dlast;
  double kT, sccTol, alpha, omega0, minw, maxw, wfac;
  int minSccIter, maxSccIter;
};
int launch_bscc_reset(hipStream_t s, const BatchSccDev& d);
int launch_bscc_begin(hipStream_t s, const BatchSccDev& d);
int launch_bscc_info(hipStream_t s, const BatchSccDev& d, const int* info);
int launch_bscc_fermi(hipStream_t s, const BatchSccDev& d, const double* w, double* fill);
int launch_bscc_outputs(hipStream_t s, const BatchSccDev& d, const long* atomStart,
                        const int* atomMol, const double* qorb, const double* eorb);
int launch_bscc_mix(hipStream_t s, const BatchSccDev& d, const double* vout);

}  // namespace dftbhip
