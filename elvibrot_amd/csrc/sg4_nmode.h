// Potentials that are sums of one- and two-mode functions: H as one sparse
// matrix over the packed rows (see sg4_nmode.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "sg4_buf.h"
#include "sg4_device.h"

namespace sg4 {

// H as CSR over the packed rows of a plan, the diagonal entry first in its
// row; with a field also the dipole operator's values on the same pattern.
// The buffers are kept and reused when the matrix is built again.
struct NModeMat {
  bool valid = false;
  int64_t rows = 0, nnz = 0;
  DevBuf ptr, col, val;   // int64 row pointers, int32 columns, FP64 values
  DevBuf val_mu, val_f;   // field matrices: values of mu; val + eps val_mu of the segment
};

// One instance of a plan, as the construction sees it.
struct NModeInst {
  int D, L, Lmax;         // L: largest |l| of its terms
  int64_t nterms, nb_ba, term0, row0, md0, ck0, lev0;
};

// The plan's host and device tables that the construction reads.
struct NModeIn {
  std::vector<NModeInst> inst;
  const std::vector<int32_t>* levels;
  const std::vector<int32_t>* nq;      // per md: points = functions (square modes)
  const std::vector<int64_t>* qoff;
  const std::vector<double>* ck;
  const std::vector<double>* T;        // kinetic matrices BtW D2 B, rounding entries zeroed
  const std::vector<int64_t>* toff;    // per md
  const TermDev* d_terms;
  const MatDev* d_md;
  const double* d_mats;
  const int32_t* d_levels;
  const int32_t* d_map;
  int64_t sum_nq, rows;
  hipStream_t stream;
};

// Index tables of a plan (they depend on its tables only, not on V).
struct NModeTables;
NModeTables* nmode_tables_create(const NModeIn& in);   // null: HIP failure
void nmode_tables_destroy(NModeTables* t);

// Builds the matrix of the device grid V and the kinetic part; with mu also
// the values of the grid function mu as an operator.  m.valid says whether
// there is one: V (and mu) must be sums of one- and two-mode functions to
// rounding on every grid point, the packed rows in lexicographic order, and
// the matrix small enough to pay.  Synchronises the stream.
int nmode_build(NModeTables* t, const NModeIn& in, const double* V, const double* mu, NModeMat& m);

// hpsi = M psi, nvec vectors in the rows layout
int nmode_apply(const NModeMat& m, int nvec, const double* psi, double* hpsi, hipStream_t st);
// The same to a column-major result, W >= nvec columns at a time: from a
// column-major block (small blocks, nmode_cols_direct) or from a rows-layout
// block of W columns.  1: no kernel for this W.
bool nmode_cols_direct(const NModeMat& m, int W);
int nmode_apply_cols(const NModeMat& m, int W, int nvec, const double* psi, double* hpsi, hipStream_t st);
int nmode_apply_to_cols(const NModeMat& m, int W, int nvec, const double* psi, double* hpsi, hipStream_t st);

}  // namespace sg4
