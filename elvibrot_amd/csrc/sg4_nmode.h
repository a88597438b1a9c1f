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
  int64_t rows = 0, nnz = 0, longest = 0;   // longest: entries of the longest row
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
NModeTables* nmode_tables_create(const NModeIn& in);   // null: HIP failure; without rows_ok where memory is short
void nmode_tables_destroy(NModeTables* t);

// Whether the packed rows are in lexicographic order (the last mode's index
// fastest), and the kinetic part K alone for such rows.  Both builders return
// with the last kernels enqueued on in.stream.
bool nmode_rows_ok(const NModeTables* t);
int nmode_build_kinetic(NModeTables* t, const NModeIn& in, NModeMat& m);

// Builds the matrix of the device grid V and the kinetic part; with mu also
// the values of the grid function mu as an operator.  m.valid says whether
// there is one: V (and mu) must be sums of one- and two-mode functions to
// rounding on every grid point, the packed rows in lexicographic order, and
// the matrix small enough to pay.
int nmode_build(NModeTables* t, const NModeIn& in, const double* V, const double* mu, NModeMat& m);

// us that building the plan's matrix m again with a grid function's values takes
double nmode_field_cost(const NModeTables* t, const NModeMat& m);

// hpsi = M psi, nvec vectors in the rows layout (val: other values on M's pattern;
// psi32: psi in FP32, written beside it)
int nmode_apply(const NModeMat& m, int nvec, const double* psi, double* hpsi, hipStream_t st,
                const double* val = nullptr, float* psi32 = nullptr);
// The same to a column-major result, W >= nvec columns at a time: from a
// column-major block (small blocks, nmode_cols_direct) or from a rows-layout
// block of W columns.  1: no kernel for this W.
bool nmode_cols_direct(const NModeMat& m, int W);
int nmode_apply_cols(const NModeMat& m, int W, int nvec, const double* psi, double* hpsi, hipStream_t st);
int nmode_apply_to_cols(const NModeMat& m, int W, int nvec, const double* psi, double* hpsi, hipStream_t st);
// val_f = val + eps val_mu
int nmode_set_field(const NModeMat& m, double eps, hipStream_t st);

// The plan's field-free FP64 operator as such a matrix, with mu's values (mu
// null: none), for about `applies` applies; *out is null when there is none or
// it would not pay.  The matrix belongs to the plan and is rebuilt by the next
// call.
int plan_field_matrix(sg4_plan* p, const double* mu, int prec, int64_t applies, NModeMat** out);
// whether the plan is the operator of the grid function mu alone (no kinetic
// part), over H's terms and grids (mu has a value per grid point of H) and free
// to run as a matrix
int plan_is_grid_function(const sg4_plan* p, const sg4_plan* H, const double* mu, hipStream_t st, bool* same);
// around a product with such a matrix, what an apply of the plan records: the
// statistics and, with timing on, the events
int plan_product_begin(sg4_plan* p, int nvec);
int plan_product_end(sg4_plan* p);
// takes a field left on the plan back
int plan_clear_field(sg4_plan* p);

// One Chebyshev order on ns complex states (columns [re | im], 2 ns), or on
// states and tangents ([re | im | t_re | t_im], 4 ns), in the pass that forms
// y = H w_k (val: the matrix values of the segment):
//   z = (y - E0 w_k + [t: mu w_k]) sc,  w_{k+1} = w_{k-1} + 2 r z  (first: r z)
// with r = sgn i, written over wm; acc = [first: c0 w_0 else acc] + c w_{k+1},
// of the states in acc, of the tangents in tacc (2 ns columns each).  last:
// acc times the phase goes to out (and tout) instead.
struct NModeOrder {
  const double* val;
  const double* wk;
  double* wm;
  double *acc, *tacc, *out, *tout;
  double c0, c, E0, sc, sgn, pr, pi;
  int first, last, ns;
};
bool nmode_order_width(int ncol);    // columns the order kernel takes
int nmode_order(const NModeMat& m, const NModeOrder& a, bool tangent, hipStream_t st);

}  // namespace sg4
