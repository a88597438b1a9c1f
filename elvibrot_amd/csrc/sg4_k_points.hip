// Type-10 and general type-1 operators, FP64, one thread per output value.
//
// Their terms are small (the work buffers of a term fit 64 KiB) and there are
// few of them, so the passes of one term are a serial chain that decides the
// time: a pass with one thread per fibre keeps N nv / n threads busy with n^2
// multiply-adds each (two waves for a 640-point term), one thread per value
// keeps N nv busy with n.  The tensors sit in LDS, element (point p, vector v)
// at [v + nv p], and (STAGE) the term's 1-D matrices beside them (3D Jacobi L=6
// x1 13.0 -> 12.8 us, 4D L=4 type 1 17.4 -> 16.4); matrices too large for that
// are read through the vector cache.  psi and H.psi are taken as they lie
// (column-major blocks need no layout kernels).
// Whole applies, us, fibres before -> values now: 3D Jacobi L=10 x5 78 -> 33,
// L=12 x24 504 -> 244, L=6 x1 26 -> 13; general type 1 5D L=5 x4 79 -> 26, 6D L=6
// x16 456 -> 297, 4D L=4 x1 47 -> 16.  With 384 / 256 threads (type 10 / type 1);
// 256 / 128: 41 / 29 for the first of each, 512 / 384: 35 / 29; eight loads in
// flight per value instead of four: 35 / 32.
#include "sg4_device.h"

namespace sg4 {

namespace {

constexpr int DMAX = MAXACT;   // modes of a term

// The modes of a term: sizes, point strides, and offsets of the matrices (in
// LDS or in the plan's array), in LDS (read at wave-uniform indices).
struct PModes {
  int nq[DMAX], nb[DMAX], A[DMAX];   // A: stride of the mode on the grid
  float invA[DMAX], invq[DMAX];
  int B[DMAX], Bt[DMAX], D1[DMAX], D2[DMAX];
};

// Fills m; STAGE: copies the matrices (B, BtW, D1 and with d2 D2) to ms.  The
// caller synchronises.
template <bool STAGE>
__device__ __forceinline__ void load_modes(PModes& m, const PArgs& a, const double* mats, const TermDev* Td,
                                           double* ms, bool d2) {
  const int D = Td->nact;
  int off = 0, A = 1;
  for (int k = 0; k < D; ++k) {
    const MatDev& q = a.md[Td->mat[k]];
    const int nq = q.nq, nb = q.nb, nm = nq * nb, ng = nq * nq;
    if (threadIdx.x == 0) {
      m.nq[k] = nq; m.nb[k] = nb; m.A[k] = A;
      m.invA[k] = 1.0f / (float)A; m.invq[k] = 1.0f / (float)nq;
      m.B[k] = STAGE ? off : (int)q.B;
      m.Bt[k] = STAGE ? off + nm : (int)q.BtW;
      m.D1[k] = STAGE ? off + 2 * nm : (int)q.D1;
      m.D2[k] = STAGE ? off + 2 * nm + ng : (int)q.D2;
    }
    if constexpr (STAGE) {   // B, BtW, D1 and D2 of a mode follow each other in the plan's array too
      const int n = 2 * nm + (d2 ? 2 : 1) * ng;
      for (int e = threadIdx.x; e < n; e += blockDim.x) ms[off + e] = mats[q.B + e];
      off += n;
    }
    A *= nq;
  }
}

// n / d for 0 <= n < 2^20 (inv = 1.0f / d): the half keeps the float product
// off the integers by more than its rounding
__device__ __forceinline__ int pdiv(int n, float inv) { return (int)(((float)n + 0.5f) * inv); }

// sum_j M[j] x[j s], j < n (M a matrix row)
__device__ __forceinline__ double row_dot(const double* __restrict__ M, const double* x, int s, int n) {
  double y0 = 0.0, y1 = 0.0;
  int j = 0;
  for (; j + 4 <= n; j += 4) {
    const double a0 = M[j], a1 = M[j + 1], a2 = M[j + 2], a3 = M[j + 3];
    const double b0 = x[j * s], b1 = x[(j + 1) * s], b2 = x[(j + 2) * s], b3 = x[(j + 3) * s];
    y0 = fma(a0, b0, y0); y1 = fma(a1, b1, y1);
    y0 = fma(a2, b2, y0); y1 = fma(a3, b3, y1);
  }
  for (; j < n; ++j) y0 = fma(M[j], x[j * s], y0);
  return y0 + y1;
}

// out (NO points along the mode) = M (NO x NI) in; A: product of the sizes
// before the mode (equal in both tensors), np: points of out
template <class F>
__device__ __forceinline__ void mode_out(const double* __restrict__ M, const double* in, int A, int NI, int NO,
                                         int np, int lg, F&& put) {
  const float invA = 1.0f / (float)A, invO = 1.0f / (float)NO;
  const int nv = 1 << lg;
  for (int e = threadIdx.x; e < np << lg; e += blockDim.x) {
    const int p = e >> lg, v = e & (nv - 1);
    const int q = pdiv(p, invA), b = pdiv(q, invO), i = q - b * NO;
    const int pa = p - q * A;
    put(e, p, row_dot(M + i * NI, in + v + ((pa + A * NI * b) << lg), A << lg, NI));
  }
}

// psi of the term into x (LDS); basis index first mode fastest
__device__ __forceinline__ void gather(const PArgs& a, const TermDev* Td, double* x) {
  const int lg = a.lg, nv = 1 << lg, v0 = blockIdx.y << lg;
  const int32_t* map = a.map + Td->boff;
  for (int e = threadIdx.x; e < Td->nb << lg; e += blockDim.x) {
    const int m = map[e >> lg], v = v0 + (e & (nv - 1));
    x[e] = m >= 0 && v < a.nvec ? a.psi[(int64_t)m * a.rs + (int64_t)v * a.vs] : 0.0;
  }
}

// basis -> grid, from x with y as the other buffer; put(e, p, value) for the
// grid values; returns the buffer (x or y) that put may store to
template <class F>
__device__ __forceinline__ double* to_grid(const PModes& m, const double* M, int D, int nb, int lg, double* x,
                                           double* y, F&& put) {
  int np = nb;
  for (int k = 0; k < D; ++k) {
    __syncthreads();
    np = np / m.nb[k] * m.nq[k];
    if (k + 1 < D) mode_out(M + m.B[k], x, m.A[k], m.nb[k], m.nq[k], np, lg, [&](int e, int, double s) { y[e] = s; });
    else mode_out(M + m.B[k], x, m.A[k], m.nb[k], m.nq[k], np, lg, [&](int e, int p, double s) { y[e] = s; put(e, p, s); });
    double* t = x; x = y; y = t;
  }
  return x;
}

// grid -> basis and the weighted scatter-add, from x with y as the other buffer
__device__ __forceinline__ void to_packed(const PArgs& a, const PModes& m, const double* M, const TermDev* Td, double* x,
                                          double* y) {
  const int D = Td->nact, lg = a.lg, nv = 1 << lg, v0 = blockIdx.y << lg;
  const int32_t* map = a.map + Td->boff;
  int np = Td->nq, A = 1;
  for (int k = 0; k < D; ++k) {
    __syncthreads();
    np = np / m.nq[k] * m.nb[k];
    if (k + 1 < D)
      mode_out(M + m.Bt[k], x, A, m.nq[k], m.nb[k], np, lg, [&](int e, int, double s) { y[e] = s; });
    else
      mode_out(M + m.Bt[k], x, A, m.nq[k], m.nb[k], np, lg, [&](int e, int p, double s) {
        const int r = map[p], v = v0 + (e & (nv - 1));
        if (r >= 0 && v < a.nvec) atomicAdd(&a.hpsi[(int64_t)r * a.rs + (int64_t)v * a.vs], Td->wgt * s);
      });
    A *= m.nb[k];
    double* t = x; x = y; y = t;
  }
}

// derivative of the grid tensor x along mode k at value e (point p)
__device__ __forceinline__ double deriv_at(const PModes& m, int k, const double* M, const double* x, int e, int p,
                                           int lg) {
  const int n = m.nq[k], A = m.A[k];
  const int q = pdiv(p, m.invA[k]), i = q - pdiv(q, m.invq[k]) * n;
  return row_dot(M + i * n, x + e - ((A * i) << lg), A << lg, n);
}

}  // namespace

// Type 10 (sub_TabOpPsi_OF_ONEDP_FOR_SGtype4 case 10, SRC/sub_Operator/
// sub_OpPsi_SG4.f90:1546-1649):  u = sqRJ psi;
//   w_i = Jac sum_j G(j,i) d1_j u;  H psi = -1/2 sum_i d1_i w_i / (Jac sqRJ) + V psi
// A point's thread forms all d1_j u and then all w_i, and later all d1_i w_i:
// two passes for the kinetic part.  LDS: D + 3 buffers (two for the transforms,
// one of which ends as psi on the grid; u; the w_i).
namespace {
template <bool STAGE>
__device__ __forceinline__ void term_t10(const PArgs& a, const KMats10& km) {
  extern __shared__ double lds[];
  __shared__ PModes m;
  const TermDev* Td = &a.terms[a.order[blockIdx.x]];
  const int lg = a.lg, D = Td->nact, NE = Td->nq << lg;
  const int64_t q0 = Td->qoff;
  double* b0 = lds;
  double* b1 = lds + NE;
  double* u = lds + 2 * NE;
  double* W = lds + 3 * NE;                 // w_i at W + i NE
  double* ms = W + D * NE;
  const double* M = STAGE ? ms : km.mats;
  load_modes<STAGE>(m, a, km.mats, Td, ms, false);
  gather(a, Td, b0);
  double* pg = to_grid(m, M, D, Td->nb, lg, b0, b1, [&](int e, int p, double s) { u[e] = km.sqRJ[q0 + p] * s; });
  __syncthreads();
  for (int e = threadIdx.x; e < NE; e += blockDim.x) {
    const int p = e >> lg;
    const double* G = km.G + (int64_t)D * D * (q0 + p);
    const double jac = km.Jac[q0 + p];
    // w_i is accumulated over j in LDS: this thread's elements only
    for (int j = 0; j < D; ++j) {
      const double du = deriv_at(m, j, M + m.D1[j], u, e, p, lg);
      for (int i = 0; i < D; ++i) {
        const double g = G[j + D * i];
        double* w = W + (int64_t)i * NE + e;
        const double s = j == 0 ? g * du : fma(g, du, *w);
        *w = j + 1 == D ? jac * s : s;
      }
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < NE; e += blockDim.x) {
    const int p = e >> lg;
    double s = 0.0;
    for (int i = 0; i < D; ++i) s += deriv_at(m, i, M + m.D1[i], W + (int64_t)i * NE, e, p, lg);
    u[e] = -0.5 * s / (km.Jac[q0 + p] * km.sqRJ[q0 + p]) + km.V[q0 + p] * pg[e];
  }
  to_packed(a, m, M, Td, u, pg);
}
}  // namespace
__global__ __launch_bounds__(512) void k_hpsi_t10_f64(PArgs a, KMats10 km) {
  if (a.stage) term_t10<true>(a, km);
  else term_t10<false>(a, km);
}

// General type-1 operator (case 1, SRC/sub_Operator/sub_OpPsi_SG4.f90
// :1488-1544):  H psi = sum_e F_e(q) D_e psi, D_e the identity, d1 along i, d2
// along i, or d1 along j then along i (the 1-D matrices of
// DerivOp_TO_RDP_OF_SmolaykRep).  A point's thread adds all terms but the mixed
// ones in one pass; a mixed derivative takes two passes (d1 along j of the whole
// tensor, then d1 along i of it at the point).  LDS: three buffers.
namespace {
template <bool STAGE>
__device__ __forceinline__ void term_t1g(const PArgs& a, const KMats1G& km) {
  extern __shared__ double lds[];
  __shared__ PModes m;
  const TermDev* Td = &a.terms[a.order[blockIdx.x]];
  const int lg = a.lg, D = Td->nact, NE = Td->nq << lg;
  double* b0 = lds;
  double* b1 = lds + NE;
  double* Y = lds + 2 * NE;
  double* ms = Y + NE;
  const double* M = STAGE ? ms : km.mats;
  load_modes<STAGE>(m, a, km.mats, Td, ms, true);
  gather(a, Td, b0);
  double* X = to_grid(m, M, D, Td->nb, lg, b0, b1, [](int, int, double) {});
  double* W = X == b0 ? b1 : b0;
  const double* F = km.F + Td->qoff;
  __syncthreads();
  for (int e = threadIdx.x; e < NE; e += blockDim.x) {
    const int p = e >> lg;
    double y = 0.0;
    for (int d = 0; d < km.nder; ++d) {
      int i = km.der[2 * d], j = km.der[2 * d + 1];
      if (i < 0 && j >= 0) { i = j; j = -1; }
      if (i >= 0 && j >= 0 && i != j) continue;      // mixed: below
      const double s = i < 0 ? X[e] : deriv_at(m, i, M + (j < 0 ? m.D1[i] : m.D2[i]), X, e, p, lg);
      y = fma(F[(int64_t)d * km.sum_nq + p], s, y);
    }
    Y[e] = y;
  }
  for (int d = 0; d < km.nder; ++d) {
    const int i = km.der[2 * d], j = km.der[2 * d + 1];
    if (i < 0 || j < 0 || i == j) continue;
    for (int e = threadIdx.x; e < NE; e += blockDim.x) W[e] = deriv_at(m, j, M + m.D1[j], X, e, e >> lg, lg);
    __syncthreads();
    for (int e = threadIdx.x; e < NE; e += blockDim.x)
      Y[e] = fma(F[(int64_t)d * km.sum_nq + (e >> lg)], deriv_at(m, i, M + m.D1[i], W, e, e >> lg, lg), Y[e]);
    __syncthreads();                                 // W is written again
  }
  to_packed(a, m, M, Td, Y, X);
}
}  // namespace
__global__ __launch_bounds__(512) void k_hpsi_t1g_f64(PArgs a, KMats1G km) {
  if (a.stage) term_t1g<true>(a, km);
  else term_t1g<false>(a, km);
}

}  // namespace sg4
