// Grid-value gradient of <phi|H|psi> for plans whose terms are all in mode
// groups: both vectors basis -> grid through register-blocked passes, then one
// pass over the item's values for the weighted products.
//
// An item is a term and up to nv vectors (any number: the output rows of a
// point are written whole when the item holds the block).  LDS: the tensor of
// phi and, unless phi and psi are the same block, that of psi, element
// (point p, vector v) at [p nv + v], and the quadrature weights of the last
// group and of the modes before it.  phi = psi (Hellmann-Feynman) is
// transformed once.  (With the product fused into the last group's pass the
// compiler kept whole matrices and offsets in scalar registers: 12 000 spills.)
//
// What bounds it: the latency of the gathers and passes of a term, as in the
// H.psi term kernels.  8D L=6 x5, phi = psi: 29 us against 407 us for the
// per-mode passes (k_grad_v: both blocks transformed, four tensors in LDS,
// chunks of 4 + 1 vectors, integer divisions by every mode's size at each
// point).
#include "sg4_device.h"

namespace sg4 {

namespace {

struct GCx {
  const double* M[3];
  double* X;             // the tensors
  const double* src[2];  // phi, psi
  const int32_t* map;
  int ntens, NE;         // tensors, values per tensor
  int AV, nfib, nvec, v0, gather;
  float invAV;
};

template <int N0, int N1, int N2>
__device__ __forceinline__ void grad_pass(const GCx& c) {
  constexpr int P = N0 * N1 * N2;
  for (int ff = threadIdx.x; ff < c.nfib * c.ntens; ff += blockDim.x) {
    const int t = ff >= c.nfib;
    const int f = t ? ff - c.nfib : ff;
    const int b = fdiv(f, c.AV, c.invAV);
    const int av = f - b * c.AV;
    double* X = c.X + (size_t)t * c.NE;
    const int base = av + c.AV * P * b;
    double x[P];
    if (c.gather) {   // group 0: av is the vector
      const double* s = (t ? c.src[1] : c.src[0]) + c.v0 + av;
#pragma unroll
      for (int J = 0; J < P; ++J) {
        const int m = c.map[P * b + J];
        x[J] = m >= 0 ? s[(int64_t)m * c.nvec] : 0.0;
      }
    } else {
#pragma unroll
      for (int J = 0; J < P; ++J) x[J] = X[base + c.AV * J];
    }
    cptr<double> M0 = (cptr<double>)uniform_ptr(c.M[0]);
    cptr<double> M1 = (cptr<double>)uniform_ptr(c.M[1]);
    cptr<double> M2 = (cptr<double>)uniform_ptr(c.M[2]);
    asm volatile("" : "+s"(M0), "+s"(M1), "+s"(M2));
    slab_mode<double, N0, 1, P>(x, M0);
    if constexpr (N1 > 1) slab_mode<double, N1, N0, P>(x, M1);
    if constexpr (N2 > 1) slab_mode<double, N2, N0 * N1, P>(x, M2);
#pragma unroll
    for (int J = 0; J < P; ++J) X[base + c.AV * J] = x[J];
  }
}

__device__ __forceinline__ void dispatch_grad(const GCx& c, int shape) {
  switch (shape) {
#define SG4_GRCASE(id, a, b, d) case id: grad_pass<a, b, d>(c); return;
    SG4_SHAPES(SG4_GRCASE)
#undef SG4_GRCASE
    default: return;
  }
}

// w times the quadrature weights of modes p0..p1-1 at their combined index e
__device__ __forceinline__ double grad_weight(const KArgs& a, const KGrad& kg, const TermDev* Td, int p0, int p1,
                                              int e, double w) {
  for (int p = p0; p < p1; ++p) {
    const int n = a.md[Td->mat[p]].nq;
    const int i = e % n;
    e /= n;
    w *= kg.qw[kg.qw_off[Td->mat[p]] + i];
  }
  return w;
}

__device__ __forceinline__ void grad_term(const KArgs& a, const KGrad& kg, const Item& it, double* lds) {
  const TermDev* Td = &a.terms[it.term];
  const int nv = it.slot;   // vectors of the item
  const bool same = kg.phi == a.psi;
  const double w = Td->wgt;
  if (Td->nact == 0) {      // one point, no transform
    const int m = a.map[Td->boff];
    for (int v = threadIdx.x; v < nv; v += blockDim.x) {
      const int64_t r = (int64_t)m * a.nvec + it.v0 + v;
      kg.grad[Td->qoff * a.nvec + it.v0 + v] = (m >= 0) ? w * kg.phi[r] * a.psi[r] : 0.0;
    }
    return;
  }
  const int N = Td->nq, G = Td->ngrp;
  GCx c;
  c.X = lds;
  c.src[0] = kg.phi;
  c.src[1] = a.psi;
  c.map = a.map + Td->boff;
  c.NE = N * nv;
  c.ntens = same ? 1 : 2;
  c.nvec = a.nvec;
  c.v0 = it.v0;
  double* Wp = lds + (size_t)c.ntens * c.NE;   // A weights of the modes before the last group,
  double* Wl;                                  // then the last group's
  int A = 1, P = 1;   // points of the modes before the current group, and of the group
  for (int g = 0; g < G; ++g) {
    A *= P;
    const int p0 = Td->gfirst[g], p1 = (g + 1 < G) ? Td->gfirst[g + 1] : Td->nact;
    P = 1;
    for (int q = 0; q < 3; ++q) {
      if (p0 + q < p1) {
        const MatDev* md = &a.md[Td->mat[p0 + q]];
        P *= md->nq;
        c.M[q] = kg.mats + md->B;
      } else {
        c.M[q] = c.M[0];
      }
    }
    c.AV = A * nv;
    c.invAV = 1.0f / (float)c.AV;
    c.nfib = c.NE / P;
    c.gather = g == 0;
    dispatch_grad(c, Td->gshape[g]);
    if (g + 1 == G) {
      Wl = Wp + A;
      for (int e = threadIdx.x; e < A + P; e += blockDim.x)
        Wp[e] = e < A ? grad_weight(a, kg, Td, 0, p0, e, w) : grad_weight(a, kg, Td, p0, p1, e - A, 1.0);
    }
    __syncthreads();
  }
  // consecutive threads: the vectors of a point, then the next point
  const double* x = lds;
  const double* y = lds + (same ? 0 : c.NE);
  double* out = kg.grad + Td->qoff * a.nvec + it.v0;
  const float invnv = 1.0f / (float)nv, invA = 1.0f / (float)A;
  for (int e = threadIdx.x; e < c.NE; e += blockDim.x) {
    const int p = fdiv(e, nv, invnv), j = fdiv(p, A, invA);
    out[(int64_t)p * a.nvec + (e - p * nv)] = Wp[p - j * A] * Wl[j] * (x[e] * y[e]);
  }
}

}  // namespace

__global__ __launch_bounds__(128) void k_grad_groups(KArgs a, KGrad kg) {
  extern __shared__ double lds[];
  grad_term(a, kg, a.items[blockIdx.x], lds);
}

}  // namespace sg4
