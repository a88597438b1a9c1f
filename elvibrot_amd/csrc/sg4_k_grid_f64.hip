// Grid paths, FP64: the type-1 kernel with the kinetic derivatives on the
// grid and the grid-value gradient kernel of the per-mode passes.
#include "sg4_grid.h"

namespace sg4 {

// The grid is either one workgroup per item or a persistent grid that walks
// the (cost-sorted) item list with stride gridDim.x.
__global__ __launch_bounds__(NT) void k_hpsi_t1_f64(KArgs a, KMats<double> km) {
  extern __shared__ double lds[];
  for (int w = blockIdx.x; w < a.nitems; w += gridDim.x) {
    if (w != (int)blockIdx.x) __syncthreads();   // LDS reuse between items
    const Item it = a.items[w];
    if (it.term < 0) continue;
    if (it.big) term_t1<double, true>(a, km, it, lds);
    else if (a.terms[it.term].ngrp > 0) term_t1_grouped<double>(a, km, it, lds);
    else term_t1<double, false>(a, km, it, lds);
  }
}

// ---------------------------------------------------------------------------
// Grid-value gradient of <phi|H|psi>: both vectors transformed basis -> grid
// (the first half of the H.psi pipeline), then the weighted product.
// LDS: four buffers of nq_t x nv.
// ---------------------------------------------------------------------------

__device__ void bg_transform(const KArgs& a, const double* mats, const TermDev* Td, const Item& it,
                             const double* src, double* b0, double* b1, double** result) {
  const int lg = it.lgnv, nv = 1 << lg;
  PassCtx<double> c;
  c.map = a.map + Td->boff; c.psi = src; c.hpsi = nullptr; c.nvec = a.nvec; c.v0 = it.v0;
  c.wgt = 1.0; c.V = nullptr; c.vshift = 0.0; c.lgnv = lg; c.coef = 1.0;
  int A = 1, Bafter = Td->nb;
  double* cur = nullptr;
  double* nxt = b0;
  for (int p = 0; p < Td->nact; ++p) {
    const MatDev* md = &a.md[Td->mat[p]];
    const int nq = md->nq, nb = md->nb;
    Bafter /= nb;
    c.MR = mats + md->B;
    c.in = cur; c.out = nxt;
    c.A = A; c.AV = A * nv; c.invAV = 1.0f / (float)c.AV;
    c.nfib = A * nv * Bafter;
    if (p == 0) dispatch_pass<double, true, IN_GATHER, OUT_STORE>(c, nb, nq);
    else dispatch_pass<double, true, IN_LDS, OUT_STORE>(c, nb, nq);
    __syncthreads();
    A *= nq;
    cur = nxt;
    nxt = (nxt == b0) ? b1 : b0;
  }
  *result = cur;
}

__global__ __launch_bounds__(NT) void k_grad_v(KArgs a, KGrad kg) {
  extern __shared__ double lds[];
  const Item it = a.items[blockIdx.x];
  const TermDev* Td = &a.terms[it.term];
  const int lg = it.lgnv, nv = 1 << lg;
  const size_t SZ = (size_t)Td->nq * nv;
  double* gphi = nullptr;
  double* gpsi = nullptr;
  if (Td->nact == 0) {   // one point, no transform
    for (int v = threadIdx.x; v < nv; v += blockDim.x) {
      const int m = a.map[Td->boff];
      const int64_t r = (int64_t)m * a.nvec + it.v0 + v;
      kg.grad[Td->qoff * a.nvec + it.v0 + v] = (m >= 0) ? Td->wgt * kg.phi[r] * a.psi[r] : 0.0;
    }
    return;
  }
  bg_transform(a, kg.mats, Td, it, kg.phi, lds, lds + SZ, &gphi);
  bg_transform(a, kg.mats, Td, it, a.psi, lds + 2 * SZ, lds + 3 * SZ, &gpsi);
  for (size_t e = threadIdx.x; e < SZ; e += blockDim.x) {
    int pt = (int)(e >> lg);
    double w = Td->wgt;
    for (int p = 0; p < Td->nact; ++p) {
      const MatDev* md = &a.md[Td->mat[p]];
      const int i = pt % md->nq;
      pt /= md->nq;
      w *= kg.qw[kg.qw_off[Td->mat[p]] + i];
    }
    kg.grad[(Td->qoff + (int64_t)(e >> lg)) * a.nvec + it.v0 + (e & (nv - 1))] = w * gphi[e] * gpsi[e];
  }
}

}  // namespace sg4
