// Potentials that are sums of one- and two-mode functions,
//   V(q) = V0 + sum_a f_a(q_a) + sum_{a<b} f_ab(q_a, q_b)
// (Henon-Heiles, vibronic-coupling models, quadratic and cubic pair force
// fields): the whole type-1 H as one sparse matrix over the packed rows.
//
// With B^T W B = I in every mode (checked for the split path) a term's matrix
// of f_ab is M_ab(l_a, l_b) = (BtW_a x BtW_b) f_ab (B_a x B_b) in modes a, b and
// the identity in the others, so the Smolyak sum over the levels of the other
// modes telescopes as it does for the kinetic part: with Lambda the sum of the
// smallest levels holding the indices of the other modes, the weights of fixed
// (l_a, l_b) sum to the coefficient of z^u, u = L - Lambda - l_a - l_b, in
// (1 - z)^-(D-2) (1 - z)^(D-1) = 1 - z.  Hence with m = L - Lambda
//   <r|V|r'> = sum_{l_a + l_b = m} M_ab - sum_{l_a + l_b = m - 1} M_ab
// (levels that hold both rows' indices), the two-mode combination technique,
// and for f_a (and c_a d_a^2) the one-mode matrix at level m = L - Lambda_a.
// This is the operator the term-by-term sum gives, without its cancellation.
//
// f_a and f_ab are read off the grid V on cuts through the middle point of the
// other modes (odd rules), then the sum is compared with V on EVERY grid
// point; V that differs beyond rounding keeps the term kernels.  Matrix
// elements below the rounding error of their own quadrature sum are zero
// (parity, band structure of polynomials) and are not stored.
//
// What bounds it: the gathers of psi rows, one 128-byte line per stored entry
// and 16 vectors.  10D L=8 Henon-Heiles (32.2 M entries, 0.39 GB): 0.44 ms at 16
// vectors (2.64 GB read, 0.19 written: 5.8 TB/s with the result to columns), 0.14
// ms at one (matrix 2.8 TB/s); the term kernels and the kinetic rows take 4.7 and
// 0.8 ms.  sg4_apply of 16 column-major vectors: 0.54 ms against 4.8.  Rows in
// order; measured slower at 16 / 1 vectors with the kernel of one column per lane
// (0.75 / 0.14 ms): 8 loads in flight 0.77 / 0.16 ms, a contiguous chunk of rows
// per XCD 0.80 / 0.15, non-temporal matrix loads 0.94 / 0.18.
#include "sg4_nmode.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <string>

namespace sg4 {

#define NM_TRY(expr)                                                              \
  do {                                                                            \
    hipError_t _e = (expr);                                                       \
    if (_e != hipSuccess) {                                                       \
      set_error(std::string("HIP error: ") + hipGetErrorString(_e) + " at " #expr); \
      return SG4_ERR_HIP;                                                         \
    }                                                                             \
  } while (0)

namespace {

constexpr int NI = SG4_MAX_N;         // 1-D indices per mode
constexpr int RL = 4;                // lanes per row and
constexpr int RT = 256 / RL;          // rows per workgroup of the row kernels
constexpr double EPS = 2.220446049250313e-16;
// A grid value may differ from the sum of its parts by the rounding of the
// parts (each the difference of up to four grid values): 64 eps of the sum of
// their magnitudes.  A matrix element below 16 eps of the absolute sum of its
// quadrature terms is rounding.
constexpr double TOL_V = 64 * EPS, TOL_M = 16 * EPS;
// Stored entries per grid point up to which the matrix is taken: an entry
// cost ~1.5 ps per vector at 10D L=8 (gather of one psi value) with one column per
// lane, ~0.85 with pairs of columns, a grid point 9.2 to 9.5 ps in the FP64 term
// kernel: matrices of four to some eight entries per point would still pay, which
// the memory and the building of the larger ones speak against.
constexpr double NNZ_PER_POINT = 4.0;
constexpr int64_t NNZ_SMALL = 1 << 18;        // always taken: the apply is one short launch
// A column-major block is read in place while nnz W^2 <= 2^24 (W columns, a
// gather touches W lines instead of one), else staged in the rows layout (one
// more launch).  In place / staged, us: 6D L=6 (160 k entries) x8 6.8 / 7.5, x16
// 9.3 / 9.4, 8D L=6 (760 k) x4 11.5 / 10.8, x8 17.5 / 15.1, 9D L=7 (5.0 M) x2
// 31.0 / 28.3.
constexpr int64_t COLS_DIRECT = (int64_t)1 << 24;
constexpr int64_t MAX_E = (int64_t)1 << 27;   // entries of the two-mode tables

// Device view of an instance.
struct NmDev {
  int D, L, LB, L1;            // L1 = Lmax + 1 (stride of the md tables)
  int64_t term0, nterms, row0, nrows;
  const int32_t* levels;       // D per term
  const MatDev* md;            // [k * L1 + l]
  const int32_t* n;            // [k * (L+1) + l] points
  const uint8_t* lam;          // [k * NI + i] smallest level holding index i
  const int32_t* pre;          // [(k * (LB+1) + b) * (NI+1) + i] rank prefix
  const int32_t* f1off;        // [k * (L+1) + l] offset of the mode's cut, -1: none
  const int32_t* f2off;        // [(p * (L+1) + la) * (L+1) + lb], -1: none
  const int32_t* s2n;          // [p * (L+1) + m] pair indices of level <= m
  const int32_t* s2off;        // [p] offset in s2 / pos
  const uint16_t* s2;          // (ja | jb << 8), by level
  const int32_t* posoff;       // [p]
  const int16_t* pos;          // [ia * nbL + ib] position in s2
  const uint8_t* pa;           // [p] modes of the pair
  const uint8_t* pb;
  const double* T;             // kinetic matrices of the instance
  const int32_t* toff;         // [k * (L+1) + l]
  const double* ck;            // D
  const int32_t* g1off;        // [k * (L+1) + l] offset in g1
  int64_t c1base;              // the instance's cuts: c1[c1base] = V0
  int npair, pair0;            // pair0: first global pair (flags, eoff)
};

// A cut of V: along one mode (nb = 1) or two.
struct Cut {
  int64_t off;                 // grid value at the middle point of the other modes, indices 0
  int32_t sa, sb, na, nb;
  int64_t out;                 // where the cut goes in c1 / f2
  int64_t fa, fb, v0;          // two modes: the one-mode cuts and V0 in c1
  int32_t pair;                // global pair, or -1
};

// work item of the two-mode matrices
struct EWork { int32_t inst, pair, m; int32_t pad; int64_t off; };

__device__ __forceinline__ int find_inst(const int64_t* first, int ninst, int64_t x) {
  int lo = 0, hi = ninst;
  while (hi - lo > 1) {
    const int mid = (lo + hi) / 2;
    if (first[mid] <= x) lo = mid; else hi = mid;
  }
  return lo;
}

// the map's entries are the lexicographic ranks of their mode indices
// (-1 beyond the basis level), the last mode's index fastest
__global__ __launch_bounds__(256) void k_nm_check_map(const NmDev* insts, const int64_t* term0,
                                                      int ninst, int64_t nterms, const TermDev* terms,
                                                      const int32_t* map, int* bad) {
  for (int64_t t = blockIdx.x; t < nterms; t += gridDim.x) {
    const NmDev& I = insts[find_inst(term0, ninst, t)];
    const int32_t* lev = I.levels + (t - I.term0) * I.D;
    const TermDev& T = terms[t];
    for (int e = threadIdx.x; e < T.nb; e += blockDim.x) {
      int rest = e, b = I.LB;
      int64_t r = 0;
      for (int k = 0; k < I.D && r >= 0; ++k) {
        const int n = I.n[k * (I.L + 1) + lev[k]];
        const int i = rest % n;
        rest /= n;
        const int li = I.lam[k * NI + i];
        if (li > b) { r = -1; break; }
        r += I.pre[(k * (I.LB + 1) + b) * (NI + 1) + i];
        b -= li;
      }
      if (map[T.boff + e] != (r < 0 ? -1 : (int32_t)(r + I.row0))) *bad = 1;
    }
  }
}

__global__ __launch_bounds__(64) void k_nm_cut1(const Cut* cuts, const double* V, double* c1) {
  const Cut c = cuts[blockIdx.x];
  for (int i = threadIdx.x; i < c.na; i += 64) c1[c.out + i] = V[c.off + (int64_t)i * c.sa];
}

// f_ab on its cut; a pair whose cuts are all rounding stays flagged zero
__global__ __launch_bounds__(64) void k_nm_cut2(const Cut* cuts, const double* V, const double* c1,
                                                double* f2, int* flag) {
  const Cut c = cuts[blockIdx.x];
  const double v0 = c1[c.v0];
  bool nz = false;
  for (int e = threadIdx.x; e < c.na * c.nb; e += 64) {
    const int ia = e % c.na, ib = e / c.na;
    const double v = V[c.off + (int64_t)ia * c.sa + (int64_t)ib * c.sb];
    const double va = c1[c.fa + ia], vb = c1[c.fb + ib];
    const double f = (v - va) - (vb - v0);
    f2[c.out + e] = f;
    nz = nz || !(fabs(f) <= TOL_V * (fabs(v) + fabs(va) + fabs(vb) + fabs(v0)));
  }
  if (nz) flag[c.pair] = 1;
}

// V against the sum of its parts on every grid point of every term
__global__ __launch_bounds__(256) void k_nm_verify(const NmDev* insts, const int64_t* term0, int ninst,
                                                   int64_t nterms, const TermDev* terms, const double* V,
                                                   const double* c1, const double* f2, const int* flag,
                                                   int* bad) {
  __shared__ int an[MAXACT], af[MAXACT], act[MAXACT], np, stop, px[120], py[120], pf[120];
  __shared__ uint8_t dig[MAXACT][256];
  const int tid = threadIdx.x;
  for (int64_t t = blockIdx.x; t < nterms; t += gridDim.x) {
    __syncthreads();                   // the previous term's tables are no longer read
    if (tid == 0) { stop = *(volatile int*)bad; np = 0; }
    __syncthreads();
    if (stop) return;                  // the same for the whole workgroup
    const NmDev& I = insts[find_inst(term0, ninst, t)];
    const int32_t* lev = I.levels + (t - I.term0) * I.D;
    const int L1 = I.L + 1;
    int na = 0;
    for (int k = 0; k < I.D; ++k)
      if (lev[k] > 0 && I.n[k * L1 + lev[k]] > 1) {
        if (tid == 0 && na < MAXACT) {
          act[na] = k;
          an[na] = I.n[k * L1 + lev[k]];
          af[na] = I.f1off[k * L1 + lev[k]];
        }
        ++na;
      }
    __syncthreads();
    if (na > MAXACT) { if (tid == 0) *bad = 1; return; }
    for (int e = tid; e < na * na; e += 256) {
      const int x = e / na, y = e % na;
      if (x >= y) continue;
      const int a = act[x], b = act[y];
      const int p = a * (2 * I.D - a - 1) / 2 + (b - a - 1);
      if (!flag[I.pair0 + p]) continue;
      const int s = atomicAdd(&np, 1);
      px[s] = x; py[s] = y;
      pf[s] = I.f2off[(p * L1 + lev[a]) * L1 + lev[b]];
    }
    __syncthreads();
    const TermDev& T = terms[t];
    const double v0 = c1[I.c1base];
    const int npairs = np;
    for (int e = tid; e < T.nq; e += 256) {
      int rest = e;
      double s = v0, mag = fabs(v0);
      bool miss = false;
      for (int j = 0; j < na; ++j) {
        const int i = rest % an[j];
        rest /= an[j];
        dig[j][tid] = (uint8_t)i;
        if (af[j] < 0) { miss = true; continue; }
        const double f = c1[af[j] + i] - v0;
        s += f;
        mag += fabs(f);
      }
      for (int q = 0; q < npairs; ++q) {
        if (pf[q] < 0) { miss = true; continue; }
        const double f = f2[pf[q] + dig[px[q]][tid] + an[px[q]] * dig[py[q]][tid]];
        s += f;
        mag += fabs(f);
      }
      const double v = V[T.qoff + e];
      if (miss || !(fabs(v - s) <= TOL_V * (mag + fabs(v)))) *bad = 1;
    }
  }
}

// one-mode matrices at every level: kinetic part c_a T_a, grid part BtW f_a B
// (KIN | GRID)
enum { G1_KIN = 1, G1_GRID = 2 };
__global__ __launch_bounds__(256) void k_nm_g1(const NmDev* insts, const int32_t* work, const double* mats,
                                               const double* c1, double* g1, int what) {
  const NmDev& I = insts[work[3 * blockIdx.x]];
  const int k = work[3 * blockIdx.x + 1], l = work[3 * blockIdx.x + 2];
  const int n = I.n[k * (I.L + 1) + l], f1 = I.f1off[k * (I.L + 1) + l];
  const MatDev& md = I.md[k * I.L1 + l];
  const double* B = mats + md.B;
  const double* Bt = mats + md.BtW;
  const double* T = I.T + I.toff[k * (I.L + 1) + l];
  double* g = g1 + I.g1off[k * (I.L + 1) + l];
  const double v0 = c1[I.c1base], c = (what & G1_KIN) ? I.ck[k] : 0.0;
  for (int e = threadIdx.x; e < n * n; e += 256) {
    const int i = e / n, j = e % n;
    double s = 0.0, m = 0.0;
    if (f1 >= 0 && n > 1 && (what & G1_GRID))
      for (int q = 0; q < n; ++q) {
        const double w = Bt[i * n + q] * B[q * n + j], v = c1[f1 + q];
        s = fma(w, v - v0, s);
        m = fma(fabs(w), fabs(v) + fabs(v0), m);
      }
    if (!(fabs(s) > TOL_M * m)) s = 0.0;
    g[e] = fma(c, T[e], s);
  }
}

// two-mode matrices E(m) of a pair over the pair indices of level <= m; eight
// lanes per element share the level pairs (12 instances: 248 us with one)
__global__ __launch_bounds__(256) void k_nm_e2(const NmDev* insts, const EWork* work, const double* mats,
                                               const double* c1, const double* f2, double* E) {
  const EWork w = work[blockIdx.x];
  const NmDev& I = insts[w.inst];
  const int p = w.pair, m = w.m, L1 = I.L + 1;
  const int a = I.pa[p], b = I.pb[p], S = I.s2n[p * L1 + m];
  const uint16_t* lst = I.s2 + I.s2off[p];
  const double v0 = c1[I.c1base];
  const int sub = threadIdx.x & 7;
  for (int e = blockIdx.y * 32 + (threadIdx.x >> 3); e < S * S; e += gridDim.y * 32) {
    const int r = lst[e / S], c = lst[e % S];
    const int ia = r & 255, ib = r >> 8, ja = c & 255, jb = c >> 8;
    const int la0 = max(1, max(I.lam[a * NI + ia], I.lam[a * NI + ja]));
    const int lb0 = max(1, max(I.lam[b * NI + ib], I.lam[b * NI + jb]));
    // level pairs l_a + l_b = m (n0 of them), then m - 1 with the minus sign
    const int n0 = max(0, m - lb0 - la0 + 1), n1 = max(0, n0 - 1);
    double sum = 0.0, mag = 0.0;
    for (int x = sub; x < n0 + n1; x += 8) {
      const int u = x >= n0, la = la0 + (u ? x - n0 : x), lb = m - u - la;
      const int off = I.f2off[(p * L1 + la) * L1 + lb];
      const int fa = I.f1off[a * L1 + la], fb = I.f1off[b * L1 + lb];
      if (off < 0 || fa < 0 || fb < 0) continue;   // levels that no row needs
      const int na = I.n[a * L1 + la], nb = I.n[b * L1 + lb];
      const MatDev& A = I.md[a * I.L1 + la];
      const MatDev& Q = I.md[b * I.L1 + lb];
      double t = 0.0;
      for (int q = 0; q < nb; ++q) {
        const double wb = mats[Q.BtW + ib * nb + q] * mats[Q.B + q * nb + jb];
        double s = 0.0, g = 0.0;
        for (int o = 0; o < na; ++o) {
          const double wa = mats[A.BtW + ia * na + o] * mats[A.B + o * na + ja];
          const double f = f2[off + o + na * q];
          s = fma(wa, f, s);
          g = fma(fabs(wa), fabs(f) + fabs(c1[fa + o]) + fabs(c1[fb + q]) + fabs(v0), g);
        }
        t = fma(wb, s, t);
        mag = fma(fabs(wb), g, mag);
      }
      sum += u ? -t : t;
    }
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) {
      sum += __shfl_xor(sum, o, 64);
      mag += __shfl_xor(mag, o, 64);
    }
    if (sub == 0) E[w.off + e] = fabs(sum) > TOL_M * mag ? sum : 0.0;
  }
}

// What the row kernels read of one grid function.
struct NmSet {
  const double* c1;
  const double* g1;
  const double* E;
  const int64_t* eoff;        // [global pair * eld + m]; -1: zero pair
};
// nonzero pairs (of V or mu) of every instance, and by mode
struct NmPairs {
  const int32_t* nz;          // instance's pairs at nzoff[inst]
  const int32_t* nzoff;
  const int32_t* adj;         // pairs holding mode k at adjoff[inst * 33 + k]
  const int32_t* adjoff;
  // row ri of a pair's matrices at level m: the ecnt[croff + ri] columns at
  // elist[loff + ri S ..] where both indices change and V or mu is nonzero
  const int64_t* loff;        // [global pair * eld + m]
  const int64_t* croff;
  uint16_t* elist;
  int32_t* ecnt;
  int eld;
};

// the column lists of NmPairs, one thread per row of a pair's matrix
__global__ __launch_bounds__(64) void k_nm_elist(const NmDev* __restrict__ insts, const EWork* work, NmSet sv,
                                                 NmSet sm, NmPairs pr) {
  const EWork w = work[blockIdx.x];
  const NmDev& I = insts[w.inst];
  const int S = I.s2n[w.pair * (I.L + 1) + w.m];
  const uint16_t* lst = I.s2 + I.s2off[w.pair];
  const int64_t g = (int64_t)(I.pair0 + w.pair) * pr.eld + w.m;
  const int64_t ov = sv.eoff[g], om = sm.eoff ? sm.eoff[g] : -1;
  for (int r = blockIdx.y * 64 + threadIdx.x; r < S; r += gridDim.y * 64) {
    uint16_t* out = pr.elist + pr.loff[g] + (int64_t)r * S;
    int n = 0;
    for (int c = 0; c < S; ++c) {
      if ((lst[c] & 255) == (lst[r] & 255) || lst[c] >> 8 == lst[r] >> 8) continue;
      const bool nz = (ov >= 0 && sv.E[ov + (int64_t)r * S + c] != 0.0) ||
                      (om >= 0 && sm.E[om + (int64_t)r * S + c] != 0.0);
      if (nz) out[n++] = (uint16_t)c;
    }
    pr.ecnt[pr.croff[g] + r] = n;
  }
}

// Entries of a packed row: counted (FILL = false) or written.  RL lanes per
// row take its tasks (one mode changed: D of them; a pair changed: one per
// nonzero pair) in rounds, a task's entries going after those of the tasks
// before it; the row's mode indices, levels and rank prefixes sit in LDS.  The
// chains of dependent table reads bound it; the propagation of 12 instances
// (which builds once) takes 4.01 / 3.88 / 3.89 / 3.94 / 4.27 ms with 1 / 2 / 4 / 8 /
// 16 lanes, setting a 6D L=6 operator 1.60 / 1.48 / 1.41 / 1.34 / 1.38 ms.  10D L=8:
// the two passes take 0.7 and 1.7 ms.  A workgroup's rows belong to one instance (its first workgroup: blk0), whose
// tables are then addressed by scalars.
template <bool FILL, bool MU>
__global__ __launch_bounds__(256) void k_nm_rows(const NmDev* __restrict__ insts, const int64_t* __restrict__ blk0,
                                                 int ninst, NmSet sv, NmSet sm, NmPairs pr, int Dmax,
                                                 int32_t* cnt, const int64_t* ptr, int32_t* col, double* val,
                                                 double* valm) {
  extern __shared__ char sh[];
  int32_t* pre = (int32_t*)sh;                     // [k][row] rank contribution before mode k
  uint8_t* dg = (uint8_t*)(pre + Dmax * RT);       // mode indices
  uint8_t* lm = dg + Dmax * RT;                    // their levels
  uint8_t* bud = lm + Dmax * RT;                   // level budget left before mode k
  __shared__ int tots[RT];
  const int sub = threadIdx.x % RL, tid = threadIdx.x / RL;
  const int ii = __builtin_amdgcn_readfirstlane(find_inst(blk0, ninst, blockIdx.x));
  const NmDev& I = insts[ii];
  const int64_t lrow = ((int64_t)blockIdx.x - blk0[ii]) * RT + tid, row = I.row0 + lrow;
  const bool on = lrow < I.nrows;
  const int D = I.D, L = I.L, LB = I.LB, L1 = L + 1;
  if (on && sub == 0) {
    int32_t left = (int32_t)lrow, done = 0;
    int b = LB, tot = 0;
    for (int k = 0; k < D; ++k) {
      const int32_t* p = I.pre + (k * (LB + 1) + b) * (NI + 1);
      int i = 0;
      while (i + 1 < NI && I.lam[k * NI + i + 1] <= b && p[i + 1] <= left) ++i;
      const int li = I.lam[k * NI + i];
      pre[k * RT + tid] = done;
      dg[k * RT + tid] = (uint8_t)i;
      lm[k * RT + tid] = (uint8_t)li;
      bud[k * RT + tid] = (uint8_t)b;
      left -= p[i];
      done += p[i];
      b -= li;
      tot += li;
    }
    tots[tid] = tot;
  }
  __syncthreads();
  if (!on) return;                                 // no barriers below; whole rows leave
  const int tot = tots[tid];
  // rank with the index of mode x replaced by ix (and of mode y > x by iy)
  auto rank2 = [&](int x, int ix, int y, int iy) {
    int bb = bud[x * RT + tid];
    int32_t r = pre[x * RT + tid] + I.pre[(x * (LB + 1) + bb) * (NI + 1) + ix];
    bb -= I.lam[x * NI + ix];
    for (int k = x + 1; k < D; ++k) {
      const int i = (k == y) ? iy : dg[k * RT + tid];
      r += I.pre[(k * (LB + 1) + bb) * (NI + 1) + i];
      bb -= I.lam[k * NI + i];
    }
    return (int32_t)(r + I.row0);
  };
  auto epos = [&](int p, int ia, int ib) {
    return (int)I.pos[I.posoff[p] + ia * I.n[I.pb[p] * L1 + L] + ib];
  };
  // element of a pair's matrix at its level m, rows (ia, ib) -> (ja, jb)
  auto eget = [&](const NmSet& s, int p, int m, int ri, int ci) {
    const int64_t o = s.eoff[(int64_t)(I.pair0 + p) * pr.eld + m];
    return o < 0 ? 0.0 : s.E[o + (int64_t)ri * I.s2n[p * L1 + m] + ci];
  };
  const int32_t* nz = pr.nz + pr.nzoff[ii];
  const int ntask = D + pr.nzoff[ii + 1] - pr.nzoff[ii];
  // the entries of a task: put(x, ix, y, iy, v, vm) for each
  auto each = [&](int task, auto&& put) {
    if (task < D) {
      const int a = task, ia = dg[a * RT + tid], la = lm[a * RT + tid], ma = L - (tot - la);
      const int na = I.n[a * L1 + ma], room = LB - (tot - la);
      const double* g = sv.g1 + I.g1off[a * L1 + ma] + ia * na;
      const double* gm = MU ? sm.g1 + I.g1off[a * L1 + ma] + ia * na : nullptr;
      const int q0 = pr.adjoff[ii * 33 + a], q1 = pr.adjoff[ii * 33 + a + 1];
      for (int j = 0; j < na; ++j) {
        if (j == ia || I.lam[a * NI + j] > room) continue;
        double v = g[j], vm = MU ? gm[j] : 0.0;
        for (int q = q0; q < q1; ++q) {
          const int p = pr.adj[q];
          const bool fst = I.pa[p] == a;
          const int o = fst ? I.pb[p] : I.pa[p], io = dg[o * RT + tid];
          const int m = L - (tot - la - lm[o * RT + tid]);
          const int ri = fst ? epos(p, ia, io) : epos(p, io, ia);
          const int ci = fst ? epos(p, j, io) : epos(p, io, j);
          v += eget(sv, p, m, ri, ci);
          if constexpr (MU) vm += eget(sm, p, m, ri, ci);
        }
        if (v != 0.0 || vm != 0.0) put(a, j, -1, 0, v, vm);
      }
    } else {
      const int p = nz[task - D], a = I.pa[p], bq = I.pb[p];
      const int ia = dg[a * RT + tid], ib = dg[bq * RT + tid];
      const int lab = lm[a * RT + tid] + lm[bq * RT + tid];
      const int m = L - (tot - lab), room = LB - (tot - lab), S = I.s2n[p * L1 + m];
      const uint16_t* lst = I.s2 + I.s2off[p];
      const int ri = epos(p, ia, ib);
      const int64_t ov = sv.eoff[(int64_t)(I.pair0 + p) * pr.eld + m];
      const int64_t om = MU ? sm.eoff[(int64_t)(I.pair0 + p) * pr.eld + m] : -1;
      const int64_t g = (int64_t)(I.pair0 + p) * pr.eld + m;
      const uint16_t* el = pr.elist + pr.loff[g] + (int64_t)ri * S;
      const int ne = pr.ecnt[pr.croff[g] + ri];
      for (int x = 0; x < ne; ++x) {
        const int c = el[x], ja = lst[c] & 255, jb = lst[c] >> 8;
        if (room < m && I.lam[a * NI + ja] + I.lam[bq * NI + jb] > room) continue;   // LB < L
        const double v = ov < 0 ? 0.0 : sv.E[ov + (int64_t)ri * S + c];
        const double vm = om < 0 ? 0.0 : sm.E[om + (int64_t)ri * S + c];
        put(a, ja, bq, jb, v, vm);
      }
    }
  };
  if constexpr (!FILL) {
    int n = 0;
    for (int task = sub; task < ntask; task += RL)
      each(task, [&](int, int, int, int, double, double) { ++n; });
    for (int o = 1; o < RL; o <<= 1) n += __shfl_xor(n, o, 64);
    if (sub == 0) cnt[row] = n + 1;
  } else {
    int64_t at = ptr[row];
    double dv = 0.0, dm = 0.0;                     // the diagonal, first in its row
    for (int task = sub; task < ntask; task += RL) {
      if (task < D) {
        const int i = dg[task * RT + tid], ma = L - (tot - lm[task * RT + tid]);
        const int o = I.g1off[task * L1 + ma] + i * (I.n[task * L1 + ma] + 1);
        dv += sv.g1[o];
        if constexpr (MU) dm += sm.g1[o];
      } else {
        const int p = nz[task - D], a = I.pa[p], bq = I.pb[p];
        const int m = L - (tot - lm[a * RT + tid] - lm[bq * RT + tid]);
        const int e = epos(p, dg[a * RT + tid], dg[bq * RT + tid]);
        dv += eget(sv, p, m, e, e);
        if constexpr (MU) dm += eget(sm, p, m, e, e);
      }
    }
    for (int o = 1; o < RL; o <<= 1) {
      dv += __shfl_xor(dv, o, 64);
      if constexpr (MU) dm += __shfl_xor(dm, o, 64);
    }
    if (sub == 0) {
      col[at] = (int32_t)row;
      val[at] = dv + sv.c1[I.c1base];
      if constexpr (MU) valm[at] = dm + sm.c1[I.c1base];
    }
    ++at;
    for (int base = 0; base < ntask; base += RL) {   // the same number of rounds in every lane of a row
      const int task = base + sub;
      int n = 0;
      if (task < ntask) each(task, [&](int, int, int, int, double, double) { ++n; });
      int before = 0, all = n;
      for (int o = 1; o < RL; o <<= 1) {
        const int y = __shfl_up(all, o, RL);
        if (sub >= o) all += y;
      }
      before = all - n;
      int64_t w = at + before;
      if (n)
        each(task, [&](int x, int ix, int y, int iy, double v, double vm) {
          col[w] = rank2(x, ix, y, iy);
          val[w] = v;
          if constexpr (MU) valm[w] = vm;
          ++w;
        });
      at += __shfl(all, RL - 1, RL);
    }
  }
}

// row pointers from the row counts: sums (and the longest row) of 1024 rows,
// their scan with the total and the longest row of all behind it, the rows
__global__ __launch_bounds__(256) void k_nm_sum(const int32_t* cnt, int64_t n, int64_t* part, int32_t* most) {
  __shared__ int64_t s[256];
  __shared__ int m[256];
  int64_t a = 0;
  int b = 0;
  for (int k = 0; k < 4; ++k) {
    const int64_t i = (int64_t)blockIdx.x * 1024 + k * 256 + threadIdx.x;
    if (i < n) { a += cnt[i]; b = max(b, cnt[i]); }
  }
  s[threadIdx.x] = a;
  m[threadIdx.x] = b;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      s[threadIdx.x] += s[threadIdx.x + o];
      m[threadIdx.x] = max(m[threadIdx.x], m[threadIdx.x + o]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) { part[blockIdx.x] = s[0]; most[blockIdx.x] = m[0]; }
}
__global__ __launch_bounds__(1024) void k_nm_scan_part(int64_t* part, const int32_t* most, int np) {
  __shared__ int64_t s[1024];
  __shared__ int longest;
  if (threadIdx.x == 0) longest = 0;
  __syncthreads();
  int64_t carry = 0;
  int len = 0;
  for (int b = 0; b < np; b += 1024) {
    const int i = b + threadIdx.x;
    const int64_t x = i < np ? part[i] : 0;
    if (i < np) len = max(len, most[i]);
    s[threadIdx.x] = x;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
      const int64_t y = (int)threadIdx.x >= o ? s[threadIdx.x - o] : 0;
      __syncthreads();
      s[threadIdx.x] += y;
      __syncthreads();
    }
    if (i < np) part[i] = carry + s[threadIdx.x] - x;
    const int64_t total = s[1023];
    __syncthreads();
    carry += total;
  }
  atomicMax(&longest, len);
  __syncthreads();
  if (threadIdx.x == 0) { part[np] = carry; part[np + 1] = longest; }
}
__global__ __launch_bounds__(1024) void k_nm_ptr(const int32_t* cnt, int64_t n, const int64_t* part,
                                                 int64_t* ptr) {
  __shared__ int64_t s[1024];
  const int64_t i = (int64_t)blockIdx.x * 1024 + threadIdx.x;
  const int64_t x = i < n ? cnt[i] : 0;
  s[threadIdx.x] = x;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    const int64_t y = (int)threadIdx.x >= o ? s[threadIdx.x - o] : 0;
    __syncthreads();
    s[threadIdx.x] += y;
    __syncthreads();
  }
  if (i < n) ptr[i] = part[blockIdx.x] + s[threadIdx.x] - x;
  if (i == n - 1) ptr[n] = part[blockIdx.x] + s[threadIdx.x];
}

struct alignas(8) Two { double x, y; };

// Workgroups of the products in x and z: a launch takes fewer than 2^32 threads
// in a direction, which 16 lanes a row reach at 2^28 rows.  The stride is a
// constant: a product of few rows would wait for the grid's size (6D L=3 x1
// 4.65 -> 4.8 us).
constexpr int64_t MAX_BLOCKS_X = (int64_t)1 << 23;
__device__ __forceinline__ int64_t block_xz() { return blockIdx.x + MAX_BLOCKS_X * blockIdx.z; }
dim3 grid_xz(int64_t blocks, int y) {
  return dim3((unsigned)std::min(blocks, MAX_BLOCKS_X), (unsigned)y,
              (unsigned)((blocks + MAX_BLOCKS_X - 1) / MAX_BLOCKS_X));
}

// hpsi(r, v) = sum_e val_e psi(col_e, v): NV * SL lanes per row, NV vectors,
// the row's entries dealt to SL slices that are added at the end.
// OUT_COLS: the result goes to the column-major block (nvec <= NV columns),
// through LDS so that a workgroup writes runs of its 256 / W rows.  IN_COLS:
// psi is column-major too (a gather of NV values touches NV lines).
template <int NV, int SL, bool COLS, bool IN_COLS>
__global__ __launch_bounds__(256) void k_nm_spmm(const int64_t* __restrict__ ptr,
                                                 const int32_t* __restrict__ col,
                                                 const double* __restrict__ val,
                                                 const double* __restrict__ psi,
                                                 double* __restrict__ hpsi, int64_t rows, int nvec,
                                                 float* __restrict__ psi32) {
  constexpr int W = NV * SL, R = 256 / W;
  __shared__ double tile[COLS ? NV * (R + 1) : 1];
  const int l = threadIdx.x % W, v = l % NV, s = l / NV;
  const int64_t r = block_xz() * R + threadIdx.x / W;
  const double* __restrict__ x0 = IN_COLS ? psi + (int64_t)min(v, nvec - 1) * rows : psi + v;
  constexpr int LD = IN_COLS ? 1 : NV;
  double a = 0.0;
  if (r < rows) {
    const int64_t e1 = ptr[r + 1];
    int64_t e = ptr[r] + s;
    double a0 = 0.0, a1 = 0.0;
    for (; e + 3 * SL < e1; e += 4 * SL) {
      int32_t c[4];
      double w[4], x[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) { c[u] = col[e + u * SL]; w[u] = val[e + u * SL]; }
#pragma unroll
      for (int u = 0; u < 4; ++u) x[u] = x0[(int64_t)c[u] * LD];
#pragma unroll
      for (int u = 0; u < 4; u += 2) { a0 = fma(w[u], x[u], a0); a1 = fma(w[u + 1], x[u + 1], a1); }
    }
    for (; e < e1; e += SL) a0 = fma(val[e], x0[(int64_t)col[e] * LD], a0);
    a = a0 + a1;
#pragma unroll
    for (int o = NV; o < W; o <<= 1) a += __shfl_xor(a, o, 64);
    if (!COLS && s == 0) {
      hpsi[r * NV + v] = a;
      if (psi32) psi32[r * NV + v] = (float)psi[r * NV + v];
    }
  }
  if constexpr (COLS) {
    if (s == 0) tile[v * (R + 1) + threadIdx.x / W] = a;
    __syncthreads();
    for (int t = threadIdx.x; t < NV * R; t += 256) {
      const int vv = t / R, rr = t % R;
      const int64_t ro = block_xz() * R + rr;
      if (vv < nvec && ro < rows) hpsi[(int64_t)vv * rows + ro] = tile[vv * (R + 1) + rr];
    }
  }
}
// The same from a rows-layout block: a lane holds PV pairs of columns (16-byte
// loads), NC lanes a row and slice, SL slices, SU entries in flight per lane.
// WIDE: blocks of NV columns of a wider block (blockIdx.y; multiples of 8: 9D
// L=7 x32 162 -> 112 us; three blocks of 4 at x12 85 -> 127, not taken).  Bound by the rate
// at which lines are requested: few lanes per line, many entries of a row per
// wave.  10D L=8 (32 M entries) x16 440 us, x8 286, x4 207, x2 155; with one
// column per lane 750, 446, 306, 197; one pair 497, 338, 225, 155; two pairs and
// 1 / 2 / 8 slices at x16 624 / 474 / 437, four pairs 452-528.
template <int NC, int PV, int SL, int SU, bool COLS, bool WIDE>
__global__ __launch_bounds__(256) void k_nm_spmm_pairs(const int64_t* __restrict__ ptr,
                                                       const int32_t* __restrict__ col,
                                                       const double* __restrict__ val,
                                                       const double* __restrict__ psi,
                                                       double* __restrict__ hpsi, int64_t rows, int nvec,
                                                       float* __restrict__ psi32) {
  constexpr int W = NC * SL, R = 256 / W, NV = 2 * NC * PV;
  __shared__ double tile[COLS ? NV * (R + 1) : 1];
  const int l = threadIdx.x % W, j = l % NC, s = l / NC, rr = threadIdx.x / W;
  const int64_t r = block_xz() * R + rr;
  const int64_t ld = WIDE ? nvec / 2 : NC * PV;           // pairs per row
  const int64_t j0 = j + (WIDE ? (int64_t)blockIdx.y * (NC * PV) : 0);
  const Two* __restrict__ x = (const Two*)psi + j0;
  Two y[PV];
#pragma unroll
  for (int p = 0; p < PV; ++p) y[p] = Two{0.0, 0.0};
  if (r < rows) {
    const int64_t e1 = ptr[r + 1];
    int64_t e = ptr[r] + s;
    for (; e + (SU - 1) * SL < e1; e += SU * SL) {
      int32_t c[SU];
      double w[SU];
      Two xv[SU][PV];
#pragma unroll
      for (int u = 0; u < SU; ++u) { c[u] = col[e + u * SL]; w[u] = val[e + u * SL]; }
#pragma unroll
      for (int u = 0; u < SU; ++u)
#pragma unroll
        for (int p = 0; p < PV; ++p) xv[u][p] = x[c[u] * ld + p * NC];
#pragma unroll
      for (int u = 0; u < SU; ++u)
#pragma unroll
        for (int p = 0; p < PV; ++p) {
          y[p].x = fma(w[u], xv[u][p].x, y[p].x);
          y[p].y = fma(w[u], xv[u][p].y, y[p].y);
        }
    }
    for (; e < e1; e += SL) {
      const double w = val[e];
      const int64_t c = col[e] * ld;
#pragma unroll
      for (int p = 0; p < PV; ++p) {
        const Two xv = x[c + p * NC];
        y[p].x = fma(w, xv.x, y[p].x);
        y[p].y = fma(w, xv.y, y[p].y);
      }
    }
  }
#pragma unroll
  for (int o = NC; o < W; o <<= 1)
#pragma unroll
    for (int p = 0; p < PV; ++p) {
      y[p].x += __shfl_xor(y[p].x, o, 64);
      y[p].y += __shfl_xor(y[p].y, o, 64);
    }
  if constexpr (!COLS) {
    if (r < rows && s == 0)
#pragma unroll
      for (int p = 0; p < PV; ++p) {
        const int64_t at = r * ld + j0 + p * NC;
        ((Two*)hpsi)[at] = y[p];
        if (psi32) {
          const Two v = ((const Two*)psi)[at];
          *(float2*)(psi32 + 2 * at) = make_float2((float)v.x, (float)v.y);
        }
      }
  } else {
    if (s == 0)
#pragma unroll
      for (int p = 0; p < PV; ++p) {
        tile[2 * (p * NC + j) * (R + 1) + rr] = y[p].x;
        tile[(2 * (p * NC + j) + 1) * (R + 1) + rr] = y[p].y;
      }
    __syncthreads();
    for (int t = threadIdx.x; t < NV * R; t += 256) {
      const int vv = t / R, ro = t % R;
      const int64_t row = block_xz() * R + ro;
      if (vv < nvec && row < rows) hpsi[(int64_t)vv * rows + row] = tile[vv * (R + 1) + ro];
    }
  }
}
// any number of vectors: SL threads per (row, vector)
template <int SL>
__global__ __launch_bounds__(256) void k_nm_spmm_any(const int64_t* __restrict__ ptr,
                                                     const int32_t* __restrict__ col,
                                                     const double* __restrict__ val,
                                                     const double* __restrict__ psi,
                                                     double* __restrict__ hpsi, int64_t rows, int nvec,
                                                     float* __restrict__ psi32) {
  const int64_t n = rows * nvec;
  const int s = threadIdx.x % SL;
  // whole groups of SL lanes stay in the loop
  for (int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) / SL; i < n; i += (int64_t)gridDim.x * (256 / SL)) {
    const int64_t r = i / nvec;
    const int v = (int)(i - r * nvec);
    const int64_t e1 = ptr[r + 1];
    int64_t e = ptr[r] + s;
    double a0 = 0.0, a1 = 0.0;
    for (; e + 3 * SL < e1; e += 4 * SL) {
      int32_t c[4];
      double w[4], x[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) { c[u] = col[e + u * SL]; w[u] = val[e + u * SL]; }
#pragma unroll
      for (int u = 0; u < 4; ++u) x[u] = psi[(int64_t)c[u] * nvec + v];
#pragma unroll
      for (int u = 0; u < 4; u += 2) { a0 = fma(w[u], x[u], a0); a1 = fma(w[u + 1], x[u + 1], a1); }
    }
    for (; e < e1; e += SL) a0 = fma(val[e], psi[(int64_t)col[e] * nvec + v], a0);
    a0 += a1;
#pragma unroll
    for (int o = 1; o < SL; o <<= 1) a0 += __shfl_xor(a0, o, 64);
    if (s != 0) continue;
    hpsi[i] = a0;
    if (psi32) psi32[i] = (float)psi[i];
  }
}

// Rows that leave the chip idle with four slices: eight shorten the chain (3
// small instances 4.0 -> 3.4 us an order, tangents 5.2 -> 4.1; 12 uneven ones,
// 130 k rows, 19.7 -> 22.3).
constexpr int64_t ORDER_FEW = 32768;

// Few rows of which one is long: its chain decides, and a wave takes a row (16 to
// 64 slices).  Many modes all coupled in pairs, us, before -> so (the term kernels
// in brackets): 32D L=2 (row of 2113 entries) x8 58 -> 13 (28), x16 61 -> 17 (29),
// 16D L=3 (1537) x8 47 -> 13 (34), 12D L=3 (865) x16 29 -> 13 (24); an order of one
// state 40 -> 5 (24) at 32D.  Rows up to 250 entries (6D L=4, 5D L=5) are faster in
// place: x8 16-18 (23).
constexpr int64_t LONG_ROW = 256;

// A Chebyshev order (NModeOrder).  A lane holds two neighbouring columns (one
// 16-byte load per entry), NC * SL lanes a row; the row's entries are dealt to
// SL slices, OU of them in flight per lane, and all slices hold the sums after
// the exchange.  The partner column (re <-> im) is the lane's other one for one
// state, NS / 2 lanes away else; mu w comes from NS lanes away.  One launch per
// order instead of the kinetic rows, the term kernel and the element-wise order
// (and, with tangents, the dipole operator's two and a copy).  Bound by the
// latency of the chain row -> column -> vector for small instances and by the
// gathers for large ones: 12 uneven instances, 6 steps of 15 orders, 35.4 -> 2.9
// ms, 20 us an order (one column per lane, two entries in flight: 3.9 and 30; SL
// 2 / 8 / 16: 3.3 / 3.1 / 3.4 ms; 2 or 6 entries: 3.1, 2.9), the adjoint gradient
// of 3 small ones 8.6 -> 1.8.
template <int NC, int SL, bool TAN>
__global__ __launch_bounds__(256) void k_nm_order(const int64_t* __restrict__ ptr,
                                                  const int32_t* __restrict__ col,
                                                  const double* __restrict__ mu, NModeOrder a,
                                                  int64_t rows) {
  constexpr int W = NC * SL, NS = TAN ? NC / 2 : NC, OU = 4;
  const int l = threadIdx.x % W, j = l % NC, s = l / NC;
  const double* __restrict__ val = a.val;
  const Two* __restrict__ x = (const Two*)a.wk;
  // whole waves stay in the loop: the exchanges need every lane of a row
  const int64_t r0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) / W;
  for (int64_t r = r0; r < rows; r += (int64_t)gridDim.x * (256 / W)) {
    const int64_t e0 = ptr[r], e1 = ptr[r + 1], at = r * NC + j;
    const bool tan = TAN && j >= NS;
    const int64_t ai = TAN ? r * NS + (tan ? j - NS : j) : at;
    Two* acc = (Two*)(tan ? a.tacc : a.acc);
    Two* out = (Two*)(tan ? a.tout : a.out);
    const Two xr = x[at];
    Two wm{0.0, 0.0}, ac{a.c0 * xr.x, a.c0 * xr.y};
    if (!a.first) {
      wm = ((const Two*)a.wm)[at];
      ac = acc[ai];
    }
    Two y{0.0, 0.0}, m{0.0, 0.0};
    for (int64_t e = e0 + s; e < e1; e += OU * SL) {
      Two xv[OU];
      double w[OU], u[OU];
#pragma unroll
      for (int k = 0; k < OU; ++k) {
        const int64_t i = min(e + k * SL, e1 - 1);
        xv[k] = x[(int64_t)col[i] * NC + j];
        w[k] = val[i];
        if constexpr (TAN) u[k] = mu[i];
      }
#pragma unroll
      for (int k = 0; k < OU; ++k) {
        if (e + k * SL >= e1) continue;
        y.x = fma(w[k], xv[k].x, y.x);
        y.y = fma(w[k], xv[k].y, y.y);
        if constexpr (TAN) {
          m.x = fma(u[k], xv[k].x, m.x);
          m.y = fma(u[k], xv[k].y, m.y);
        }
      }
    }
#pragma unroll
    for (int o = NC; o < W; o <<= 1) {
      y.x += __shfl_xor(y.x, o, 64);
      y.y += __shfl_xor(y.y, o, 64);
      if constexpr (TAN) {
        m.x += __shfl_xor(m.x, o, 64);
        m.y += __shfl_xor(m.y, o, 64);
      }
    }
    Two z{y.x - a.E0 * xr.x, y.y - a.E0 * xr.y};
    if constexpr (TAN) {
      const double mx = __shfl_xor(m.x, NS, 64), my = __shfl_xor(m.y, NS, 64);
      if (tan) {
        z.x += mx;
        z.y += my;
      }
    }
    z.x *= a.sc;
    z.y *= a.sc;
    // the partner's z and the sign of the imaginary unit on this column
    const bool im = NS > 1 && (j & (NS / 2));
    const double sx = im ? a.sgn : -a.sgn, sy = NS == 1 ? a.sgn : sx;
    Two zp{z.y, z.x};
    if constexpr (NS > 1) zp = Two{__shfl_xor(z.x, NS / 2, 64), __shfl_xor(z.y, NS / 2, 64)};
    Two wn{sx * zp.x, sy * zp.y};
    if (!a.first) wn = Two{fma(2.0 * sx, zp.x, wm.x), fma(2.0 * sy, zp.y, wm.y)};
    ac.x = fma(a.c, wn.x, ac.x);
    ac.y = fma(a.c, wn.y, ac.y);
    if (a.last) {
      Two ap{ac.y, ac.x};
      if constexpr (NS > 1) ap = Two{__shfl_xor(ac.x, NS / 2, 64), __shfl_xor(ac.y, NS / 2, 64)};
      const double px = im ? a.pi : -a.pi, py = NS == 1 ? a.pi : px;
      if (s == 0) out[ai] = Two{ac.x * a.pr + ap.x * px, ac.y * a.pr + ap.y * py};
    } else if (s == 0) {
      ((Two*)a.wm)[at] = wn;
      acc[ai] = ac;
    }
  }
}

__global__ __launch_bounds__(256) void k_nm_field(const double* __restrict__ val,
                                                  const double* __restrict__ mu, double eps,
                                                  double* __restrict__ out, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
    out[i] = fma(eps, mu[i], val[i]);
}

__global__ void k_nm_zero(int* p, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
}

// a host byte block whose sections become device pointers after one copy
struct Blob {
  std::vector<char> h;
  template <class T>
  size_t add(const std::vector<T>& v) {
    const size_t o = (h.size() + 15) & ~(size_t)15;
    h.resize(o + sizeof(T) * std::max<size_t>(v.size(), 1));
    if (!v.empty()) std::memcpy(&h[o], v.data(), sizeof(T) * v.size());
    return o;
  }
};

int upload(const Blob& b, DevBuf& d, hipStream_t st) {
  int rc;
  if (d.n < b.h.size() && (rc = d.alloc(b.h.size()))) return rc;
  NM_TRY(hipMemcpyAsync(d.p, b.h.data(), b.h.size(), hipMemcpyHostToDevice, st));
  NM_TRY(hipStreamSynchronize(st));   // the host block is pageable and goes away
  return SG4_OK;
}

int ensure(DevBuf& d, size_t bytes) { return d.n >= bytes && d.p ? SG4_OK : d.alloc(std::max<size_t>(bytes, 256)); }

}  // namespace

struct NModeTables {
  bool rows_ok = false;            // the packed rows are in lexicographic order
  bool cuts = true, ok = false;    // V can be cut through middle points; both
  DevBuf blob, insts, work, ck;    // tables; NmDev of every instance; build workspace; c_k
  DevBuf e_v, e_mu, elist, lists;
  std::vector<NmDev> dev;          // host copies (device pointers inside)
  size_t o_term0 = 0, o_blk0 = 0, o_cut1 = 0, o_cut2 = 0, o_g1work = 0, o_none = 0;
  int ncut1 = 0, ncut2 = 0, ng1 = 0, npairs = 0, Lmax = 0, Dmax = 0;
  int64_t nc1 = 0, nf2 = 0, ng1v = 0, nterms = 0, nblk = 0;
  bool v_ready = false;            // V's part of work, e_v and v_flags hold the plan's operator
  std::vector<int> v_flags;
  std::vector<int32_t> pair_inst, pair_s2n;   // per global pair: instance; [pair * (Lmax+1) + m]
};

void nmode_tables_destroy(NModeTables* t) { delete t; }

NModeTables* nmode_tables_create(const NModeIn& in) {
  auto t = std::make_unique<NModeTables>();
  // a plan without them: no sparse matrices, K from the host
  auto no_memory = [] { return new NModeTables; };
  const int ni = (int)in.inst.size();
  t->dev.resize(ni);
  for (const NModeInst& I : in.inst) {
    t->Lmax = std::max(t->Lmax, I.L);
    t->Dmax = std::max(t->Dmax, I.D);
    t->nterms += I.nterms;
  }
  Blob blob;
  struct Off { size_t n, lam, pre, f1off, f2off, s2n, s2off, s2, posoff, pos, pa, pb, T, toff, g1off; };
  std::vector<Off> off(ni);
  std::vector<Cut> cut1, cut2;
  std::vector<int32_t> g1work;
  std::vector<int64_t> term0, blk0;
  for (int x = 0; x < ni; ++x) {
    const NModeInst& I = in.inst[x];
    NmDev& d = t->dev[x];
    const int D = I.D, L = I.L, L1 = L + 1, M1 = I.Lmax + 1;
    d.D = D; d.L = L; d.L1 = M1;
    d.term0 = I.term0; d.nterms = I.nterms; d.row0 = I.row0; d.nrows = I.nb_ba;
    auto nn = [&](int k, int l) { return (*in.nq)[I.md0 + (int64_t)k * M1 + l]; };
    std::vector<int32_t> n(D * L1);
    for (int k = 0; k < D; ++k)
      for (int l = 0; l <= L; ++l) {
        n[k * L1 + l] = nn(k, l);
        if (n[k * L1 + l] > NI || (l && n[k * L1 + l] < n[k * L1 + l - 1])) return t.release();
        // the middle point is shared by the rules of a mode when they are odd
        if (n[k * L1 + l] % 2 == 0 || n[k * L1] != 1) t->cuts = false;
      }
    std::vector<uint8_t> lam(D * NI, 255);
    for (int k = 0; k < D; ++k)
      for (int i = 0; i < NI; ++i)
        for (int l = 0; l <= L; ++l)
          if (n[k * L1 + l] > i) { lam[k * NI + i] = (uint8_t)l; break; }
    // basis level from the number of packed rows
    int LB = -1;
    std::vector<int64_t> cnt((D + 1) * L1, 0);
    for (int b = 0; b <= L; ++b) cnt[D * L1 + b] = 1;
    for (int k = D - 1; k >= 0; --k)
      for (int b = 0; b <= L; ++b)
        for (int i = 0; i < NI && lam[k * NI + i] <= b; ++i) cnt[k * L1 + b] += cnt[(k + 1) * L1 + b - lam[k * NI + i]];
    for (int b = 0; b <= L; ++b)
      if (cnt[b] == I.nb_ba) LB = b;
    if (LB < 0 || I.nb_ba > INT32_MAX) return t.release();
    d.LB = LB;
    std::vector<int32_t> pre((size_t)D * (LB + 1) * (NI + 1), -1);
    for (int k = 0; k < D; ++k)
      for (int b = 0; b <= LB; ++b) {
        int64_t s = 0;
        for (int i = 0; i <= NI; ++i) {
          pre[((size_t)k * (LB + 1) + b) * (NI + 1) + i] = (int32_t)s;
          if (i == NI || lam[k * NI + i] > b) break;
          s += cnt[(k + 1) * L1 + b - lam[k * NI + i]];
        }
      }
    // cuts: for every (mode, level) and (pair, levels >= 1) the first term that
    // has them; the other modes at their middle points
    const int np = t->cuts ? D * (D - 1) / 2 : 0;
    d.npair = np;
    d.pair0 = t->npairs;
    std::vector<uint8_t> pa(np), pb(np);
    for (int a = 0, p = 0; a < D && np; ++a)
      for (int b = a + 1; b < D; ++b, ++p) { pa[p] = (uint8_t)a; pb[p] = (uint8_t)b; }
    std::vector<int32_t> f1off(D * L1, -1), f2off((size_t)np * L1 * L1, -1);
    d.c1base = t->nc1;
    t->nc1 += 1;
    std::vector<int> act;
    std::vector<int64_t> stride(D);
    bool centre = false;
    std::vector<Cut> c2;
    for (int64_t tt = 0; tt < I.nterms && t->cuts; ++tt) {
      const int32_t* lev = &(*in.levels)[I.lev0 + tt * D];
      act.clear();
      int64_t s = 1, mid = (*in.qoff)[I.term0 + tt];
      for (int k = 0; k < D; ++k) {
        const int nk = n[k * L1 + lev[k]];
        stride[k] = s;
        mid += s * (nk / 2);
        s *= nk;
        if (nk > 1) act.push_back(k);
      }
      auto cut = [&](int a, int b) {
        Cut c{};
        const int na = n[a * L1 + lev[a]];
        c.sa = (int32_t)stride[a]; c.na = na; c.sb = 0; c.nb = 1; c.pair = -1;
        c.off = mid - stride[a] * (na / 2);
        if (b >= 0) {
          const int nb = n[b * L1 + lev[b]];
          c.sb = (int32_t)stride[b]; c.nb = nb;
          c.off -= stride[b] * (nb / 2);
        }
        return c;
      };
      if (!centre) {
        Cut c{};
        c.off = mid; c.na = 1; c.nb = 1; c.out = d.c1base; c.pair = -1;
        cut1.push_back(c);
        centre = true;
      }
      for (size_t u = 0; u < act.size(); ++u) {
        const int a = act[u];
        if (f1off[a * L1 + lev[a]] < 0) {
          Cut c = cut(a, -1);
          c.out = t->nc1;
          f1off[a * L1 + lev[a]] = (int32_t)c.out;
          t->nc1 += c.na;
          cut1.push_back(c);
        }
        for (size_t w = u + 1; w < act.size(); ++w) {
          const int b = act[w], p = a * (2 * D - a - 1) / 2 + (b - a - 1);
          int32_t& o = f2off[((size_t)p * L1 + lev[a]) * L1 + lev[b]];
          if (o >= 0) continue;
          Cut c = cut(a, b);
          c.out = t->nf2;
          c.pair = d.pair0 + p;
          c.v0 = d.c1base;
          c.fa = lev[a]; c.fb = lev[b];   // resolved below
          c2.push_back(c);
          o = (int32_t)t->nf2;
          t->nf2 += (int64_t)c.na * c.nb;
        }
      }
      if (t->nf2 > INT32_MAX || t->nc1 > INT32_MAX) return t.release();
    }
    for (Cut& c : c2) {
      const int p = c.pair - d.pair0;
      c.fa = f1off[pa[p] * L1 + (int)c.fa];
      c.fb = f1off[pb[p] * L1 + (int)c.fb];
      cut2.push_back(c);
    }
    // pair indices by level, and their positions
    std::vector<int32_t> s2n((size_t)np * L1), s2off(np), posoff(np);
    std::vector<uint16_t> s2;
    std::vector<int16_t> pos;
    std::map<std::vector<int32_t>, std::pair<int32_t, int32_t>> known;   // modes of equal sizes share a list
    for (int p = 0; p < np; ++p) {
      const int a = pa[p], b = pb[p], nA = n[a * L1 + L], nB = n[b * L1 + L];
      std::vector<int32_t> key(n.begin() + a * L1, n.begin() + (a + 1) * L1);
      key.insert(key.end(), n.begin() + b * L1, n.begin() + (b + 1) * L1);
      auto f = known.find(key);
      const bool fresh = f == known.end();
      if (fresh) f = known.emplace(key, std::make_pair((int32_t)s2.size(), (int32_t)pos.size())).first;
      s2off[p] = f->second.first;
      posoff[p] = f->second.second;
      if (fresh) pos.resize(pos.size() + (size_t)nA * nB, -1);
      int c = 0;
      for (int m = 0; m <= L; ++m) {
        for (int ia = 0; ia < nA; ++ia)
          for (int ib = 0; ib < nB; ++ib)
            if (lam[a * NI + ia] + lam[b * NI + ib] == m) {
              if (fresh) {
                s2.push_back((uint16_t)(ia | ib << 8));
                pos[posoff[p] + (size_t)ia * nB + ib] = (int16_t)c;
              }
              ++c;
            }
        s2n[(size_t)p * L1 + m] = c;
      }
      if (c > INT16_MAX) return t.release();
      t->pair_inst.push_back(x);
    }
    std::vector<int32_t> g1off(D * L1), toff(D * L1);
    std::vector<double> T;
    for (int k = 0; k < D; ++k) {
      for (int l = 0; l <= L; ++l) {
        const int nk = n[k * L1 + l];
        g1off[k * L1 + l] = (int32_t)t->ng1v;
        t->ng1v += (int64_t)nk * nk;
        toff[k * L1 + l] = (int32_t)T.size();
        const double* src = in.T->data() + (*in.toff)[I.md0 + (int64_t)k * M1 + l];
        T.insert(T.end(), src, src + (size_t)nk * nk);
        g1work.insert(g1work.end(), {x, k, l});
      }
    }
    if (t->ng1v > INT32_MAX) return t.release();
    term0.push_back(I.term0);
    blk0.push_back(t->nblk);
    t->nblk += (I.nb_ba + RT - 1) / RT;
    Off& o = off[x];
    o.n = blob.add(n); o.lam = blob.add(lam); o.pre = blob.add(pre); o.f1off = blob.add(f1off);
    o.f2off = blob.add(f2off); o.s2n = blob.add(s2n); o.s2off = blob.add(s2off); o.s2 = blob.add(s2);
    o.posoff = blob.add(posoff); o.pos = blob.add(pos); o.pa = blob.add(pa); o.pb = blob.add(pb);
    o.T = blob.add(T); o.toff = blob.add(toff); o.g1off = blob.add(g1off);
    for (int p = 0; p < np; ++p)
      for (int m = 0; m <= t->Lmax; ++m) t->pair_s2n.push_back(m <= L ? s2n[(size_t)p * L1 + m] : 0);
    t->npairs += np;
  }
  t->ncut1 = (int)cut1.size();
  t->ncut2 = (int)cut2.size();
  t->ng1 = (int)g1work.size() / 3;
  t->o_term0 = blob.add(term0);
  t->o_blk0 = blob.add(blk0);
  t->o_cut1 = blob.add(cut1);
  t->o_cut2 = blob.add(cut2);
  t->o_g1work = blob.add(g1work);
  t->o_none = blob.add(std::vector<int32_t>((size_t)ni * 33 + 33, 0));   // no pairs
  int rc = upload(blob, t->blob, in.stream);
  if (!rc) rc = t->ck.alloc(sizeof(double) * in.ck->size());
  if (rc) return rc == SG4_ERR_OOM ? no_memory() : nullptr;
  char* B = t->blob.as<char>();
  for (int x = 0; x < ni; ++x) {
    const NModeInst& I = in.inst[x];
    NmDev& d = t->dev[x];
    const Off& o = off[x];
    d.levels = in.d_levels + I.lev0;
    d.md = in.d_md + I.md0;
    d.n = (int32_t*)(B + o.n); d.lam = (uint8_t*)(B + o.lam); d.pre = (int32_t*)(B + o.pre);
    d.f1off = (int32_t*)(B + o.f1off); d.f2off = (int32_t*)(B + o.f2off); d.s2n = (int32_t*)(B + o.s2n);
    d.s2off = (int32_t*)(B + o.s2off); d.s2 = (uint16_t*)(B + o.s2); d.posoff = (int32_t*)(B + o.posoff);
    d.pos = (int16_t*)(B + o.pos); d.pa = (uint8_t*)(B + o.pa); d.pb = (uint8_t*)(B + o.pb);
    d.T = (double*)(B + o.T); d.toff = (int32_t*)(B + o.toff); d.ck = t->ck.as<double>() + I.ck0;
    d.g1off = (int32_t*)(B + o.g1off);
  }
  Blob ib;
  ib.add(t->dev);
  rc = upload(ib, t->insts, in.stream);
  if (!rc) rc = ensure(t->work, 256);
  if (rc) return rc == SG4_ERR_OOM ? no_memory() : nullptr;
  // the packed rows in lexicographic order?
  int* bad = t->work.as<int>();
  hipLaunchKernelGGL(k_nm_zero, dim3(1), dim3(64), 0, in.stream, bad, 1);
  hipLaunchKernelGGL(k_nm_check_map, dim3((unsigned)std::min<int64_t>(t->nterms, 16384)), dim3(256), 0,
                     in.stream, t->insts.as<NmDev>(), (const int64_t*)(B + t->o_term0), ni, t->nterms,
                     in.d_terms, in.d_map, bad);
  int h = 1;
  if (hipMemcpyAsync(&h, bad, sizeof(int), hipMemcpyDeviceToHost, in.stream) != hipSuccess ||
      hipStreamSynchronize(in.stream) != hipSuccess) {
    set_error("HIP error while checking the packed rows");
    return nullptr;
  }
  t->rows_ok = h == 0;
  t->ok = t->rows_ok && t->cuts;
  return t.release();
}

namespace {
size_t up(size_t b) { return (b + 255) & ~(size_t)255; }

// Build workspace: for V and for mu the cuts, two-mode functions, one-mode
// matrices and pair flags (then the verdict); the row counts and their scan.
struct Work {
  double *c1[2], *f2[2], *g1[2];
  int* flag[2];
  int32_t *cnt, *most;
  int64_t* part;
  int npart;
  int layout(NModeTables* t, int64_t rows) {
    npart = (int)((rows + 1023) / 1024);
    const size_t b_c1 = up(8 * t->nc1), b_f2 = up(8 * (t->nf2 + 1)), b_g1 = up(8 * t->ng1v),
                 b_fl = up(4 * ((size_t)t->npairs + 1)), b_set = b_c1 + b_f2 + b_g1 + b_fl,
                 b_cnt = up(4 * rows), b_part = up(8 * ((size_t)npart + 2));
    if (int rc = ensure(t->work, 2 * b_set + b_cnt + b_part + 4 * (size_t)npart)) return rc;
    char* W = t->work.as<char>();
    for (int s = 0; s < 2; ++s) {
      char* w = W + s * b_set;
      c1[s] = (double*)w;
      f2[s] = (double*)(w + b_c1);
      g1[s] = (double*)(w + b_c1 + b_f2);
      flag[s] = (int*)(w + b_c1 + b_f2 + b_g1);
    }
    cnt = (int32_t*)(W + 2 * b_set);
    part = (int64_t*)(W + 2 * b_set + b_cnt);
    most = (int32_t*)(W + 2 * b_set + b_cnt + b_part);
    return SG4_OK;
  }
};

// the row counts' sum and the longest row (synchronises)
int scan_rows(const Work& w, int64_t rows, hipStream_t st, int64_t* nnz, int64_t* longest) {
  hipLaunchKernelGGL(k_nm_sum, dim3(w.npart), dim3(256), 0, st, w.cnt, rows, w.part, w.most);
  hipLaunchKernelGGL(k_nm_scan_part, dim3(1), dim3(1024), 0, st, w.part, w.most, w.npart);
  int64_t h[2] = {0, 0};
  NM_TRY(hipMemcpyAsync(h, w.part + w.npart, sizeof(h), hipMemcpyDeviceToHost, st));
  NM_TRY(hipGetLastError());
  NM_TRY(hipStreamSynchronize(st));
  *nnz = h[0];
  *longest = h[1];
  return SG4_OK;
}
}  // namespace

// Host lists, cuts and the check of every pair, and a row's tasks, one per pair:
// beyond the launches and copies of any build (150 us) 32D L=2 (496 pairs) takes
// 3290 us, 21D 1500, 12D L=3 (66) 570; then the entries: 10D L=8 (32 M) 4100.
double nmode_field_cost(const NModeTables* t, const NModeMat& m) {
  int pairs = 0;
  for (int g = 0; g < t->npairs && g < (int)t->v_flags.size(); ++g) pairs += t->v_flags[g] != 0;
  return 150.0 + 6.5 * pairs + 1.3e-4 * (double)m.nnz;
}

bool nmode_rows_ok(const NModeTables* t) { return t && t->rows_ok; }

int nmode_build_kinetic(NModeTables* t, const NModeIn& in, NModeMat& m) {
  m.valid = false;
  const hipStream_t st = in.stream;
  const int64_t rows = in.rows;
  Work w;
  int rc;
  if ((rc = w.layout(t, rows))) return rc;
  char* B = t->blob.as<char>();
  const NmDev* insts = t->insts.as<NmDev>();
  t->v_ready = false;
  NM_TRY(hipMemcpyAsync(t->ck.p, in.ck->data(), sizeof(double) * in.ck->size(), hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(k_nm_zero, dim3(8), dim3(256), 0, st, (int*)w.c1[1], (int)(2 * t->nc1));   // V0 = 0
  hipLaunchKernelGGL(k_nm_g1, dim3(t->ng1), dim3(256), 0, st, insts, (const int32_t*)(B + t->o_g1work),
                     in.d_mats, w.c1[1], w.g1[1], G1_KIN);
  const NmSet set{w.c1[1], w.g1[1], nullptr, nullptr};
  const int32_t* none = (const int32_t*)(B + t->o_none);
  const NmPairs pr{none, none, none, none, nullptr, nullptr, nullptr, nullptr, 0};
  const dim3 rg((unsigned)t->nblk);
  const size_t rl = (size_t)t->Dmax * RT * 7;
  const int64_t* blk0 = (const int64_t*)(B + t->o_blk0);
  const int ni = (int)in.inst.size();
  hipLaunchKernelGGL((k_nm_rows<false, false>), rg, dim3(256), rl, st, insts, blk0, ni, set, set, pr, t->Dmax,
                     w.cnt, nullptr, nullptr, nullptr, nullptr);
  int64_t nnz = 0, longest = 0;
  if ((rc = scan_rows(w, rows, st, &nnz, &longest))) return rc;
  if ((rc = ensure(m.ptr, 8 * (rows + 1))) || (rc = ensure(m.col, 4 * nnz)) || (rc = ensure(m.val, 8 * nnz)))
    return rc;
  hipLaunchKernelGGL(k_nm_ptr, dim3(w.npart), dim3(1024), 0, st, w.cnt, rows, w.part, m.ptr.as<int64_t>());
  hipLaunchKernelGGL((k_nm_rows<true, false>), rg, dim3(256), rl, st, insts, blk0, ni, set, set, pr, t->Dmax,
                     w.cnt, m.ptr.as<int64_t>(), m.col.as<int32_t>(), m.val.as<double>(), nullptr);
  NM_TRY(hipGetLastError());
  m.rows = rows;
  m.nnz = nnz;
  m.longest = longest;
  m.valid = true;
  return SG4_OK;
}

int nmode_build(NModeTables* t, const NModeIn& in, const double* V, const double* mu, NModeMat& m) {
  m.valid = false;
  if (!t || !t->ok) return SG4_OK;
  const bool have_v = mu && t->v_ready;   // V's functions and matrices, made when the operator was set
  if (!have_v) t->v_ready = false;
  const hipStream_t st = in.stream;
  const int ni = (int)in.inst.size(), nset = mu ? 2 : 1, eld = t->Lmax + 1;
  const int64_t rows = in.rows;
  int rc;
  Work w;
  if (w.layout(t, rows)) return SG4_OK;   // no memory: term kernels
  char* B = t->blob.as<char>();
  auto& c1 = w.c1;
  auto& f2 = w.f2;
  auto& g1 = w.g1;
  auto& flag = w.flag;
  int32_t* cnt = w.cnt;
  int64_t* part = w.part;
  const NmDev* insts = t->insts.as<NmDev>();
  const int64_t* term0 = (const int64_t*)(B + t->o_term0);
  const int64_t* blk0 = (const int64_t*)(B + t->o_blk0);
  if (!have_v)
    NM_TRY(hipMemcpyAsync(t->ck.p, in.ck->data(), sizeof(double) * in.ck->size(), hipMemcpyHostToDevice, st));
  std::vector<int> hf[2];
  for (int s = have_v ? 1 : 0; s < nset; ++s) {
    const double* G = s ? mu : V;
    hipLaunchKernelGGL(k_nm_zero, dim3(8), dim3(256), 0, st, flag[s], t->npairs + 1);
    hipLaunchKernelGGL(k_nm_cut1, dim3(t->ncut1), dim3(64), 0, st, (const Cut*)(B + t->o_cut1), G, c1[s]);
    if (t->ncut2)
      hipLaunchKernelGGL(k_nm_cut2, dim3(t->ncut2), dim3(64), 0, st, (const Cut*)(B + t->o_cut2), G, c1[s],
                         f2[s], flag[s]);
    hipLaunchKernelGGL(k_nm_verify, dim3((unsigned)std::min<int64_t>(t->nterms, 16384)), dim3(256), 0, st,
                       insts, term0, ni, t->nterms, in.d_terms, G, c1[s], f2[s], flag[s],
                       flag[s] + t->npairs);
    hipLaunchKernelGGL(k_nm_g1, dim3(t->ng1), dim3(256), 0, st, insts, (const int32_t*)(B + t->o_g1work),
                       in.d_mats, c1[s], g1[s], s ? G1_GRID : G1_GRID | G1_KIN);
    hf[s].resize(t->npairs + 1);
    NM_TRY(hipMemcpyAsync(hf[s].data(), flag[s], sizeof(int) * hf[s].size(), hipMemcpyDeviceToHost, st));
  }
  if (have_v) hf[0] = t->v_flags;
  NM_TRY(hipGetLastError());
  NM_TRY(hipStreamSynchronize(st));
  for (int s = 0; s < nset; ++s)
    if (hf[s][t->npairs]) return SG4_OK;   // not a sum of one- and two-mode functions
  // two-mode matrices of the nonzero pairs
  std::vector<EWork> ew[2];
  std::vector<int64_t> eoff[2];
  int64_t ne[2] = {0, 0};
  int Smax = 0;
  for (int s = 0; s < nset; ++s) {
    eoff[s].assign((size_t)t->npairs * eld, -1);
    for (int g = 0; g < t->npairs; ++g) {
      if (!hf[s][g]) continue;
      const int x = t->pair_inst[g];
      for (int l = 0; l <= t->dev[x].L; ++l) {
        const int S = t->pair_s2n[(size_t)g * eld + l];
        eoff[s][(size_t)g * eld + l] = ne[s];
        ew[s].push_back(EWork{x, g - t->dev[x].pair0, l, 0, ne[s]});
        ne[s] += (int64_t)S * S;
        Smax = std::max(Smax, S);
      }
      if (ne[s] > MAX_E) return SG4_OK;
    }
  }
  std::vector<int32_t> nz, nzoff(1, 0), adj, adjoff((size_t)ni * 33 + 33, 0);
  for (int x = 0; x < ni; ++x) {
    const NmDev& d = t->dev[x];
    std::vector<std::vector<int32_t>> by(d.D);
    for (int a = 0, p = 0; a < d.D; ++a)
      for (int b = a + 1; b < d.D; ++b, ++p)
        if (hf[0][d.pair0 + p] || (mu && hf[1][d.pair0 + p])) {
          nz.push_back(p);
          by[a].push_back(p);
          by[b].push_back(p);
        }
    nzoff.push_back((int32_t)nz.size());
    for (int k = 0; k < d.D; ++k) {
      adjoff[(size_t)x * 33 + k] = (int32_t)adj.size();
      adj.insert(adj.end(), by[k].begin(), by[k].end());
      adjoff[(size_t)x * 33 + k + 1] = (int32_t)adj.size();
    }
  }
  // column lists of the pairs that are nonzero in V or mu
  std::vector<EWork> uw;
  std::vector<int64_t> loff((size_t)t->npairs * eld, 0), croff((size_t)t->npairs * eld, 0);
  int64_t nl = 0, nr = 0;
  for (int g = 0; g < t->npairs; ++g) {
    if (!hf[0][g] && !(mu && hf[1][g])) continue;
    const int x = t->pair_inst[g];
    for (int l = 0; l <= t->dev[x].L; ++l) {
      const int S = t->pair_s2n[(size_t)g * eld + l];
      loff[(size_t)g * eld + l] = nl;
      croff[(size_t)g * eld + l] = nr;
      uw.push_back(EWork{x, g - t->dev[x].pair0, l, 0, 0});
      nl += (int64_t)S * S;
      nr += S;
    }
  }
  Blob lb;
  size_t o_ew[2], o_eoff[2];
  for (int s = 0; s < nset; ++s) { o_ew[s] = lb.add(ew[s]); o_eoff[s] = lb.add(eoff[s]); }
  const size_t o_nz = lb.add(nz), o_nzoff = lb.add(nzoff), o_adj = lb.add(adj), o_adjoff = lb.add(adjoff),
               o_uw = lb.add(uw), o_loff = lb.add(loff), o_croff = lb.add(croff);
  if ((rc = upload(lb, t->lists, st))) return rc == SG4_ERR_OOM ? SG4_OK : rc;
  if (ensure(t->e_v, 8 * ne[0]) || (mu && ensure(t->e_mu, 8 * ne[1])) ||
      ensure(t->elist, up(2 * nl) + 4 * nr))
    return SG4_OK;
  char* LB = t->lists.as<char>();
  DevBuf* eb[2] = {&t->e_v, &t->e_mu};
  NmSet set[2] = {};
  for (int s = 0; s < nset; ++s) {
    set[s] = NmSet{c1[s], g1[s], eb[s]->as<double>(), (const int64_t*)(LB + o_eoff[s])};
    if (!ew[s].empty() && (s || !have_v))
      hipLaunchKernelGGL(k_nm_e2, dim3((unsigned)ew[s].size(), (unsigned)std::min(256, (Smax * Smax + 31) / 32)),
                         dim3(256), 0, st, insts, (const EWork*)(LB + o_ew[s]), in.d_mats, c1[s], f2[s],
                         eb[s]->as<double>());
  }
  const NmPairs pr{(const int32_t*)(LB + o_nz), (const int32_t*)(LB + o_nzoff), (const int32_t*)(LB + o_adj),
                   (const int32_t*)(LB + o_adjoff), (const int64_t*)(LB + o_loff),
                   (const int64_t*)(LB + o_croff), t->elist.as<uint16_t>(),
                   (int32_t*)(t->elist.as<char>() + up(2 * nl)), eld};
  if (!uw.empty())
    hipLaunchKernelGGL(k_nm_elist, dim3((unsigned)uw.size(), (unsigned)((Smax + 63) / 64)), dim3(64), 0, st, insts,
                       (const EWork*)(LB + o_uw), set[0], set[1], pr);
  const dim3 rg((unsigned)t->nblk);
  const size_t rl = (size_t)t->Dmax * RT * 7;
  if (mu)
    hipLaunchKernelGGL((k_nm_rows<false, true>), rg, dim3(256), rl, st, insts, blk0, ni, set[0], set[1], pr,
                       t->Dmax, cnt, nullptr, nullptr, nullptr, nullptr);
  else
    hipLaunchKernelGGL((k_nm_rows<false, false>), rg, dim3(256), rl, st, insts, blk0, ni, set[0], set[1], pr,
                       t->Dmax, cnt, nullptr, nullptr, nullptr, nullptr);
  int64_t nnz = 0, longest = 0;
  if ((rc = scan_rows(w, rows, st, &nnz, &longest))) return rc;
  if (nnz > NNZ_SMALL && nnz > NNZ_PER_POINT * (double)in.sum_nq) return SG4_OK;
  if (ensure(m.ptr, 8 * (rows + 1)) || ensure(m.col, 4 * nnz) || ensure(m.val, 8 * nnz) ||
      (mu && (ensure(m.val_mu, 8 * nnz) || ensure(m.val_f, 8 * nnz))))
    return SG4_OK;
  hipLaunchKernelGGL(k_nm_ptr, dim3(w.npart), dim3(1024), 0, st, cnt, rows, part, m.ptr.as<int64_t>());
  if (mu)
    hipLaunchKernelGGL((k_nm_rows<true, true>), rg, dim3(256), rl, st, insts, blk0, ni, set[0], set[1], pr,
                       t->Dmax, cnt, m.ptr.as<int64_t>(), m.col.as<int32_t>(), m.val.as<double>(),
                       m.val_mu.as<double>());
  else
    hipLaunchKernelGGL((k_nm_rows<true, false>), rg, dim3(256), rl, st, insts, blk0, ni, set[0], set[1], pr,
                       t->Dmax, cnt, m.ptr.as<int64_t>(), m.col.as<int32_t>(), m.val.as<double>(), nullptr);
  NM_TRY(hipGetLastError());
  m.rows = rows;
  m.nnz = nnz;
  m.longest = longest;
  m.valid = true;
  t->v_ready = true;
  t->v_flags = hf[0];
  return SG4_OK;
}

namespace {
bool long_rows(const NModeMat& m) { return m.longest > LONG_ROW && m.rows <= ORDER_FEW; }

template <bool COLS, bool IN_COLS>
int spmm(const NModeMat& m, int W, int nvec, const double* psi, double* hpsi, hipStream_t st,
         const double* val, float* psi32 = nullptr) {
  const int64_t* ptr = m.ptr.as<int64_t>();
  const int32_t* col = m.col.as<int32_t>();
#define SG4_SPMM(NV, SL)                                                                              \
  hipLaunchKernelGGL((k_nm_spmm<NV, SL, COLS, IN_COLS>), grid_xz((m.rows * NV * SL + 255) / 256, 1),           \
                     dim3(256), 0, st, ptr, col, val, psi, hpsi, m.rows, nvec, psi32)
#define SG4_PAIRS(NC, PV, SL, SU, WIDE)                                                                \
  hipLaunchKernelGGL((k_nm_spmm_pairs<NC, PV, SL, SU, COLS, WIDE>),                                    \
                     grid_xz((m.rows * NC * SL + 255) / 256, WIDE ? W / (2 * NC * PV) : 1),            \
                     dim3(256), 0, st, ptr, col, val, psi, hpsi, m.rows, nvec, psi32)
  if constexpr (IN_COLS) {
    switch (W) {
      case 1: SG4_SPMM(1, 8); break;
      case 2: SG4_SPMM(2, 4); break;
      case 4: SG4_SPMM(4, 4); break;
      case 8: SG4_SPMM(8, 1); break;
      case 16: SG4_SPMM(16, 1); break;
      default: return 1;
    }
  } else {
    const bool lg = long_rows(m);
    switch (W) {
      case 1: SG4_SPMM(1, 8); break;
      case 2: SG4_PAIRS(1, 1, 8, 2, false); break;
      case 4: SG4_PAIRS(1, 2, 8, 2, false); break;
      case 8:
        if (lg) SG4_PAIRS(2, 2, 32, 2, false);
        else SG4_PAIRS(2, 2, 8, 2, false);
        break;
      case 16:
        if (lg) SG4_PAIRS(4, 2, 16, 2, false);
        else SG4_PAIRS(4, 2, 4, 2, false);
        break;
      default:
        if constexpr (COLS) return 1;
        else if (W % 16 == 0 && lg) SG4_PAIRS(4, 2, 16, 2, true);
        else if (W % 16 == 0) SG4_PAIRS(4, 2, 4, 2, true);
        else if (W % 8 == 0 && lg) SG4_PAIRS(2, 2, 32, 2, true);
        else if (W % 8 == 0) SG4_PAIRS(2, 2, 8, 2, true);
        else return 1;
    }
  }
#undef SG4_PAIRS
#undef SG4_SPMM
  NM_TRY(hipGetLastError());
  return SG4_OK;
}
}  // namespace

int nmode_apply(const NModeMat& m, int nvec, const double* psi, double* hpsi, hipStream_t st, const double* val,
                float* psi32) {
  if (!val) val = m.val.as<double>();
  const int rc = spmm<false, false>(m, nvec, nvec, psi, hpsi, st, val, psi32);
  if (rc <= 0) return rc;
  const int sl = long_rows(m) ? 16 : 1;
  hipLaunchKernelGGL(sl == 1 ? k_nm_spmm_any<1> : k_nm_spmm_any<16>,
                     dim3((unsigned)std::min<int64_t>((m.rows * nvec * sl + 255) / 256, (int64_t)1 << 20)), dim3(256), 0,
                     st, m.ptr.as<int64_t>(), m.col.as<int32_t>(), val, psi, hpsi, m.rows, nvec, psi32);
  NM_TRY(hipGetLastError());
  return SG4_OK;
}

bool nmode_cols_direct(const NModeMat& m, int W) {
  return W <= 16 && (W & (W - 1)) == 0 && m.nnz * W * W <= COLS_DIRECT && (W < 8 || !long_rows(m));
}

int nmode_apply_cols(const NModeMat& m, int W, int nvec, const double* psi, double* hpsi, hipStream_t st) {
  return spmm<true, true>(m, W, nvec, psi, hpsi, st, m.val.as<double>());
}

int nmode_apply_to_cols(const NModeMat& m, int W, int nvec, const double* psi, double* hpsi, hipStream_t st) {
  return spmm<true, false>(m, W, nvec, psi, hpsi, st, m.val.as<double>());
}

bool nmode_order_width(int ncol) { return ncol == 2 || ncol == 4 || ncol == 8 || ncol == 16; }

int nmode_order(const NModeMat& m, const NModeOrder& a, bool tangent, hipStream_t st) {
  const int64_t* ptr = m.ptr.as<int64_t>();
  const int32_t* col = m.col.as<int32_t>();
  const double* mu = m.val_mu.as<double>();
  auto grid = [&](int w) {
    return dim3((unsigned)std::min<int64_t>((m.rows * w + 255) / 256, (int64_t)1 << 20));
  };
  const int nc = (tangent ? 4 : 2) * a.ns;
  const bool few = m.rows <= ORDER_FEW;
#define SG4_ORDER(NC, SL, TAN) \
  hipLaunchKernelGGL((k_nm_order<NC, SL, TAN>), grid(NC * SL), dim3(256), 0, st, ptr, col, mu, a, m.rows)
  if (long_rows(m)) {   // a wave per row
    if (tangent) {
      if (nc == 4) SG4_ORDER(2, 32, true);
      else if (nc == 8) SG4_ORDER(4, 16, true);
      else SG4_ORDER(8, 8, true);
    } else {
      if (nc == 2) SG4_ORDER(1, 64, false);
      else if (nc == 4) SG4_ORDER(2, 32, false);
      else if (nc == 8) SG4_ORDER(4, 16, false);
      else SG4_ORDER(8, 8, false);
    }
  } else if (tangent) {
    if (nc == 4 && few) SG4_ORDER(2, 8, true);
    else if (nc == 4) SG4_ORDER(2, 4, true);
    else if (nc == 8) SG4_ORDER(4, 4, true);
    else SG4_ORDER(8, 2, true);
  } else {
    if (nc == 2 && few) SG4_ORDER(1, 8, false);
    else if (nc == 2) SG4_ORDER(1, 4, false);
    else if (nc == 4 && few) SG4_ORDER(2, 8, false);
    else if (nc == 4) SG4_ORDER(2, 4, false);
    else if (nc == 8) SG4_ORDER(4, 4, false);
    else SG4_ORDER(8, 2, false);
  }
#undef SG4_ORDER
  NM_TRY(hipGetLastError());
  return SG4_OK;
}

int nmode_set_field(const NModeMat& m, double eps, hipStream_t st) {
  hipLaunchKernelGGL(k_nm_field, dim3((unsigned)std::min<int64_t>((m.nnz + 255) / 256, 65536)), dim3(256), 0, st,
                     m.val.as<double>(), m.val_mu.as<double>(), eps, m.val_f.as<double>(), m.nnz);
  NM_TRY(hipGetLastError());
  return SG4_OK;
}

}  // namespace sg4
