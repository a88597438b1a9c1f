// Dense products of the device block Davidson over packed vectors: blocks of
// a few to ~100 rows of length n = nb_ba (1.26 M at 10D L=8), so every
// product is a pass over HBM with a tiny output.
//
//   gram:    C (m x q) = A B^T, A: m rows, B: q rows (stride lda, ldb), the
//            inner dimension n long, on the FP64 matrix cores: a wave keeps up
//            to 4 x 2 tiles of 16 x 16 and takes 16 columns at a time straight
//            from memory into operand registers (no LDS, no barrier in the
//            loop); the workgroups' partials go to a work array and a second
//            kernel adds them, one wave per output, in a fixed order
//            (deterministic, no atomics).
//   combine: Y (k x n) = beta Y + U X, U (k x d) small, X: d rows: 32 columns
//            per wave and step, X straight into operand registers, U in LDS in
//            operand order; one column per thread with U by scalar loads where U
//            exceeds 64 KiB and where the matrix cores have little to do.
// Bound by HBM for the Davidson's shapes.  At 10D L=8 (n = 1.26 M), us, before
// (LDS tiles and 4 x 4 register blocks; one column per thread with U from
// scalar loads) -> now, and the floor at the copy rate of 4.9 TB/s: gram 8 x 8
// 65 -> 34 (33), 20 x 20 191 -> 86 (82), 60 x 16 305 -> 165 (156), 100 x 16 465 ->
// 283 (238), 84 x 84 1825 -> 1111 (library split-K product 300-600); combine 16 x 48
// 158 -> 149 (131), 20 x 60 244 -> 193 (164), 36 x 84 703 -> 352 (246), 64 x 64 1035
// -> 367 (262).  1024 or 2048 gram workgroups: 187, 209 for
// 60 x 16 (more partials).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "sg4_internal.h"

namespace sg4 {
namespace {

constexpr int GMAX = 124;      // rows of A or B
constexpr int GBLK = 512;      // 4 x 4 output blocks at most
constexpr int GNB = 2048;      // partials per output that the work array is sized for
constexpr int GWGS = 512;      // workgroups of a gram (per group of tiles)
// Workgroups of a combine: with U of more than 16 rows 2048 that stay and load it
// once (n = 1.26 M, 36 x 84 352 us, one per tile 468), with fewer rows one per tile
// of columns (8 x 8 of the same, beta = 1, 47 -> 42, 16 x 16 120 -> 111).
constexpr int64_t CWG = 2048, CWG16 = 65535;
// A combine with one thread per column where the matrix cores have little to do:
// few rows of X, which the writes of whole Y rows bound (n = 1.26 M, us, matrix
// cores / threads: 16 x 4 beta 1 64 / 58, 32 x 8 146 / 106, 36 x 8 159 / 120), and
// few rows of Y beyond the caches (1 x 60 115 / 107, 4 x 124 253 / 233; 4 x 60 of
// 400 k 35 / 39) or one or two of them (1 x 124 of 100 k 26 / 22).
constexpr int64_t THREADS_N = 1 << 19, THREADS_X = 48000000;
constexpr int THREADS_D = 8, THREADS_K = 4, THREADS_K2 = 2, THREADS_D2 = 48;
constexpr int CMAXU = 8192;    // entries of U (k d) at most
constexpr int CK = 16;         // outputs of the scalar combine per pass over X (k <= 16)
constexpr int CKW = 48;        // the same for wider k (k > 48: several passes)

typedef double f64x4 __attribute__((ext_vector_type(4)));
struct __attribute__((packed, aligned(8))) D4 { double v[4]; };   // 32 bytes at 8-byte alignment

// Partial sums of C = A B^T over the columns of this workgroup: TA x TB tiles
// of 16 x 16 on v_mfma_f64_16x16x4.  A wave takes 16 columns at a time; lane l
// holds columns 4 (l/16) .. +3 of row l%16 of every tile (a row's 16 columns
// are one 128-byte line), and product s of the four uses column 4 (l/16) + s
// of both operands, so nothing goes through LDS.  blockIdx.y: group of tiles;
// swap: A and B are exchanged (the wider one in the TA tiles).
template <int TA, int TB>
__global__ __launch_bounds__(256) void k_gram_part(int m, int q, int64_t n, const double* __restrict__ A,
                                                   int64_t lda, const double* __restrict__ B, int64_t ldb,
                                                   int swap, double* __restrict__ part) {
  __shared__ double red[4][256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, kq = lane >> 4;
  const int gb = (q + 16 * TB - 1) / (16 * TB);
  const int i0 = (blockIdx.y / gb) * 16 * TA, j0 = (blockIdx.y % gb) * 16 * TB;
  const double* pa[TA];
  const double* pb[TB];
#pragma unroll
  for (int t = 0; t < TA; ++t) pa[t] = A + (int64_t)min(i0 + 16 * t + r, m - 1) * lda + 4 * kq;
#pragma unroll
  for (int t = 0; t < TB; ++t) pb[t] = B + (int64_t)min(j0 + 16 * t + r, q - 1) * ldb + 4 * kq;
  f64x4 acc[TA][TB];
#pragma unroll
  for (int x = 0; x < TA; ++x)
#pragma unroll
    for (int y = 0; y < TB; ++y) acc[x][y] = f64x4{0.0, 0.0, 0.0, 0.0};
  auto products = [&](const D4 (&a)[TA], const D4 (&b)[TB]) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int x = 0; x < TA; ++x)
#pragma unroll
        for (int y = 0; y < TB; ++y)
          acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[x].v[s], b[y].v[s], acc[x][y], 0, 0, 0);
  };
  const int64_t full = n / 16, step = (int64_t)gridDim.x * 4;
  int64_t t = (int64_t)blockIdx.x * 4 + wave;
  for (; t < full; t += step) {
    D4 a[TA], b[TB];
#pragma unroll
    for (int x = 0; x < TA; ++x) a[x] = *(const D4*)(pa[x] + 16 * t);
#pragma unroll
    for (int y = 0; y < TB; ++y) b[y] = *(const D4*)(pb[y] + 16 * t);
    products(a, b);
  }
  if (t == full && 16 * full < n) {   // the columns beyond the last whole block, the others zero
    D4 a[TA], b[TB];
#pragma unroll
    for (int s = 0; s < 4; ++s) {       // without a branch, so that the loads go out together
      const int64_t o = min(16 * full + s, n - 1 - 4 * kq);
#pragma unroll
      for (int x = 0; x < TA; ++x) a[x].v[s] = pa[x][o];
#pragma unroll
      for (int y = 0; y < TB; ++y) b[y].v[s] = pb[y][o];
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const bool in = 16 * full + 4 * kq + s < n;
#pragma unroll
      for (int x = 0; x < TA; ++x) a[x].v[s] = in ? a[x].v[s] : 0.0;
#pragma unroll
      for (int y = 0; y < TB; ++y) b[y].v[s] = in ? b[y].v[s] : 0.0;
    }
    products(a, b);
  }
  // the four waves' sums in wave order; output (i, j) of a tile: value i / 4 of
  // lane 16 (i % 4) + j
  const int64_t nb = gridDim.x;
#pragma unroll
  for (int x = 0; x < TA; ++x)
#pragma unroll
    for (int y = 0; y < TB; ++y) {
      __syncthreads();
#pragma unroll
      for (int u = 0; u < 4; ++u) red[wave][(4 * u + kq) * 16 + r] = acc[x][y][u];
      __syncthreads();
      const int i = i0 + 16 * x + threadIdx.x / 16, j = j0 + 16 * y + threadIdx.x % 16;
      if (i < m && j < q) {
        const double s = (red[0][threadIdx.x] + red[1][threadIdx.x]) + (red[2][threadIdx.x] + red[3][threadIdx.x]);
        part[(swap ? (int64_t)j * m + i : (int64_t)i * q + j) * nb + blockIdx.x] = s;
      }
    }
}

// C[e] = sum over the nb workgroup partials of output e: one wave per output,
// lane l adding partials l, l + 64, ..., then a fixed shuffle tree (the same
// order on every call)
__global__ __launch_bounds__(256) void k_gram_sum(int mq, int nb, const double* __restrict__ part,
                                                  double* __restrict__ C) {
  const int lane = threadIdx.x & 63;
  const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (e >= mq) return;                          // uniform over the wave
  double s = 0.0;
  for (int b = lane; b < nb; b += 64) s += part[(int64_t)e * nb + b];
  for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
  if (lane == 0) C[e] = s;
}

// Y (16 RT rows from i0) = beta Y + U X for 32 columns per wave and step, on
// v_mfma_f64_16x16x4: lane l holds columns 2 (l%16), +1 of row 4 s + l/16 of X
// (256 bytes of a row per wave and load) for two column tiles, U sits in LDS in
// operand order, zero beyond k and d.
template <int RT>
__global__ __launch_bounds__(256) void k_combine_mfma(int k, int d, int64_t n, const double* __restrict__ U,
                                                      const double* __restrict__ X, int64_t ldx, double beta,
                                                      double* __restrict__ Y, int64_t ldy) {
  extern __shared__ double ul[];   // [(s RT + rt) 64 + lane]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, kq = lane >> 4;
  const int ks = (d + 3) >> 2, i0 = blockIdx.y * 16 * RT;
  for (int e = threadIdx.x; e < ks * RT * 64; e += 256) {
    const int l = e & 63, st = e >> 6, rt = st % RT, s = st / RT;
    const int i = i0 + 16 * rt + (l & 15), j = 4 * s + (l >> 4);
    ul[e] = (i < k && j < d) ? U[(int64_t)i * d + j] : 0.0;
  }
  __syncthreads();
  const int64_t nblk = (n + 31) / 32;
  for (int64_t t = (int64_t)blockIdx.x * 4 + wave; t < nblk; t += (int64_t)gridDim.x * 4) {
    const int64_t c = 32 * t + 2 * r;
    const bool in0 = c < n, in1 = c + 1 < n;
    f64x4 acc[RT][2];
#pragma unroll
    for (int x = 0; x < RT; ++x) acc[x][0] = acc[x][1] = f64x4{0.0, 0.0, 0.0, 0.0};
    auto product = [&](int s, double x0, double x1) {
#pragma unroll
      for (int x = 0; x < RT; ++x) {
        const double u = ul[(s * RT + x) * 64 + lane];
        acc[x][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(u, x0, acc[x][0], 0, 0, 0);
        acc[x][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(u, x1, acc[x][1], 0, 0, 0);
      }
    };
    if (32 * t + 32 <= n) {   // uniform over the wave: a matrix instruction takes all lanes
      const double* p = X + (int64_t)kq * ldx + c;
      int s = 0;
      for (; 4 * s + 16 <= d; s += 4) {     // four steps' loads in flight
        double a[4], b[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const double* w = p + (int64_t)4 * (s + u) * ldx;
          a[u] = w[0];
          b[u] = w[1];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) product(s + u, a[u], b[u]);
      }
      for (; s < ks; ++s) {
        const bool row = 4 * s + kq < d;
        const double* w = p + (int64_t)4 * s * ldx;
        product(s, row ? w[0] : 0.0, row ? w[1] : 0.0);
      }
    } else {                                // the last columns
      for (int s = 0; s < ks; ++s) {
        const bool row = 4 * s + kq < d;
        const double* w = X + (int64_t)(4 * s + kq) * ldx + c;
        product(s, row && in0 ? w[0] : 0.0, row && in1 ? w[1] : 0.0);
      }
    }
#pragma unroll
    for (int x = 0; x < RT; ++x)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = i0 + 16 * x + 4 * u + kq;
        if (i >= k) continue;
        double* y = Y + (int64_t)i * ldy + c;
        if (in0) y[0] = beta == 0.0 ? acc[x][0][u] : fma(beta, y[0], acc[x][0][u]);
        if (in1) y[1] = beta == 0.0 ? acc[x][1][u] : fma(beta, y[1], acc[x][1][u]);
      }
  }
}

// Y rows i0..i0+CK-1 for the columns of this thread; U entries are read
// straight from global memory at wave-uniform addresses (scalar loads, one
// SGPR operand per FMA), X once per pass.
template <int CK>
__global__ __launch_bounds__(256) void k_combine(int k, int d, int64_t n, const double* __restrict__ U,
                                                 const double* __restrict__ X, int64_t ldx, double beta,
                                                 double* __restrict__ Y, int64_t ldy) {
  for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < n; r += (int64_t)gridDim.x * blockDim.x) {
    for (int i0 = 0; i0 < k; i0 += CK) {
      double acc[CK];
#pragma unroll
      for (int u = 0; u < CK; ++u) acc[u] = 0.0;
      int j = 0;
      for (; j + 4 <= d; j += 4) {               // four loads in flight
        double x[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) x[t] = X[(int64_t)(j + t) * ldx + r];
#pragma unroll
        for (int u = 0; u < CK; ++u)
          if (i0 + u < k) {
            const double* ur = U + (int64_t)(i0 + u) * d + j;
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[u] = fma(ur[t], x[t], acc[u]);
          }
      }
      for (; j < d; ++j) {
        const double x = X[(int64_t)j * ldx + r];
#pragma unroll
        for (int u = 0; u < CK; ++u)
          if (i0 + u < k) acc[u] = fma(U[(int64_t)(i0 + u) * d + j], x, acc[u]);
      }
#pragma unroll
      for (int u = 0; u < CK; ++u)
        if (i0 + u < k) {
          double* y = Y + (int64_t)(i0 + u) * ldy + r;
          *y = (beta == 0.0) ? acc[u] : fma(beta, *y, acc[u]);
        }
    }
  }
}

#define BK_TRY(expr)                                                              \
  do {                                                                            \
    hipError_t _e = (expr);                                                       \
    if (_e != hipSuccess) {                                                       \
      set_error(std::string("HIP error: ") + hipGetErrorString(_e) + " at " #expr); \
      return SG4_ERR_HIP;                                                         \
    }                                                                             \
  } while (0)

}  // namespace
}  // namespace sg4

using namespace sg4;

extern "C" {

int sg4_block_gram_work(int32_t m, int32_t q, int64_t* nwork) {
  if (!nwork) { set_error("null argument"); return SG4_ERR_ARG; }
  if (m < 1 || q < 1 || m > GMAX || q > GMAX || ((m + 3) / 4) * ((q + 3) / 4) > GBLK) {
    set_error("sg4_block_gram: m, q <= 124 with ceil(m/4) ceil(q/4) <= 512 expected");
    return SG4_ERR_ARG;
  }
  *nwork = (int64_t)GNB * m * q;
  return SG4_OK;
}

int sg4_block_gram(sg4_plan* p, int32_t m, int32_t q, int64_t n, const double* A, int64_t lda,
                   const double* B, int64_t ldb, double* C, double* work, int64_t nwork) {
  if (!p || !A || !B || !C || !work) { set_error("null argument"); return SG4_ERR_ARG; }
  int64_t need;
  int rc;
  if ((rc = sg4_block_gram_work(m, q, &need))) return rc;
  if (n < 1 || lda < n || ldb < n) { set_error("sg4_block_gram: bad n or row strides"); return SG4_ERR_ARG; }
  if (nwork < (int64_t)m * q) { set_error("sg4_block_gram: work array too small"); return SG4_ERR_ARG; }
  if ((rc = device_block(p, A, "A")) || (rc = device_block(p, B, "B")) ||
      (rc = device_block(p, C, "C")) || (rc = device_block(p, work, "work")))
    return rc;
  const hipStream_t st = (hipStream_t)plan_stream(p);
  const int64_t nwave = (n + 63) / 64;
  const int nb = (int)std::max<int64_t>(1, std::min<int64_t>({(int64_t)GWGS, (nwave + 3) / 4, nwork / ((int64_t)m * q)}));
  const bool swap = q > m;                     // the wider block in the row tiles
  const int M = swap ? q : m, Q = swap ? m : q;
  const double *a = swap ? B : A, *b = swap ? A : B;
  const int64_t la = swap ? ldb : lda, lb = swap ? lda : ldb;
  const int ta = M <= 16 ? 1 : M <= 32 ? 2 : 4, tb = Q <= 16 ? 1 : 2;
  const dim3 grid((unsigned)nb, (unsigned)(((M + 16 * ta - 1) / (16 * ta)) * ((Q + 16 * tb - 1) / (16 * tb))));
#define SG4_GRAM(TA, TB) \
  hipLaunchKernelGGL((k_gram_part<TA, TB>), grid, dim3(256), 0, st, M, Q, n, a, la, b, lb, swap, work)
  if (tb == 1) {
    if (ta == 1) SG4_GRAM(1, 1); else if (ta == 2) SG4_GRAM(2, 1); else SG4_GRAM(4, 1);
  } else {
    if (ta == 2) SG4_GRAM(2, 2); else SG4_GRAM(4, 2);
  }
#undef SG4_GRAM
  BK_TRY(hipGetLastError());
  const int mq = m * q;
  hipLaunchKernelGGL(k_gram_sum, dim3((mq + 3) / 4), dim3(256), 0, st, mq, nb, work, C);
  BK_TRY(hipGetLastError());
  return SG4_OK;
}

int sg4_block_combine(sg4_plan* p, int32_t k, int32_t d, int64_t n, const double* U, const double* X,
                      int64_t ldx, double beta, double* Y, int64_t ldy) {
  if (!p || !U || !X || !Y) { set_error("null argument"); return SG4_ERR_ARG; }
  if (k < 1 || d < 1 || (int64_t)k * d > CMAXU || n < 1 || ldx < n || ldy < n) {
    set_error("sg4_block_combine: k d <= 8192, n >= 1 and row strides >= n expected");
    return SG4_ERR_ARG;
  }
  int rc;
  if ((rc = device_block(p, U, "U")) || (rc = device_block(p, X, "X")) || (rc = device_block(p, Y, "Y")))
    return rc;
  const char* xb = (const char*)X;
  const char* yb = (const char*)Y;
  const int64_t xe = 8 * ((int64_t)(d - 1) * ldx + n), ye = 8 * ((int64_t)(k - 1) * ldy + n);
  if (xb < yb + ye && yb < xb + xe) { set_error("sg4_block_combine: X and Y overlap"); return SG4_ERR_ARG; }
  const hipStream_t st = (hipStream_t)plan_stream(p);
  const int rt = k <= 16 ? 1 : k <= 32 ? 2 : 4;
  const size_t lds = sizeof(double) * 64 * rt * (size_t)((d + 3) / 4);
  const bool threads = (d <= THREADS_D && n >= THREADS_N) || (k <= THREADS_K && d * n > THREADS_X) ||
                       (k <= THREADS_K2 && d >= THREADS_D2);
  if (lds <= 64 * 1024 && !threads) {
    const dim3 grid((unsigned)std::min<int64_t>((n + 127) / 128, rt == 1 ? CWG16 : CWG), (unsigned)((k + 16 * rt - 1) / (16 * rt)));
    if (rt == 1) hipLaunchKernelGGL(k_combine_mfma<1>, grid, dim3(256), lds, st, k, d, n, U, X, ldx, beta, Y, ldy);
    else if (rt == 2) hipLaunchKernelGGL(k_combine_mfma<2>, grid, dim3(256), lds, st, k, d, n, U, X, ldx, beta, Y, ldy);
    else hipLaunchKernelGGL(k_combine_mfma<4>, grid, dim3(256), lds, st, k, d, n, U, X, ldx, beta, Y, ldy);
    BK_TRY(hipGetLastError());
    return SG4_OK;
  }
  const unsigned nb = (unsigned)std::min<int64_t>((n + 255) / 256, 65535);
  if (k <= CK)
    hipLaunchKernelGGL(k_combine<CK>, dim3(nb), dim3(256), 0, st, k, d, n, U, X, ldx, beta, Y, ldy);
  else
    hipLaunchKernelGGL(k_combine<CKW>, dim3(nb), dim3(256), 0, st, k, d, n, U, X, ldx, beta, Y, ldy);
  BK_TRY(hipGetLastError());
  return SG4_OK;
}

}  // extern "C"
