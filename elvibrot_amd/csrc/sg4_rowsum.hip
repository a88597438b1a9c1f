// Sum over the Smolyak terms, row by row (see sg4_rowsum.h).
//
// k_rs_add reads one place (nvec values) of the block per stored place of a row:
// random lines, bound by the rate of line fetches (10D L=8 x16: 31.5 M places of
// 64 B in FP32 ~0.65 ms, 128 B in FP64 ~0.9 ms).  Neighbouring segments share
// lines when their rows are neighbours in the terms' grids and list their
// places in the same order, so rows are numbered by first appearance in the
// map and their places sorted: split precision 8D L=6 x2 56 us (rows in packed
// order, places as the atomics of the fill left them), 39 (places sorted), 34.
//
// The map is inverted on the device, one number (the totals) read back: 9D L=7
// 1.1 ms of kernels, 10D L=8 6.7 (counts and fill 4.7: atomics on the rows that
// most terms hold; sort 1.1).  With the rows' order and segments made on the host
// the whole took 1.9 and 16 ms.
#include "sg4_rowsum.h"

#include <algorithm>
#include <map>

namespace sg4 {

namespace {

constexpr int RS_SEG = 64;                       // places per segment (one per lane of k_rs_sort)
constexpr int RS_LOADS = 8;                      // places in flight per lane
constexpr int RS_LANES = 4;                      // log2 of the lanes per segment, at least
constexpr int RS_BATCH = 8;                      // fill launches
constexpr int SCAN = 1024;                       // items per workgroup of a scan
constexpr size_t RS_MAX_BYTES = size_t(16) << 30; // results held per plan
constexpr size_t RS_MAX_BLOCKS = 8;
constexpr int RS_WEIGHTS = 256;                 // distinct term weights
// A segment's indices run up to RS_LOADS times its lanes beyond its end, in 32
// bits; a launch with a lane per place of every segment takes 2^32 threads.
constexpr int64_t RS_PLACES = INT32_MAX - 4096, RS_SEGMENTS = (int64_t(1) << 32) / RS_SEG - 4;
constexpr uint32_t RS_MULTI = 0x80000000u;

#define RS_TRY(x)                                     \
  do {                                                \
    const hipError_t e_ = (x);                        \
    if (e_ != hipSuccess) {                           \
      set_error(std::string("HIP: ") + hipGetErrorString(e_)); \
      return SG4_ERR_HIP;                             \
    }                                                 \
  } while (0)

__global__ __launch_bounds__(256) void k_rs_init(int32_t* cnt, int32_t* first, int32_t* order, int64_t n) {
  for (int64_t i = blockIdx.x * 256LL + threadIdx.x; i < n; i += gridDim.x * 256LL) {
    cnt[i] = 0;
    first[i] = INT32_MAX;
    order[i] = -1;
  }
}

// places per row and the row's first place
__global__ __launch_bounds__(256) void k_rs_count(const int32_t* map, int64_t n, int32_t* cnt, int32_t* first) {
  for (int64_t i = blockIdx.x * 256LL + threadIdx.x; i < n; i += gridDim.x * 256LL) {
    const int m = map[i];
    if (m < 0) continue;
    atomicAdd(&cnt[m], 1);
    if (first[m] > i) atomicMin(&first[m], (int32_t)i);
  }
}

// the rows that appear first in term t: their number (FILL: the rows, in the
// order of their places, from base[t] on)
template <bool FILL>
__global__ __launch_bounds__(256) void k_rs_first(const int32_t* map, const int32_t* first, const TermDev* terms,
                                                  int64_t nterms, int32_t* num, const int32_t* base, int32_t* rows) {
  __shared__ int s[256];
  for (int64_t t = blockIdx.x; t < nterms; t += gridDim.x) {
    const int64_t b = terms[t].boff;
    const int n = terms[t].nb;
    int done = 0;
    for (int p0 = 0; p0 < n; p0 += 256) {
      const int p = p0 + threadIdx.x;
      const int m = p < n ? map[b + p] : -1;
      const int x = m >= 0 && first[m] == (int32_t)(b + p);
      s[threadIdx.x] = x;
      __syncthreads();
      for (int o = 1; o < 256; o <<= 1) {
        const int y = (int)threadIdx.x >= o ? s[threadIdx.x - o] : 0;
        __syncthreads();
        s[threadIdx.x] += y;
        __syncthreads();
      }
      if (FILL && x) rows[base[t] + done + s[threadIdx.x] - 1] = m;
      done += s[255];
      __syncthreads();
    }
    if (!FILL && threadIdx.x == 0) num[t] = done;
  }
}

// What a scan adds up: the rows that first appear in term i, or (order) the
// places of the row that is i-th in the order and, in the upper half, its segments.
__device__ __forceinline__ uint64_t scan_item(const int32_t* num, const int32_t* order, int64_t i) {
  if (!order) return (uint32_t)num[i];
  const int r = order[i];
  if (r < 0) return 0;                // rows that no term holds
  const uint32_t n = (uint32_t)num[r];
  return (uint64_t)((n + RS_SEG - 1) / RS_SEG) << 32 | n;
}

// inclusive scan over the workgroup (SCAN threads); s: SCAN values of LDS
__device__ __forceinline__ uint64_t scan_block(uint64_t x, uint64_t* s) {
  s[threadIdx.x] = x;
  __syncthreads();
  for (int o = 1; o < SCAN; o <<= 1) {
    const uint64_t y = (int)threadIdx.x >= o ? s[threadIdx.x - o] : 0;
    __syncthreads();
    s[threadIdx.x] += y;
    __syncthreads();
  }
  return s[threadIdx.x];
}

// sums of SCAN items each, then their exclusive scan with the total behind it
__global__ __launch_bounds__(SCAN) void k_rs_sums(const int32_t* num, const int32_t* order, int64_t n, uint64_t* part) {
  __shared__ uint64_t s[SCAN];
  const int64_t i = (int64_t)blockIdx.x * SCAN + threadIdx.x;
  const uint64_t x = scan_block(i < n ? scan_item(num, order, i) : 0, s);
  if (threadIdx.x == SCAN - 1) part[blockIdx.x] = x;
}
__global__ __launch_bounds__(SCAN) void k_rs_scan(uint64_t* part, int np) {
  __shared__ uint64_t s[SCAN];
  uint64_t carry = 0;
  for (int b = 0; b < np; b += SCAN) {
    const int i = b + threadIdx.x;
    const uint64_t x = i < np ? part[i] : 0, y = scan_block(x, s);
    if (i < np) part[i] = carry + y - x;
    carry += s[SCAN - 1];
    __syncthreads();                  // s is written again
  }
  if (threadIdx.x == 0) part[np] = carry;
}

// the terms' first rows in the order (from num, in place)
__global__ __launch_bounds__(SCAN) void k_rs_base(int32_t* num, int64_t n, const uint64_t* part) {
  __shared__ uint64_t s[SCAN];
  const int64_t i = (int64_t)blockIdx.x * SCAN + threadIdx.x;
  const uint64_t x = i < n ? scan_item(num, nullptr, i) : 0, y = part[blockIdx.x] + scan_block(x, s) - x;
  if (i < n) num[i] = (int32_t)y;
}

// the segments of the rows in the order, and (in place of the counts) where a
// row's places start; nseg, places: the totals that seg was sized for
__global__ __launch_bounds__(SCAN) void k_rs_segs(int32_t* cnt, const int32_t* order, int64_t n, const uint64_t* part,
                                                  int32_t* seg, int64_t nseg, int32_t places) {
  __shared__ uint64_t s[SCAN];
  const int64_t i = (int64_t)blockIdx.x * SCAN + threadIdx.x;
  const uint64_t x = i < n ? scan_item(cnt, order, i) : 0, y = part[blockIdx.x] + scan_block(x, s) - x;
  if (i == 0) seg[nseg] = places;
  if (x == 0) return;
  const int r = order[i], at = (int)(uint32_t)y, num = (int)(uint32_t)x;
  int64_t k = (int64_t)(y >> 32);
  for (int o = 0; o < num; o += RS_SEG, ++k) {
    seg[k] = at + o;
    seg[nseg + 1 + k] = (int32_t)((uint32_t)r | (num > RS_SEG ? RS_MULTI : 0u));
  }
  cnt[r] = at;
}

// places of the terms [t0, t1); the launches go up the terms
__global__ __launch_bounds__(256) void k_rs_fill(const int32_t* map, const TermDev* terms, const uint8_t* tw,
                                                 int64_t t0, int64_t t1, int shift, int32_t* cursor, uint32_t* pos,
                                                 uint8_t* wi) {
  for (int64_t t = t0 + blockIdx.x; t < t1; t += gridDim.x) {
    const int64_t b = terms[t].boff;
    const int n = terms[t].nb;
    const uint32_t w = wi ? 0u : (uint32_t)((uint64_t)tw[t] << shift);
    for (int p = threadIdx.x; p < n; p += 256) {
      const int m = map[b + p];
      if (m < 0) continue;
      const int e = atomicAdd(&cursor[m], 1);
      pos[e] = (uint32_t)(b + p) | w;
      if (wi) wi[e] = tw[t];
    }
  }
}

// one wave per segment: its places in increasing order
__global__ __launch_bounds__(256) void k_rs_sort(uint32_t* pos, uint8_t* wi, const int32_t* seg, int64_t nseg,
                                                 uint32_t mask) {
  const int64_t s = (blockIdx.x * 256LL + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  if (s >= nseg) return;                // whole waves
  const int e = seg[s] + lane;
  const bool on = e < seg[s + 1];
  const uint32_t full = on ? pos[e] : 0u;
  uint32_t key = on ? (full & mask) : 0xffffffffu, val = full, w = on && wi ? wi[e] : 0u;
  for (int k = 2; k <= 64; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      const uint32_t ok = __shfl_xor(key, j), ov = __shfl_xor(val, j), ow = __shfl_xor(w, j);
      const bool low = ((lane & j) == 0) == ((lane & k) == 0);
      if (low ? ok < key : ok > key) { key = ok; val = ov; w = ow; }
    }
  if (on) pos[e] = val;
  if (on && wi) wi[e] = (uint8_t)w;
}

template <class T, int V> struct alignas(sizeof(T) * V) Pack { T x[V]; };

// 2^(lg + ls) lanes per segment: 2^lg hold V vectors each, the places are dealt
// to 2^ls slices, RS_LOADS places in flight per lane.  A row of one segment is
// added without an atomic.
template <class T, int V>
__global__ __launch_bounds__(256) void k_rs_add(const uint32_t* __restrict__ pos, const uint8_t* __restrict__ wi,
                                                const double* __restrict__ wtab,
                                                int nw, int shift, const int32_t* __restrict__ seg, int64_t nseg,
                                                const T* __restrict__ out, int nvec, int lg, int ls,
                                                double* hpsi) {
  __shared__ double wt[RS_WEIGHTS];
  if constexpr (sizeof(T) == 4) {
    if ((int)threadIdx.x < nw) wt[threadIdx.x] = wtab[threadIdx.x];
    __syncthreads();
  }
  const int64_t s0 = (blockIdx.x * 256LL + threadIdx.x) >> (lg + ls);
  const bool on = s0 < nseg;          // whole lane groups
  const int64_t s = on ? s0 : nseg - 1;
  const int sl = (int)(threadIdx.x >> lg) & ((1 << ls) - 1);
  const int v1 = ((int)(threadIdx.x & ((1 << lg) - 1)) + ((int)blockIdx.y << lg)) * V;
  const int v = v1 < nvec ? v1 : 0;
  const int e0 = seg[s], e1 = seg[s + 1];
  const uint32_t row = (uint32_t)seg[nseg + 1 + s];
  const uint32_t mask = (uint32_t)((1ull << shift) - 1);
  double acc[V];
#pragma unroll
  for (int j = 0; j < V; ++j) acc[j] = 0.0;
  for (int e = e0 + sl; e < e1; e += RS_LOADS << ls) {
    uint32_t p[RS_LOADS];
    Pack<T, V> x[RS_LOADS];
#pragma unroll
    for (int k = 0; k < RS_LOADS; ++k) p[k] = pos[min(e + (k << ls), e1 - 1)];
#pragma unroll
    for (int k = 0; k < RS_LOADS; ++k) x[k] = *(const Pack<T, V>*)(out + (int64_t)(p[k] & mask) * nvec + v);
#pragma unroll
    for (int k = 0; k < RS_LOADS; ++k) {
      if (e + (k << ls) >= e1) continue;
      double w = 1.0;
      if constexpr (sizeof(T) == 4) w = wt[wi ? wi[e + (k << ls)] : (uint64_t)p[k] >> shift];
#pragma unroll
      for (int j = 0; j < V; ++j) {
        if constexpr (sizeof(T) == 4) acc[j] += w * (double)x[k].x[j];
        else acc[j] += x[k].x[j];
      }
    }
  }
  for (int o = 1 << lg; o < 1 << (lg + ls); o <<= 1)
#pragma unroll
    for (int j = 0; j < V; ++j) acc[j] += __shfl_xor(acc[j], o);
  if (!on || sl != 0 || v1 >= nvec) return;
  double* h = hpsi + (int64_t)(row & ~RS_MULTI) * nvec + v;
#pragma unroll
  for (int j = 0; j < V; ++j) {
    if (row & RS_MULTI) atomicAdd(h + j, acc[j]);
    else h[j] += acc[j];
  }
}

template <class T, int V>
int add(const RowSum& s, const T* out, int nvec, double* hpsi, hipStream_t st) {
  int lg = 0;
  while ((V << lg) < nvec && lg < 3) ++lg;
  const int ls = RS_LANES > lg ? RS_LANES - lg : 0;
  const int64_t nb = ((s.nseg << (lg + ls)) + 255) / 256;
  hipLaunchKernelGGL((k_rs_add<T, V>), dim3((unsigned)nb, (unsigned)((nvec + (V << lg) - 1) / (V << lg))), dim3(256),
                     0, st, s.pos.as<uint32_t>(), s.wi.as<uint8_t>(), s.wtab.as<double>(), s.nw, s.shift, s.seg.as<int32_t>(), s.nseg,
                     out, nvec, lg, ls, hpsi);
  RS_TRY(hipGetLastError());
  return SG4_OK;
}

}  // namespace

int rowsum_build(RowSum& s, const int32_t* d_map, int64_t sum_nb, int64_t rows, const TermDev* d_terms,
                 const std::vector<TermDev>& terms, hipStream_t st) {
  if (s.tried) return SG4_OK;
  s.tried = true;
  if (sum_nb >= RS_PLACES || rows >= INT32_MAX) return SG4_OK;
  std::map<double, int> ids;
  std::vector<double> tab;
  std::vector<uint8_t> tw(terms.size());
  for (size_t t = 0; t < terms.size(); ++t) {
    const auto it = ids.emplace(terms[t].wgt, (int)tab.size());
    if (it.second) tab.push_back(terms[t].wgt);
    if (tab.size() > RS_WEIGHTS) return SG4_OK;
    tw[t] = (uint8_t)it.first->second;
  }
  int shift = 0;
  while (sum_nb >> shift) ++shift;
  const bool apart = ((uint64_t)(tab.size() - 1) << shift) >> 32;
  if (apart) shift = 32;
  const int64_t nt = (int64_t)terms.size();
  const int ntp = (int)((nt + SCAN - 1) / SCAN), nrp = (int)((rows + SCAN - 1) / SCAN);
  // one workspace: partial sums, then counts, first places and order of the
  // rows, the terms' first rows, the terms' weight indices
  const size_t b_part = 8 * ((size_t)std::max(ntp, nrp) + 1), b_rows = 4 * (size_t)rows;
  DevBuf ws;
  if (ws.alloc(b_part + 3 * b_rows + 4 * (size_t)nt + (size_t)nt) || s.wtab.alloc(8 * tab.size())) return SG4_OK;
  uint64_t* part = ws.as<uint64_t>();
  int32_t *cnt = (int32_t*)(ws.as<char>() + b_part), *first = cnt + rows, *order = first + rows, *num = order + rows;
  uint8_t* dtw = (uint8_t*)(num + nt);
  const dim3 blk(256), sblk(SCAN), tg((unsigned)std::min<int64_t>(nt, 8192));
  RS_TRY(hipMemcpyAsync(dtw, tw.data(), nt, hipMemcpyHostToDevice, st));
  RS_TRY(hipMemcpyAsync(s.wtab.p, tab.data(), 8 * tab.size(), hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(k_rs_init, dim3(512), blk, 0, st, cnt, first, order, rows);
  hipLaunchKernelGGL(k_rs_count, dim3(2048), blk, 0, st, d_map, sum_nb, cnt, first);
  hipLaunchKernelGGL(k_rs_first<false>, tg, blk, 0, st, d_map, first, d_terms, nt, num, (const int32_t*)nullptr,
                     (int32_t*)nullptr);
  hipLaunchKernelGGL(k_rs_sums, dim3(ntp), sblk, 0, st, num, (const int32_t*)nullptr, nt, part);
  hipLaunchKernelGGL(k_rs_scan, dim3(1), sblk, 0, st, part, ntp);
  hipLaunchKernelGGL(k_rs_base, dim3(ntp), sblk, 0, st, num, nt, part);
  hipLaunchKernelGGL(k_rs_first<true>, tg, blk, 0, st, d_map, first, d_terms, nt, (int32_t*)nullptr, num, order);
  hipLaunchKernelGGL(k_rs_sums, dim3(nrp), sblk, 0, st, cnt, order, rows, part);
  hipLaunchKernelGGL(k_rs_scan, dim3(1), sblk, 0, st, part, nrp);
  RS_TRY(hipGetLastError());
  uint64_t total = 0;
  RS_TRY(hipMemcpyAsync(&total, part + nrp, sizeof(total), hipMemcpyDeviceToHost, st));
  RS_TRY(hipStreamSynchronize(st));
  const int64_t nseg = (int64_t)(total >> 32), places = (int64_t)(uint32_t)total;
  if (nseg == 0 || nseg >= RS_SEGMENTS) return SG4_OK;
  if (s.pos.alloc(4 * (size_t)places) || (apart && s.wi.alloc((size_t)places)) ||
      s.seg.alloc(4 * (2 * (size_t)nseg + 1))) {
    (void)s.pos.alloc(0);
    (void)s.wi.alloc(0);
    return SG4_OK;
  }
  hipLaunchKernelGGL(k_rs_segs, dim3(nrp), sblk, 0, st, cnt, order, rows, part, s.seg.as<int32_t>(), nseg, (int32_t)places);
  for (int i = 0; i < RS_BATCH; ++i) {
    const int64_t t0 = nt * i / RS_BATCH, t1 = nt * (i + 1) / RS_BATCH;
    if (t1 > t0)
      hipLaunchKernelGGL(k_rs_fill, dim3((unsigned)std::min<int64_t>(t1 - t0, 8192)), blk, 0, st, d_map, d_terms,
                         dtw, t0, t1, shift, cnt, s.pos.as<uint32_t>(), s.wi.as<uint8_t>());
  }
  hipLaunchKernelGGL(k_rs_sort, dim3((unsigned)((nseg + 3) / 4)), blk, 0, st, s.pos.as<uint32_t>(),
                     s.wi.as<uint8_t>(), s.seg.as<int32_t>(), nseg, (uint32_t)((1ull << shift) - 1));
  RS_TRY(hipGetLastError());
  RS_TRY(hipStreamSynchronize(st));
  s.nseg = nseg;
  s.nw = (int)tab.size();
  s.shift = shift;
  s.ok = true;
  return SG4_OK;
}

void* rowsum_held(const RowSum& s, hipStream_t st, size_t bytes) {
  for (const auto& o : s.out)
    if (o->stream == st && o->buf.n >= bytes) return o->buf.p;
  return nullptr;
}

bool rowsum_fits(const RowSum& s, hipStream_t st, size_t bytes) {
  size_t held = 0, blocks = 0;
  for (const auto& o : s.out)
    if (o->stream != st) { held += o->buf.n; ++blocks; }
  return bytes < s.failed && blocks < RS_MAX_BLOCKS && held + bytes <= RS_MAX_BYTES;
}

void* rowsum_alloc(RowSum& s, hipStream_t st, size_t bytes) {
  RowSum::Out* o = nullptr;
  for (const auto& x : s.out)
    if (x->stream == st) o = x.get();
  const size_t had = o ? o->buf.n : 0;
  if (!o) {
    s.out.push_back(std::make_unique<RowSum::Out>());
    o = s.out.back().get();
    o->stream = st;
  }
  if (o->buf.alloc(bytes) == SG4_OK) return o->buf.p;   // freeing waits for the applies that still use it
  s.failed = bytes;
  if (!had || o->buf.alloc(had)) rowsum_drop(s, st);
  return nullptr;
}

void rowsum_drop(RowSum& s, hipStream_t st) {
  s.out.erase(std::remove_if(s.out.begin(), s.out.end(), [&](const auto& o) { return o->stream == st; }), s.out.end());
}

int rowsum_add(const RowSum& s, const double* out, int nvec, double* hpsi, hipStream_t st) {
  return nvec % 2 ? add<double, 1>(s, out, nvec, hpsi, st) : add<double, 2>(s, out, nvec, hpsi, st);
}
int rowsum_add(const RowSum& s, const float* out, int nvec, double* hpsi, hipStream_t st) {
  if (nvec % 2) return add<float, 1>(s, out, nvec, hpsi, st);
  return nvec % 4 ? add<float, 2>(s, out, nvec, hpsi, st) : add<float, 4>(s, out, nvec, hpsi, st);
}

}  // namespace sg4
