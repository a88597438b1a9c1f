// Sum over the Smolyak terms of the term kernels' results, row by row.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <memory>
#include <vector>

#include "sg4_buf.h"
#include "sg4_device.h"

namespace sg4 {

// The map inverted: for every packed row the places (offsets in the map) of
// the terms that hold it.  A segment is at most RS_SEG consecutive places of
// one row; bit 31 of its row marks a row of several segments.
struct RowSum {
  bool tried = false, ok = false;
  int64_t nseg = 0;
  int shift = 0, nw = 0;
  DevBuf pos;      // uint32, rows after rows: place | (index of its term's weight << shift)
  DevBuf wi;       // uint8 weight indices where they do not fit beside the place (shift = 32)
  DevBuf wtab;     // the distinct term weights
  DevBuf seg;      // int32: nseg + 1 starts in pos, then nseg rows
  // the terms' results of one apply: a block per stream, replaced by a larger one
  // when a wider apply needs it, unless graphs hold it (keep)
  struct Out { hipStream_t stream; DevBuf buf; };
  std::vector<std::unique_ptr<Out>> out;
};

// places and segments from the map; not ok (and no error) when they do not
// fit the index types or the device memory
int rowsum_build(RowSum& s, const int32_t* d_map, int64_t sum_nb, int64_t rows, const TermDev* d_terms,
                 const std::vector<TermDev>& terms, hipStream_t st);
// the stream's block of at least `bytes`, or null (none within the limits; alloc = false: none held);
// keep: the stream's smaller blocks stay
void* rowsum_block(RowSum& s, hipStream_t st, size_t bytes, bool alloc, bool keep);
// hpsi(r, v) += the row's places of out (float: times the term weights)
int rowsum_add(const RowSum& s, const double* out, int nvec, double* hpsi, hipStream_t st);
int rowsum_add(const RowSum& s, const float* out, int nvec, double* hpsi, hipStream_t st);

}  // namespace sg4
