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
  // when a wider apply needs it
  struct Out { hipStream_t stream; DevBuf buf; };
  std::vector<std::unique_ptr<Out>> out;
  size_t failed = SIZE_MAX;   // the smallest block that the device had no memory for
};

// places and segments from the map; not ok (and no error) when they do not
// fit the index types or the device memory
int rowsum_build(RowSum& s, const int32_t* d_map, int64_t sum_nb, int64_t rows, const TermDev* d_terms,
                 const std::vector<TermDev>& terms, hipStream_t st);
// the stream's block if it holds `bytes`, or null
void* rowsum_held(const RowSum& s, hipStream_t st, size_t bytes);
// whether a block of `bytes` in place of the stream's is within the limits of a
// plan (and not known to exceed the device's memory)
bool rowsum_fits(const RowSum& s, hipStream_t st, size_t bytes);
// a block of `bytes` in place of the stream's, or null (the stream keeps what it had)
void* rowsum_alloc(RowSum& s, hipStream_t st, size_t bytes);
void rowsum_drop(RowSum& s, hipStream_t st);   // gives the stream's block back
// hpsi(r, v) += the row's places of out (float: times the term weights)
int rowsum_add(const RowSum& s, const double* out, int nvec, double* hpsi, hipStream_t st);
int rowsum_add(const RowSum& s, const float* out, int nvec, double* hpsi, hipStream_t st);

}  // namespace sg4
