// Device allocation owned by a plan (or by one call).
#pragma once
#include <hip/hip_runtime.h>

#include <string>

#include "sg4_internal.h"

namespace sg4 {

struct DevBuf {
  void* p = nullptr;
  size_t n = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf() { if (p) (void)hipFree(p); }
  int alloc(size_t bytes) {
    if (p) { (void)hipFree(p); p = nullptr; }
    n = bytes;
    if (bytes == 0) return SG4_OK;
    if (hipMalloc(&p, bytes) != hipSuccess) {
      (void)hipGetLastError();
      set_error("device allocation of " + std::to_string(bytes) + " bytes failed");
      p = nullptr;
      n = 0;
      return SG4_ERR_OOM;
    }
    return SG4_OK;
  }
  template <class T> T* as() const { return (T*)p; }
};

}  // namespace sg4
