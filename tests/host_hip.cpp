// Stand-in for the HIP runtime on a machine without a GPU, for tests of the
// library's host side: device memory is host memory, copies are memcpy, kernels
// do not run, and every call that matters is kept in a log.  Loaded with global
// visibility before the library, its symbols take the place of the runtime's.
// Fresh memory is filled with one 32-bit word (hh_fill), so that a test chooses
// what the kernels that did not run have left behind (allocations beyond 1 GiB
// are zeros and take no memory until they are written).
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::string g_log;
std::map<const void*, std::string> g_names;
std::map<void*, size_t> g_mem;
int g_fill = 0, g_capturing = 0, g_fail_record = 0;
long g_allow = -1;          // allocations that succeed before one fails; -1: all
size_t g_limit = 0;         // bytes of device memory; 0: unlimited
size_t g_held = 0;
int g_handles = 0;
hipError_t g_last = hipSuccess;
constexpr size_t BIG = size_t(1) << 30;
struct Cfg { dim3 g, b; size_t lds; hipStream_t st; } g_cfg;

void note(const std::string& s) { g_log += s + "\n"; }
std::string num(size_t x) { return std::to_string(x); }
std::string at(const void* p) { return num((size_t)p); }
}  // namespace

extern "C" {
void hh_fill(int word) { g_fill = word; }
void hh_capturing(int on) { g_capturing = on; }
void hh_allow(long n) { g_allow = n; }
void hh_limit(size_t bytes) { g_limit = bytes; }
void hh_fail_record(int n) { g_fail_record = n; }   // the n-th event record from now on fails
size_t hh_held() { return g_held; }
const char* hh_log() { return g_log.c_str(); }
void hh_clear() { g_log.clear(); }

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
  g_names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t st) { g_cfg = Cfg{g, b, lds, st}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* st) {
  *g = g_cfg.g; *b = g_cfg.b; *lds = g_cfg.lds; *st = g_cfg.st;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t st) {
  note("launch " + g_names[f] + " " + num(g.x) + " " + num(g.y) + " " + num(g.z) + " " + num(b.x) + " " + at(st));
  // the runtime's limit: fewer than 2^32 threads in every direction
  if ((size_t)g.x * b.x >> 32 || (size_t)g.y * b.y >> 32 || g.y > 65535 || g.z > 65535)
    return g_last = hipErrorInvalidConfiguration;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  *p = nullptr;
  if ((g_limit && g_held + n > g_limit) || (g_allow >= 0 && g_allow-- == 0)) {
    note("nomem " + num(n));
    return hipErrorOutOfMemory;
  }
  if (n > BIG) {
    *p = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  } else {
    *p = std::malloc(n + 256);
    for (size_t i = 0; i < n / 4; ++i) ((int*)*p)[i] = g_fill;
  }
  g_mem[*p] = n;
  g_held += n;
  note("malloc " + num(n) + " " + at(*p));
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  const auto i = g_mem.find(p);
  if (i == g_mem.end()) return hipErrorInvalidValue;
  note("free " + num(i->second) + " " + at(p));
  g_held -= i->second;
  if (i->second > BIG) munmap(p, i->second);
  else std::free(p);
  g_mem.erase(i);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { note("memcpy " + num(n)); std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
  note("memcpyasync " + num(n) + " " + at(st));
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)(size_t)(0x1000 + 16 * ++g_handles); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t st) { note("sync " + at(st)); return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* c) {
  *c = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { g_capturing = 1; note("capture"); return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { g_capturing = 0; note("endcapture"); *g = nullptr; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) { *e = nullptr; return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { note("graphdestroy"); return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)(size_t)(0x1000 + 16 * ++g_handles); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t st) {
  if (g_fail_record > 0 && --g_fail_record == 0) return hipErrorUnknown;
  note("record " + at(st));
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600*, int) { return hipErrorUnknown; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { static void* s = std::malloc(size_t(256) << 20); *p = s; return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  std::memset(a, 0, sizeof(*a));
  a->type = hipMemoryTypeDevice;
  a->devicePointer = (void*)p;
  return hipSuccess;
}
}
