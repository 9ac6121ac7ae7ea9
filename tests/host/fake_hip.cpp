#include "fake_hip.h"

#include <chrono>
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>

namespace fake {
std::function<void(const Launch&)> on_launch;
long mallocs_left = -1, pinned_left = -1, instantiates_left = -1, capture_us = 0, replay_us = 0, mallocs = 0, captures = 0;

static std::mutex mu;
static std::map<char*, size_t>& blocks() {
  static std::map<char*, size_t> m;
  return m;
}
static std::map<const void*, std::string>& names() {   // registered before main()
  static std::map<const void*, std::string> m;
  return m;
}
static bool capturing = false;
static hipError_t last_error = hipSuccess;
static struct { dim3 grid, block; size_t shmem; hipStream_t stream; } pushed;

static hipError_t alloc(void** p, size_t n, long* left, hipError_t none) {
  std::lock_guard<std::mutex> lk(mu);
  if (*left == 0) return last_error = none;
  if (*left > 0) --*left;
  *p = calloc(1, n ? n : 1);
  blocks()[(char*)*p] = n;
  return hipSuccess;
}
static hipError_t release(void* p) {
  std::lock_guard<std::mutex> lk(mu);
  if (p && !blocks().erase((char*)p)) {
    std::fprintf(stderr, "free of %p, which is not allocated\n", p);
    std::abort();
  }
  free(p);
  return hipSuccess;
}
size_t live() {
  std::lock_guard<std::mutex> lk(mu);
  return blocks().size();
}
size_t bytes_at(const void* p) {
  std::lock_guard<std::mutex> lk(mu);
  auto it = blocks().upper_bound((char*)p);
  if (it == blocks().begin()) return 0;
  --it;
  const size_t off = (const char*)p - it->first;
  return off < it->second ? it->second - off : 0;
}
template <typename H>
static hipError_t handle(H* h) {
  static long next = 0;
  *h = (H)(++next * 16);
  return hipSuccess;
}
}  // namespace fake

using namespace fake;

extern "C" {
void** __hipRegisterFatBinary(const void*) {
  static void* h;
  return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*, void*, dim3*, dim3*,
                           int*) {
  int st = 0;
  char* d = abi::__cxa_demangle(device, nullptr, nullptr, &st);
  std::string s = st == 0 ? d : device;
  free(d);
  if (s.rfind("void ", 0) == 0) s = s.substr(5);
  names()[host] = s.substr(0, s.find('('));
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t stream) {
  pushed = {grid, block, shmem, stream};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, hipStream_t* stream) {
  *grid = pushed.grid;
  *block = pushed.block;
  *shmem = pushed.shmem;
  *stream = pushed.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, hipStream_t) {
  if (on_launch) on_launch(Launch{names()[f], grid.x, block.x, args});
  return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n) {
  ++mallocs;
  return alloc(p, n, &mallocs_left, hipErrorOutOfMemory);
}
hipError_t hipFree(void* p) { return release(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return alloc(p, n, &pinned_left, hipErrorOutOfMemory); }
hipError_t hipHostFree(void* p) { return release(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void**, const void*) { return hipErrorInvalidSymbol; }

hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = last_error;
  last_error = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1.0f;
  return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  capturing = true;
  ++captures;
  if (capture_us) std::this_thread::sleep_for(std::chrono::microseconds(capture_us));
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  capturing = false;
  return handle(g);
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  if (instantiates_left == 0) {
    *e = nullptr;
    return last_error = hipErrorOutOfMemory;
  }
  if (instantiates_left > 0) --instantiates_left;
  return handle(e);
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
  if (replay_us) std::this_thread::sleep_for(std::chrono::microseconds(replay_us));
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}
