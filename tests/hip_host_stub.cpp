// A HIP runtime without a device, for tests of the library's host code on the
// CPU: device memory is host memory, copies are done at once, kernels are not
// run.  It counts launches, remembers destroyed streams (a call on one is
// counted, not followed) and fails a chosen hipMemcpyAsync or launch.
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <set>

namespace {
std::mutex lock;
std::set<hipStream_t> streams;  // those not destroyed
std::atomic<long> ordinary{0}, cooperative{0}, dead_uses{0}, live_streams{0};
std::atomic<void*> last_pinned{nullptr};
std::atomic<long> copy_countdown{0}, coop_countdown{0};

void use(hipStream_t s) {
  if (!s) return;
  std::lock_guard<std::mutex> hold(lock);
  if (!streams.count(s)) ++dead_uses;
}
bool fails(std::atomic<long>& c) { return c.load() > 0 && c.fetch_sub(1) == 1; }

struct Config {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
};
thread_local Config config;
}  // namespace

extern "C" {
long stub_ordinary() { return ordinary; }
long stub_cooperative() { return cooperative; }
long stub_dead_uses() { return dead_uses; }
long stub_live_streams() { return live_streams; }
void* stub_last_pinned() { return last_pinned; }
void stub_fail_copy(long nth) { copy_countdown = nth; }         // the nth copy from now
void stub_fail_cooperative(long nth) { coop_countdown = nth; }  // the nth such launch

hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 100000;
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void*) {
  std::memset(a, 0, sizeof(*a));
  a->numRegs = 128;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  *p = std::calloc(n ? n : 1, 1);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  const hipError_t e = hipMalloc(p, n);
  last_pinned = *p;
  return e;
}
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static void* scratch = std::calloc(1, 64u << 20);
  *p = scratch;
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t q) {
  use(q);
  if (fails(copy_countdown)) return hipErrorUnknown;
  std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h,
                            hipMemcpyKind, hipStream_t q) {
  use(q);
  for (size_t k = 0; k < h; ++k)
    std::memmove(static_cast<char*>(d) + k * dp, static_cast<const char*>(s) + k * sp, w);
  return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) { std::memset(p, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t q) {
  use(q);
  std::memset(p, v, n);
  return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t* q) {
  std::lock_guard<std::mutex> hold(lock);
  *q = reinterpret_cast<hipStream_t>(std::malloc(8));  // kept: no address comes twice
  streams.insert(*q);
  ++live_streams;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t q) {
  use(q);
  std::lock_guard<std::mutex> hold(lock);
  if (streams.erase(q)) --live_streams;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t q) { use(q); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = reinterpret_cast<hipEvent_t>(std::malloc(8));
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t q) { use(q); return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.0f; return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t q) {
  use(q);
  ++ordinary;
  return hipSuccess;
}
hipError_t hipLaunchCooperativeKernel(const void*, dim3, dim3, void**, unsigned, hipStream_t q) {
  use(q);
  if (fails(coop_countdown)) return hipErrorUnknown;
  ++cooperative;
  return hipSuccess;
}

// what hipcc's generated host code calls
void** __hipRegisterFatBinary(const void*) {
  static void* handle = nullptr;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*,
                           void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  config = Config{g, b, lds, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
  *g = config.grid;
  *b = config.block;
  *lds = config.lds;
  *s = config.stream;
  return hipSuccess;
}
}  // extern "C"
