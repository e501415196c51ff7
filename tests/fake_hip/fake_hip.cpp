// A HIP runtime without a GPU, for tests of the library's host code: device
// memory is host memory, copies happen at once, kernels do nothing.  It counts
// the work queued since the last synchronisation (once pinned memory exists, which
// that work may read), and makes the n-th call that can fail (an allocation, a
// copy, a launch) return an error.  It lists the kernels launched, by name.  Load it with
// RTLD_GLOBAL before liborion_hip.so, whose HIP calls then come here.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
int calls = 0, fail_at = 0, queued = 0, pinned = 0, mallocs = 0, copies = 0;
hipError_t last = hipSuccess;
bool fails() { return ++calls == fail_at; }
void queue() { queued += pinned > 0; }
hipError_t error(hipError_t e) { return last = e; }
char symbol_memory[256];
std::map<const void*, std::string> kernels;
std::string launched;
struct Launch {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
} launch;
}  // namespace

extern "C" {
void fake_hip_fail_at(int n) { calls = queued = 0, fail_at = n; }
int fake_hip_calls() { return calls; }
const char* fake_hip_launched() { return launched.c_str(); }
void fake_hip_clear_launched() { launched.clear(); }
int fake_hip_queued() { return queued; }
int fake_hip_mallocs() { return mallocs; }
int fake_hip_copies() { return copies; }

hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_t* p, int) {
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->name, "fake");
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  p->totalGlobalMem = size_t(1) << 34;
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) { return *f = *t = size_t(1) << 34, hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
hipError_t hipMalloc(void** p, size_t bytes) {
  if (fails()) return error(hipErrorOutOfMemory);
  ++mallocs;
  *p = std::calloc(bytes, 1);
  return hipSuccess;
}
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  if (fails()) return error(hipErrorOutOfMemory);
  ++pinned;
  *p = std::calloc(bytes, 1);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  --pinned;
  return std::free(p), hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { return *p = symbol_memory, hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  if (fails()) return error(hipErrorUnknown);
  queue(), ++copies;
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemcpy2DAsync(void*, size_t, const void*, size_t, size_t, size_t, hipMemcpyKind,
                            hipStream_t) {
  if (fails()) return error(hipErrorUnknown);
  queue(), ++copies;
  return hipSuccess;
}
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) {
  if (fails()) return error(hipErrorUnknown);
  queue();
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  return *s = reinterpret_cast<hipStream_t>(&launch), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return queued = 0, hipSuccess; }
hipError_t hipDeviceSynchronize() { return queued = 0, hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  return *e = reinterpret_cast<hipEvent_t>(&launch), hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return queued = 0, hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0, hipSuccess; }

// What a kernel launch compiles to.
void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*,
                           void*, void*, int*) {
  kernels[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
  return launch = {grid, block, shared, stream}, hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared,
                                     hipStream_t* stream) {
  *grid = launch.grid, *block = launch.block, *shared = launch.shared, *stream = launch.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void**, size_t, hipStream_t) {
  if (fails()) return error(hipErrorLaunchFailure);
  launched += kernels[f] + " " + std::to_string(grid.z) + "\n";
  queue();
  return hipSuccess;
}
}
