// The HIP calls that libwebgpt_amd.so makes, on host memory: allocations and copies are the host's, a kernel launch does
// nothing but count, and launch `host_hip_fail_at` (from 1; 0: none) or allocation `host_hip_alloc_fail_at` fails instead; the error
// stays until hipGetLastError has been asked. Loaded in front of the library
// (RTLD_GLOBAL) it takes the place of the HIP runtime in that process, so that the library's host code can be tested
// without a GPU, its error paths among them.
#include <cstdlib>
#include <cstring>

#include <hip/hip_runtime_api.h>

extern "C" {
int host_hip_launches = 0, host_hip_fail_at = 0;
int host_hip_allocs = 0, host_hip_alloc_fail_at = 0, host_hip_frees = 0;
int host_hip_unwaited = 0;  // launches since the last wait for the stream

static dim3 cfg_grid, cfg_block;
static size_t cfg_shared;
static hipStream_t cfg_stream;
static float symbol[1 << 20];

hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t s) {
  cfg_grid = grid, cfg_block = block, cfg_shared = shared, cfg_stream = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* s) {
  *grid = cfg_grid, *block = cfg_block, *shared = cfg_shared, *s = cfg_stream;
  return hipSuccess;
}
static hipError_t last = hipSuccess;
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
  ++host_hip_launches;
  if (host_hip_launches == host_hip_fail_at) return last = hipErrorLaunchFailure;
  ++host_hip_unwaited;
  return hipSuccess;
}
hipError_t hipGetLastError(void) {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "an error of the host's own"; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  memset(p, 0, sizeof *p);
  strcpy(p->name, "host");
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { return *p = symbol, hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
static hipError_t allocate(void** p, size_t n) {
  if (++host_hip_allocs == host_hip_alloc_fail_at || !(*p = malloc(n))) return last = hipErrorOutOfMemory;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) { return allocate(p, n); }
hipError_t hipFree(void* p) { return ++host_hip_frees, free(p), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return allocate(p, n); }
hipError_t hipHostFree(void* p) { return free(p), hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemset(void* d, int v, size_t n) { return memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return memset(d, v, n), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = reinterpret_cast<hipStream_t>(symbol), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return host_hip_unwaited = 0, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = reinterpret_cast<hipEvent_t>(symbol), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
}
