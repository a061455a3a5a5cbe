// The part of the HIP runtime that the BERT driver and the kernel library call,
// on host memory and without kernels: loaded in front of the real one it lets
// the driver's host code run where there is no GPU, and refuses the allocation it
// is told to.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>

namespace {
long g_count, g_failAt = -1, g_launches;
size_t g_live;
std::map<void *, size_t> g_sizes;
hipError_t take(void **p, size_t bytes) {
  *p = nullptr;
  if (g_count++ == g_failAt)
    return hipErrorOutOfMemory;
  *p = calloc(bytes ? bytes : 1, 1);
  g_sizes[*p] = bytes;
  g_live += bytes;
  return hipSuccess;
}
hipError_t give(void *p) {
  if (p) {
    if (!g_sizes.count(p))
      abort(); // never allocated, or freed before
    g_live -= g_sizes[p];
    g_sizes.erase(p);
    free(p);
  }
  return hipSuccess;
}
} // namespace

extern "C" {
void hostHipFailAt(long n) { // the n-th allocation from now on (from 0), or none (-1)
  g_count = 0;
  g_failAt = n;
}
long hostHipAllocations() { return g_count; }
long hostHipLaunches() { return g_launches; }
size_t hostHipLiveBytes() { return g_live; }

hipError_t hipMalloc(void **p, size_t bytes) { return take(p, bytes); }
hipError_t hipFree(void *p) { return give(p); }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { return take(p, bytes); }
hipError_t hipHostFree(void *p) { return give(p); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  return memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) { return memset(d, v, n), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(malloc(1));
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { return free(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *c) {
  *c = hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = reinterpret_cast<hipEvent_t>(malloc(1));
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { return free(e), hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  memset(p, 0, sizeof(*p));
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { return *n = 1, hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return g_launches++, hipSuccess; }
}
