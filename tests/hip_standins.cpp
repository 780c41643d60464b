// Stand-ins for the parts of the HIP runtime that the library's memory and copies use, on host memory: loaded
// before the runtime (LD_PRELOAD), they let a test without a GPU make a chosen call fail.  Kernels are not run.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>

namespace {
int events_made = 0, blocks_refused = 0;
}

extern "C" {
int standin_blocks_refused() { return blocks_refused; }
hipError_t hipGetDeviceCount(int *count) { return *count = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *props, int) {
  memset(props, 0, sizeof *props);
  strcpy(props->gcnArchName, "gfx950");
  props->multiProcessorCount = 256;
  props->totalGlobalMem = size_t(1) << 32;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **ptr, const void *) { return *ptr = malloc(1 << 20), hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *stream, unsigned) { return *stream = reinterpret_cast<hipStream_t>(1), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
// STANDIN_LARGEST=bytes: larger blocks cannot be had
hipError_t hipMalloc(void **ptr, size_t size) {
  const char *largest = getenv("STANDIN_LARGEST");
  if (largest && size > strtoull(largest, nullptr, 10)) return ++blocks_refused, hipErrorOutOfMemory;
  return *ptr = malloc(size), hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipFree(void *ptr) { return free(ptr), hipSuccess; }
hipError_t hipHostMalloc(void **ptr, size_t size, unsigned) { return *ptr = malloc(size), hipSuccess; }
hipError_t hipHostFree(void *ptr) { return free(ptr), hipSuccess; }
hipError_t hipMemcpy(void *dst, const void *src, size_t size, hipMemcpyKind) { return memcpy(dst, src, size), hipSuccess; }
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t size, hipMemcpyKind, hipStream_t) { return memcpy(dst, src, size), hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return hipSuccess; }
// STANDIN_FAIL_EVENT=n: the n-th event cannot be made
hipError_t hipEventCreateWithFlags(hipEvent_t *event, unsigned) {
  const char *fail = getenv("STANDIN_FAIL_EVENT");
  if (fail && ++events_made == atoi(fail)) return hipErrorOutOfMemory;
  return *event = reinterpret_cast<hipEvent_t>(1), hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t event, hipStream_t) { return event ? hipSuccess : hipErrorInvalidHandle; }
hipError_t hipEventSynchronize(hipEvent_t event) { return event ? hipSuccess : hipErrorInvalidHandle; }
}
