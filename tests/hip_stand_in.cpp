// A stand-in for the HIP runtime on a machine without a GPU: device memory is
// host memory, at most `memory_limit` bytes of it, and nothing is launched.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>
#include <cstdlib>
#include <cstring>
#include <map>

uint64_t memory_limit = ~0ull, memory_used = 0, memory_peak = 0;
hipMemoryType column_type = hipMemoryTypeHost;
static std::map<void*, size_t> device;
static int handles = 0;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  if (memory_used + n > memory_limit) return hipErrorOutOfMemory;
  *p = calloc(1, n ? n : 1);
  device[*p] = n;
  memory_used += n;
  if (memory_used > memory_peak) memory_peak = memory_used;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  memory_used -= device[p];
  device.erase(p);
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  memset(a, 0, sizeof(*a));
  a->type = column_type;
  a->devicePointer = const_cast<void*>(p);
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof(*p));
  p->multiProcessorCount = 256;
  p->sharedMemPerBlock = 65536;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 163840; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = reinterpret_cast<hipEvent_t>(&handles); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = reinterpret_cast<hipStream_t>(&handles); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return ""; }
}
