// Host code of libscn_hip.so with the HIP runtime's calls replaced by the ones below: no GPU is used, kernels are counted and not run.
// Usage: host_checks NAME; prints "ok" and returns 0, or says which check failed.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../include/scn_hip.h"
#include "../../sparseconvnet_amd/csrc/conv_common.h"

static int mallocs, fail_malloc = -1, launches;  // fail_malloc: that many succeed, the next two fail (the library tries twice)
static bool fail_launch, capturing;
static hipError_t last = hipSuccess;

extern "C" {
hipError_t hipMalloc(void **p, size_t bytes) {
  if (fail_malloc >= 0 && (mallocs == fail_malloc || mallocs == fail_malloc + 1)) {
    mallocs++;
    return last = hipErrorOutOfMemory;
  }
  mallocs++;
  *p = calloc(1, bytes);
  return hipSuccess;
}
hipError_t hipFree(void *p) { return free(p), hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
  *p = calloc(1, bytes);
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) { return a->device = 0, hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) {
  launches++;
  return fail_launch ? last = hipErrorLaunchFailure : hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = (hipEvent_t)malloc(8), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
  return *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone, hipSuccess;
}
}

#define CHECK(x)                                            \
  do {                                                      \
    if (!(x)) {                                             \
      printf("%s:%d: %s\n", __FILE__, __LINE__, #x);        \
      exit(1);                                              \
    }                                                       \
  } while (0)

using namespace scn;

// A failed allocation is reported by its own error and not once more by the next launch.
static void failed_allocation() {
  mallocs = 0;
  fail_malloc = 0;
  bool threw = false;
  try {
    pool_alloc(5000, POOL_COMPUTE);
  } catch (const std::exception &) {
    threw = true;
  }
  fail_malloc = -1;
  CHECK(threw && mallocs == 2 && hipGetLastError() == hipSuccess);
}

int main(int argc, char **argv) {
  const char *name = argc > 1 ? argv[1] : "";
  if (!strcmp(name, "failed_allocation")) failed_allocation();
  else return printf("no check of that name\n"), 2;
  printf("ok\n");
  return 0;
}
