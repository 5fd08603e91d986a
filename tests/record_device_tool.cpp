// Test helper: which GPU is current while an output record's buffers are
// allocated and its kernel is launched, for a context on GPU 1 and a caller
// whose current GPU is 0.  Its own definitions of the HIP calls below take the
// place of the runtime's in the solver's library, so no GPU is needed.
#include "cgfdm_internal.h"
#include <cstdio>
#include <cstdlib>

static int current = 0;

extern "C" {
hipError_t hipGetDevice(int* d) { *d = current; return hipSuccess; }
hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { std::printf("malloc %d\n", current); *p = std::malloc(n); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = std::malloc(n); return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { std::printf("launch %d\n", current); return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
}

int main() {
  cgfdm::Ctx c;
  c.device = 1;
  const cgfdm::RecordDims d{8, 9, 10, 1, 2, 3, 1};
  uint32_t *dev = nullptr, *host = nullptr;
  if (cgfdm::alloc_record(c, d, &dev, &host)) return 1;
  std::printf("after %d\n", current);
  if (cgfdm::gather_record(c, d, dev, host)) return 1;
  std::printf("after %d\n", current);
  std::free(dev);
  std::free(host);
  return 0;
}
