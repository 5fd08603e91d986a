// One output record (io_fault.cu:16-275, io_wave_{xy,xz,yz}.cu) gathered on
// the device: the 13 fault fields and the three velocity components of the
// three wave slices, as the 32-bit words the files hold, in one buffer that
// one copy brings to the host.
//
// An xz slice is one column of every plane, an xy slice one row.  Copied
// piece by piece they were a transfer per plane and component, for xz of the
// whole plane (a record at 200 x 160 x 120: 600 copies of 110 KB and 600 of
// 0.7 KB).  A record is a few MB: what is left is one small kernel, one copy
// to pinned memory and the file writes.  Ten steps and a record on that grid:
// 33.6 -> 16.9 ms (the steps alone are 15.5).
#include "cgfdm_internal.h"

namespace cgfdm {

namespace {

struct RecordArgs {
  FaultDev F;
  const float* W;
  uint32_t* out;
  RecordDims d;
  long words, fault_words;
  int py, jpad;
  long pyz;
};

__global__ void __launch_bounds__(256) record_kernel(RecordArgs a) {
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= a.words) return;
  const FaultDev& F = a.F;
  const long n2 = (long)a.d.nj * a.d.nk;
  long r = idx;
  uint32_t w = 0;
  if (r < a.fault_words) {
    const int v = (int)(r / n2);
    const long q = r - v * n2;
    auto f32 = [&](const float* p) { return __float_as_uint(p[q]); };
    auto f64 = [&](const double* p) { return p ? __float_as_uint((float)p[q]) : 0u; };
    switch (v) {  // uniform but for the threads at a field's end
      case 0: w = f32(F.Vs1); break;
      case 1: w = f32(F.Vs2); break;
      case 2: w = f32(F.Tn); break;
      case 3: w = f32(F.Ts1); break;
      case 4: w = f32(F.Ts2); break;
      case 5: w = f64(F.slip); break;
      case 6: w = f64(F.State); break;
      case 7: w = (uint32_t)F.rup_index_y[q]; break;
      case 8: w = (uint32_t)F.rup_index_z[q]; break;
      case 9: w = f32(F.rup_sensor); break;
      case 10: w = f64(F.TP_T); break;
      case 11: w = f64(F.TP_P); break;
      case 12: w = f32(F.init_t0); break;
      default: break;
    }
    a.out[idx] = w;
    return;
  }
  r -= a.fault_words;
  // slices: component, then the slice's rows (xy: i of j words; xz: i of k; yz: k of j)
  int i, j, k, c;
  const long nxy = (long)a.d.ni * a.d.nj, nxz = (long)a.d.ni * a.d.nk;
  if (r < 3 * nxy) {
    c = (int)(r / nxy);
    r -= c * nxy;
    i = (int)(r / a.d.nj);
    j = (int)(r - (long)i * a.d.nj);
    k = a.d.kz;
  } else if (r < 3 * (nxy + nxz)) {
    r -= 3 * nxy;
    c = (int)(r / nxz);
    r -= c * nxz;
    i = (int)(r / a.d.nk);
    k = (int)(r - (long)i * a.d.nk);
    j = a.d.jy;
  } else {
    r -= 3 * (nxy + nxz);
    c = (int)(r / n2);
    r -= c * n2;
    k = (int)(r / a.d.nj);
    j = (int)(r - (long)k * a.d.nj);
    i = a.d.ix;
  }
  a.out[idx] = __float_as_uint(a.W[((long)(i + 3) * 9 + c) * a.pyz + (long)(k + 3) * a.py + a.jpad + j + 3]);
}

}  // namespace

// A record's words on the context's GPU and in pinned host memory.
hipError_t alloc_record(Ctx& c, const RecordDims& d, uint32_t** dev, uint32_t** host) {
  const OnDevice on(c);
  const size_t bytes = (size_t)d.words() * sizeof(uint32_t);
  if (hipError_t e = hipMalloc(dev, bytes)) return e;
  return hipHostMalloc(host, bytes, hipHostMallocDefault);
}

// Gathers the record of the current wavefield and waits for it in `host`
// (pinned, d.words() words).
hipError_t gather_record(Ctx& c, const RecordDims& d, uint32_t* dev, uint32_t* host) {
  const OnDevice on(c);
  RecordArgs a{};
  a.F = c.f;
  a.W = c.cur;
  a.out = dev;
  a.d = d;
  a.words = d.words();
  a.fault_words = d.fault_words();
  a.py = c.d.py; a.jpad = c.d.jpad; a.pyz = c.d.pyz;
  hipLaunchKernelGGL(record_kernel, dim3((unsigned)((d.words() + 255) / 256)), dim3(256), 0, c.stream, a);
  if (hipError_t e = hipGetLastError()) return e;
  if (hipError_t e = hipMemcpyAsync(host, dev, d.words() * sizeof(uint32_t), hipMemcpyDeviceToHost, c.stream)) return e;
  return hipStreamSynchronize(c.stream);
}

}  // namespace cgfdm
