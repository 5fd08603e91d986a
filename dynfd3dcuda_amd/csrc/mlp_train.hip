// Learned Newton guess: device copy of the network, evaluation, gradient and
// training kernels (extension; no counterpart in the reference).
//
// The network and its parameter blob are described in mlp.h.  Training keeps
// FP32 master parameters P (the blob layout) and, before every batch, packs
// them into the device copy the rate-state kernel uses, so the forward pass
// of training has exactly the roundings of inference: layer-2 weights and
// first hidden layer in bf16, FP32 elsewhere and in all sums.  The backward
// pass runs in FP32 and treats the bf16 rounding as identity (gradients with
// respect to P).  Loss: mean over samples of (o - t')^2 with
// o the network output before de-standardisation and t' = (t - ymean)/yscale.
#include "cgfdm_internal.h"
#include "mlp.h"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <random>
#include <vector>

namespace cgfdm {

// Scratch of cgfdm_mlp_forward_noalloc: the packed network (an MlpDev) in
// static device memory, one copy per GPU, held until the process ends, so
// that call allocates nothing.  Every call on a GPU overwrites that GPU's
// copy: calls that overlap on one GPU race.
constexpr size_t kMlpScratchBytes = 32768;
static_assert(sizeof(MlpDev) <= kMlpScratchBytes, "the scratch holds one packed network");
static __device__ __align__(256) unsigned char scratch[kMlpScratchBytes];

// offsets of the parameter blob
constexpr int kOffW1 = 10, kOffB1 = kOffW1 + kMlpH * kMlpIn, kOffW2 = kOffB1 + kMlpH,
              kOffB2 = kOffW2 + kMlpH * kMlpH, kOffW3 = kOffB2 + kMlpH, kOffB3 = kOffW3 + kMlpH;
static_assert(kOffB3 + 1 == kMlpParams, "blob layout");

// P (FP32 blob) -> MlpDev, one thread per packed element (4096 threads)
__global__ void __launch_bounds__(256) mlp_pack_kernel(const float* __restrict__ P, MlpDev* __restrict__ m) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < kMlpH * kMlpH) m->W2[t >> 6][t & 63] = f2bf(P[kOffW2 + t]);
  if (t < kMlpH * kMlpIn) m->W1[t / kMlpIn][t % kMlpIn] = P[kOffW1 + t];
  if (t < kMlpH) {
    m->b1[t] = P[kOffB1 + t];
    m->b2[t] = P[kOffB2 + t];
    m->w3[t] = P[kOffW3 + t];
  }
  if (t < 4) {
    m->xmean[t] = P[t];
    m->xscale[t] = P[4 + t];
  }
  if (t == 0) {
    m->ymean = P[8];
    m->yscale = P[9];
    m->b3 = P[kOffB3];
  }
}

// Network output for n samples (feat [n][4]): mode 0 with the wavefront
// matrix-instruction form used in the rate-state kernel, mode 1 scalar.
__global__ void __launch_bounds__(64) mlp_forward_kernel(const MlpDev* __restrict__ m, const float* __restrict__ feat,
                                                         long n, float* __restrict__ out, int mode) {
  const long s = (long)blockIdx.x * 64 + threadIdx.x;
  const bool ok = s < n;
  float f[4];
  for (int i = 0; i < 4; i++) f[i] = ok ? feat[4 * s + i] : 0.0f;
  const float y = mode == 0 ? mlp_guess_wave(m, f) : mlp_forward_scalar(m, f);
  if (ok) out[s] = y;
}

struct GradArgs {
  const MlpDev* m;
  const float* feat;    // [n][4]
  const float* target;  // [n] log10 slip rate
  const int* idx;       // sample order, or null for 0..count-1
  long first, count;    // samples idx[first .. first+count)
  float gscale;         // 2 / count
  float* part;          // [gridDim.x][kGradRow] sums of each block
};

constexpr int kGradWaves = 4;          // wavefronts of a gradient block
constexpr int kGradBlocks = 256;       // blocks at most: one per CU
constexpr int kGradRow = kMlpParams + 1;  // gradient, then the sum of squared errors

// Blocks of the gradient kernel for a batch of count samples.
inline int grad_blocks(long count) {
  return (int)std::min<long>((count + 16 * kGradWaves - 1) / (16 * kGradWaves), kGradBlocks);
}

// Gradient of the loss over a batch, on the matrix cores: a wavefront takes
// 16 samples at a time and keeps its sums of all parameters in registers.
// With g = lane / 16 and c = lane % 16, the matrix instructions hand out their
// result as D[4 g + r][c] and take operand element r of k-slot g, so a result
// is the next product's operand as it stands when the contracted index is its
// row.  The hidden layers are therefore computed in both orientations, rows
// of units ("u", unit 16 t + 4 g + r of sample c) and rows of samples ("s",
// sample 4 g + r at unit 16 t + c), and nothing goes through LDS:
//   z2 (u and s)   bf16 products, FP32 sums, as in the forward pass
//   dW2 = dz2 h1^T   samples contracted: s operands, FP32 products
//   dz1 = W2^T dz2   hidden units contracted: u operand, FP32 products
// 128 FP32 and 32 bf16 matrix instructions per 16 samples.  The blocks' sums
// go to rows of a buffer that a second kernel adds up.  A scalar form (a lane
// per sample, products summed through LDS, every block adding its 4555 words
// to the same addresses) took 570 us at 60000 samples and 2.0 ms at 500000;
// this one 34 and 184 us, of which the FP32 matrix instructions are about a
// third (one wavefront per SIMD: 447 registers), and the sum kernel 4 us.
__global__ void __launch_bounds__(64 * kGradWaves, 1) mlp_grad_kernel(GradArgs a) {
  __shared__ __align__(16) float sW1[kMlpH][kMlpIn], sb1[kMlpH], sb2[kMlpH], sw3[kMlpH];
  __shared__ float sum[kGradWaves][kGradRow];
  const MlpDev* __restrict__ m = a.m;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g = lane >> 4, c = lane & 15;
  for (int t = tid; t < kMlpH * kMlpIn; t += 64 * kGradWaves) sW1[t / kMlpIn][t % kMlpIn] = m->W1[t / kMlpIn][t % kMlpIn];
  if (tid < kMlpH) {
    sb1[tid] = m->b1[tid];
    sb2[tid] = m->b2[tid];
    sw3[tid] = m->w3[tid];
  }
  __syncthreads();
  bf16x4 w2[4][4];      // [t][k][r]: W2[16 t + c][16 k + 4 g + r]
  float w2t[4][4][4];   // [k][t][r]: W2[16 k + 4 g + r][16 t + c]
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint16_t* q = &m->W2[16 * t + c][16 * k + 4 * g];
      w2[t][k] = bf16x4{(short)q[0], (short)q[1], (short)q[2], (short)q[3]};
#pragma unroll
      for (int r = 0; r < 4; r++) w2t[k][t][r] = bf2f(m->W2[16 * k + 4 * g + r][16 * t + c]);
    }
  f32x4 gW2[4][4];  // hidden unit 16 [.] + 4 g + r, first-layer unit 16 [.] + c
  float gW1[4][kMlpIn], gb1[4], gb2[4], gw3[4], gb3 = 0.0f, lsum = 0.0f;
#pragma unroll
  for (int t = 0; t < 4; t++) {
    gb1[t] = gb2[t] = gw3[t] = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      gW2[t][k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      gW1[t][k] = 0.0f;
    }
  }
  const long ntile = (a.count + 15) / 16;
  for (long tile = (long)blockIdx.x * kGradWaves + w; tile < ntile; tile += (long)gridDim.x * kGradWaves) {
    const long q = tile * 16 + c;
    const bool ok = q < a.count;
    long s = 0;
    if (ok) s = a.idx ? (long)a.idx[a.first + q] : a.first + q;
    float x[kMlpIn], xs[kMlpIn][4];  // standardised features of sample c, and of samples 4 g + r
#pragma unroll
    for (int i = 0; i < kMlpIn; i++) {
      x[i] = ok ? (a.feat[4 * s + i] - m->xmean[i]) * m->xscale[i] : 0.0f;
#pragma unroll
      for (int r = 0; r < 4; r++) xs[i][r] = __shfl(x[i], 4 * g + r);
    }
    const float tn = ok ? (a.target[s] - m->ymean) / m->yscale : 0.0f;
    bf16x4 h1u[4];
    float h1s[4][4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int u = 16 * t + 4 * g + r, v = 16 * t + c;
        float zu = sb1[u], zs = sb1[v];
#pragma unroll
        for (int i = 0; i < kMlpIn; i++) {
          zu = fmaf(sW1[u][i], x[i], zu);
          zs = fmaf(sW1[v][i], xs[i][r], zs);
        }
        h1u[t][r] = (short)f2bf(fmaxf(zu, 0.0f));
        h1s[t][r] = bf2f(f2bf(fmaxf(zs, 0.0f)));
      }
    }
    f32x4 zu[4], zs[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
      zu[t] = zs[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int k = 0; k < 4; k++) {
        zu[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w2[t][k], h1u[k], zu[t], 0, 0, 0);
        zs[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(h1u[k], w2[t][k], zs[t], 0, 0, 0);
      }
    }
    float o = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int u = 16 * t + 4 * g + r;
        zu[t][r] = fmaxf(zu[t][r] + sb2[u], 0.0f);
        o += sw3[u] * zu[t][r];
      }
    o += __shfl_xor(o, 16);
    o += __shfl_xor(o, 32);
    const float e = ok ? o + m->b3 - tn : 0.0f;
    const float dout = a.gscale * e;
    lsum += e * e;
    gb3 += dout;
    float ds[4];
#pragma unroll
    for (int r = 0; r < 4; r++) ds[r] = __shfl(dout, 4 * g + r);
    // dz2 in both orientations (in place of the layer's values)
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const float b2 = sb2[16 * t + c], w3 = sw3[16 * t + c];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        zu[t][r] = zu[t][r] > 0.0f ? dout * sw3[16 * t + 4 * g + r] : 0.0f;
        const float h2 = fmaxf(zs[t][r] + b2, 0.0f);
        gw3[t] += ds[r] * h2;
        zs[t][r] = h2 > 0.0f ? ds[r] * w3 : 0.0f;
        gb2[t] += zs[t][r];
      }
    }
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int t = 0; t < 4; t++)
#pragma unroll
        for (int k = 0; k < 4; k++) gW2[t][k] = __builtin_amdgcn_mfma_f32_16x16x4f32(zs[t][r], h1s[k][r], gW2[t][k], 0, 0, 0);
    f32x4 d1[4];
#pragma unroll
    for (int t = 0; t < 4; t++) d1[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int t = 0; t < 4; t++) d1[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(zu[k][r], w2t[k][t][r], d1[t], 0, 0, 0);
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float d = h1s[t][r] > 0.0f ? d1[t][r] : 0.0f;
        gb1[t] += d;
#pragma unroll
        for (int i = 0; i < kMlpIn; i++) gW1[t][i] += d * xs[i][r];
      }
  }
  // this wavefront's sums, then the block's
  auto over_g = [](float v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
  };
  auto over_c = [](float v) {
    for (int k = 1; k < 16; k *= 2) v += __shfl_xor(v, k);
    return v;
  };
  float* row = sum[w];
#pragma unroll
  for (int t = 0; t < 4; t++) {
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
      for (int r = 0; r < 4; r++) row[kOffW2 + (16 * t + 4 * g + r) * kMlpH + 16 * k + c] = gW2[t][k][r];
    const int u = 16 * t + c;
    const float b1 = over_g(gb1[t]), b2 = over_g(gb2[t]), w3 = over_g(gw3[t]);
    float w1[kMlpIn];
#pragma unroll
    for (int i = 0; i < kMlpIn; i++) w1[i] = over_g(gW1[t][i]);
    if (g == 0) {
      row[kOffB1 + u] = b1;
      row[kOffB2 + u] = b2;
      row[kOffW3 + u] = w3;
#pragma unroll
      for (int i = 0; i < kMlpIn; i++) row[kOffW1 + u * kMlpIn + i] = w1[i];
    }
  }
  gb3 = over_c(gb3);
  lsum = over_c(lsum);
  if (lane < kOffW1) row[lane] = 0.0f;
  if (lane == 0) {
    row[kOffB3] = gb3;
    row[kMlpParams] = lsum;
  }
  __syncthreads();
  for (int p = tid; p < kGradRow; p += 64 * kGradWaves) {
    float v = sum[0][p];
    for (int k = 1; k < kGradWaves; k++) v += sum[k][p];
    a.part[(size_t)blockIdx.x * kGradRow + p] = v;
  }
}

// Sums the blocks' rows: grad set, the loss (lscale times the squared errors)
// added to.  32 parameters x 8 row groups per block.
__global__ void __launch_bounds__(256) mlp_grad_sum_kernel(const float* __restrict__ part, int nrow,
                                                           float* __restrict__ grad, float* __restrict__ loss,
                                                           float lscale) {
  __shared__ float s[8][33];
  const int c = threadIdx.x & 31, q = threadIdx.x >> 5, p = blockIdx.x * 32 + c;
  float v = 0.0f;
  if (p < kGradRow) {
#pragma unroll 8
    for (int r = q; r < nrow; r += 8) v += part[(size_t)r * kGradRow + p];
  }
  s[q][c] = v;
  __syncthreads();
  if (q == 0 && p < kGradRow) {
    for (int k = 1; k < 8; k++) v += s[k][c];
    if (p < kMlpParams) grad[p] = v;
    else loss[0] += v * lscale;
  }
}

__global__ void __launch_bounds__(256) mlp_fill_kernel(float* __restrict__ p, int n) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = 0.0f;
}

// Adam (Kingma & Ba 2015) on the trainable entries of P (all but the
// standardisation constants), bias-corrected, step t >= 1.
__global__ void __launch_bounds__(256) mlp_adam_kernel(float* __restrict__ P, const float* __restrict__ g,
                                                       float* __restrict__ m1, float* __restrict__ m2, float lr,
                                                       float c1, float c2) {
  const int t = kOffW1 + blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= kMlpParams) return;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float gi = g[t];
  const float u = b1 * m1[t] + (1.0f - b1) * gi;
  const float v = b2 * m2[t] + (1.0f - b2) * gi * gi;
  m1[t] = u;
  m2[t] = v;
  P[t] -= lr * (u / c1) / (sqrtf(v / c2) + eps);
}

namespace {

struct DevBuf {
  void* p = nullptr;
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
  template <class T>
  T* alloc(size_t n) {
    if (hipMalloc(&p, std::max<size_t>(n, 1) * sizeof(T)) != hipSuccess) p = nullptr;
    return (T*)p;
  }
};

struct Stream {
  hipStream_t s = nullptr;
  Stream() {  // s stays null on failure, which the callers check
    if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess) s = nullptr;
  }
  ~Stream() {
    if (s) (void)hipStreamDestroy(s);
  }
};

int hip_ok(hipError_t e, const char* what, std::string& err) {
  if (e == hipSuccess) return 0;
  err = std::string(what) + ": " + hipGetErrorString(e);
  return 1;
}

void pack_on(hipStream_t s, const float* P, MlpDev* m) {
  hipLaunchKernelGGL(mlp_pack_kernel, dim3(16), dim3(256), 0, s, P, m);
}

// grad: kMlpParams words and, behind them, the rows of the blocks' sums
size_t grad_words(long count) { return kMlpParams + (size_t)grad_blocks(count) * kGradRow; }

void grad_on(hipStream_t s, const MlpDev* m, const float* feat, const float* target, const int* idx, long first,
             long count, float lscale, float* grad, float* loss) {
  GradArgs a;
  a.m = m; a.feat = feat; a.target = target; a.idx = idx; a.first = first; a.count = count;
  a.gscale = 2.0f / (float)count;
  a.part = grad + kMlpParams;
  const int grid = grad_blocks(count);
  if (grid > 0) hipLaunchKernelGGL(mlp_grad_kernel, dim3(grid), dim3(64 * kGradWaves), 0, s, a);
  hipLaunchKernelGGL(mlp_grad_sum_kernel, dim3((kGradRow + 31) / 32), dim3(256), 0, s, a.part, grid, grad, loss, lscale);
}

}  // namespace

int mlp_upload(Ctx& c, const float* blob, long n) {
  if (n != kMlpParams) return 1;
  MlpDev h;
  mlp_pack(blob, &h);
  if (!c.mlp_dev && hipMalloc(&c.mlp_dev, sizeof(MlpDev)) != hipSuccess) {
    c.mlp_dev = nullptr;
    return 1;
  }
  return hipMemcpy(c.mlp_dev, &h, sizeof(MlpDev), hipMemcpyHostToDevice) != hipSuccess;
}

namespace {
constexpr int kScratchDevices = 64;
void* g_scratch_dev[kScratchDevices] = {};  // device address of `scratch` on each GPU
std::mutex g_scratch_mu;
}  // namespace

// The address of this GPU's `scratch`, looked up once per device with that
// device current (the host symbol is only a stand-in for the device array).
int mlp_scratch_address(void** ptr, std::string& err) {
  int dev = 0;
  if (hip_ok(hipGetDevice(&dev), "hipGetDevice", err)) return 1;
  if (dev < 0 || dev >= kScratchDevices) { err = "device index out of range for the scratch table"; return 1; }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_dev[dev]) {
    void* p = nullptr;
    if (hip_ok(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)", err)) return 1;
    g_scratch_dev[dev] = p;
  }
  *ptr = g_scratch_dev[dev];
  return 0;
}

// cgfdm_mlp_forward with the caller's device arrays and the static scratch:
// the same pack and forward kernels, queued on `s`, no allocation.
int mlp_forward_noalloc_host(const float* P, const float* feat, long n, float* out, int mode, hipStream_t s,
                             std::string& err) {
  void* sp = nullptr;
  if (mlp_scratch_address(&sp, err)) return 1;
  MlpDev* m = (MlpDev*)sp;
  pack_on(s, P, m);
  if (n > 0) hipLaunchKernelGGL(mlp_forward_kernel, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, s, m, feat, n, out, mode);
  return hip_ok(hipGetLastError(), "mlp forward launch", err);
}

int mlp_forward_host(const float* blob, const float* feat, long n, float* out, int mode, std::string& err) {
  Stream st;
  DevBuf bP, bm, bf, bo;
  float* P = bP.alloc<float>(kMlpParams);
  MlpDev* m = bm.alloc<MlpDev>(1);
  float* f = bf.alloc<float>(4 * n);
  float* o = bo.alloc<float>(n);
  if (!st.s || !P || !m || !f || !o) { err = "hipMalloc failed"; return 1; }
  if (hip_ok(hipMemcpyAsync(P, blob, kMlpParams * sizeof(float), hipMemcpyHostToDevice, st.s), "copy", err)) return 1;
  if (n > 0 && hip_ok(hipMemcpyAsync(f, feat, 4 * n * sizeof(float), hipMemcpyHostToDevice, st.s), "copy", err)) return 1;
  pack_on(st.s, P, m);
  if (n > 0) hipLaunchKernelGGL(mlp_forward_kernel, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, st.s, m, f, n, o, mode);
  if (n > 0 && hip_ok(hipMemcpyAsync(out, o, n * sizeof(float), hipMemcpyDeviceToHost, st.s), "copy", err)) return 1;
  return hip_ok(hipStreamSynchronize(st.s), "mlp forward", err);
}

int mlp_grad_host(const float* blob, const float* feat, const float* target, long n, float* grad, float* loss,
                  std::string& err) {
  Stream st;
  DevBuf bP, bm, bf, bt, bg, bl;
  float* P = bP.alloc<float>(kMlpParams);
  MlpDev* m = bm.alloc<MlpDev>(1);
  float* f = bf.alloc<float>(4 * n);
  float* t = bt.alloc<float>(n);
  float* g = bg.alloc<float>(grad_words(n));
  float* l = bl.alloc<float>(1);
  if (!st.s || !P || !m || !f || !t || !g || !l) { err = "hipMalloc failed"; return 1; }
  if (hip_ok(hipMemcpyAsync(P, blob, kMlpParams * sizeof(float), hipMemcpyHostToDevice, st.s), "copy", err) ||
      hip_ok(hipMemcpyAsync(f, feat, 4 * n * sizeof(float), hipMemcpyHostToDevice, st.s), "copy", err) ||
      hip_ok(hipMemcpyAsync(t, target, n * sizeof(float), hipMemcpyHostToDevice, st.s), "copy", err))
    return 1;
  pack_on(st.s, P, m);
  hipLaunchKernelGGL(mlp_fill_kernel, dim3(1), dim3(64), 0, st.s, l, 1);
  grad_on(st.s, m, f, t, nullptr, 0, n, 1.0f / (float)n, g, l);
  if (hip_ok(hipMemcpyAsync(grad, g, kMlpParams * sizeof(float), hipMemcpyDeviceToHost, st.s), "copy", err) ||
      hip_ok(hipMemcpyAsync(loss, l, sizeof(float), hipMemcpyDeviceToHost, st.s), "copy", err))
    return 1;
  return hip_ok(hipStreamSynchronize(st.s), "mlp grad", err);
}

int mlp_train_host(float* blob, const float* feat, const float* target, long n, int epochs, int batch, float lr,
                   unsigned seed, float* loss_hist, std::string& err) {
  Stream st;
  DevBuf bP, bm, bf, bt, bg, bl, bm1, bm2, bi;
  float* P = bP.alloc<float>(kMlpParams);
  MlpDev* m = bm.alloc<MlpDev>(1);
  float* f = bf.alloc<float>(4 * n);
  float* t = bt.alloc<float>(n);
  float* g = bg.alloc<float>(grad_words(std::min<long>(batch, n)));
  float* l = bl.alloc<float>(epochs);
  float* m1 = bm1.alloc<float>(kMlpParams);
  float* m2 = bm2.alloc<float>(kMlpParams);
  int* idx = bi.alloc<int>(n);
  if (!st.s || !P || !m || !f || !t || !g || !l || !m1 || !m2 || !idx) { err = "hipMalloc failed"; return 1; }
  if (hip_ok(hipMemcpyAsync(P, blob, kMlpParams * sizeof(float), hipMemcpyHostToDevice, st.s), "copy", err) ||
      hip_ok(hipMemcpyAsync(f, feat, 4 * n * sizeof(float), hipMemcpyHostToDevice, st.s), "copy", err) ||
      hip_ok(hipMemcpyAsync(t, target, n * sizeof(float), hipMemcpyHostToDevice, st.s), "copy", err))
    return 1;
  const int fb = (kMlpParams + 255) / 256;
  hipLaunchKernelGGL(mlp_fill_kernel, dim3(fb), dim3(256), 0, st.s, m1, kMlpParams);
  hipLaunchKernelGGL(mlp_fill_kernel, dim3(fb), dim3(256), 0, st.s, m2, kMlpParams);
  hipLaunchKernelGGL(mlp_fill_kernel, dim3((epochs + 255) / 256), dim3(256), 0, st.s, l, epochs);
  std::mt19937 rng(seed);
  std::vector<int> perm(n);
  for (long i = 0; i < n; i++) perm[i] = (int)i;
  long step = 0;
  const double beta1 = 0.9, beta2 = 0.999;  // as in mlp_adam_kernel
  for (int e = 0; e < epochs; e++) {
    // cosine decay of the step size from lr to lr/20 over the epochs
    const double ph = epochs > 1 ? (double)e / (epochs - 1) : 0.0;
    const float lr_e = (float)(lr * (0.05 + 0.95 * 0.5 * (1.0 + std::cos(3.141592653589793 * ph))));
    std::shuffle(perm.begin(), perm.end(), rng);
    // the order buffer is rewritten only after the previous epoch's kernels have read it
    if (hip_ok(hipStreamSynchronize(st.s), "mlp train", err) ||
        hip_ok(hipMemcpyAsync(idx, perm.data(), n * sizeof(int), hipMemcpyHostToDevice, st.s), "copy", err))
      return 1;
    for (long first = 0; first < n; first += batch) {
      const long cnt = std::min<long>(batch, n - first);
      pack_on(st.s, P, m);
      grad_on(st.s, m, f, t, idx, first, cnt, 1.0f / (float)n, g, l + e);
      step++;
      const float c1 = (float)(1.0 - std::pow(beta1, (double)step)), c2 = (float)(1.0 - std::pow(beta2, (double)step));
      hipLaunchKernelGGL(mlp_adam_kernel, dim3((kMlpParams - kOffW1 + 255) / 256), dim3(256), 0, st.s, P, g, m1, m2,
                         lr_e, c1, c2);
    }
  }
  if (hip_ok(hipGetLastError(), "mlp train launch", err) ||
      hip_ok(hipMemcpyAsync(blob, P, kMlpParams * sizeof(float), hipMemcpyDeviceToHost, st.s), "copy", err) ||
      hip_ok(hipMemcpyAsync(loss_hist, l, epochs * sizeof(float), hipMemcpyDeviceToHost, st.s), "copy", err))
    return 1;
  return hip_ok(hipStreamSynchronize(st.s), "mlp train", err);
}

}  // namespace cgfdm
