// Wave stage kernel of the CGFDM time step for CDNA4 (gfx950): the
// HBM-bound hot path.
//
// One fused kernel computes the velocity-stress RHS on the curvilinear grid
// (wave_deriv_cu, wave.cu:8-494), adds the ADE-PML terms and advances their
// auxiliary fields (abs_deriv_{x,y,z}_cu, pml{x,y,z}.cu), applies the RK4
// stage combine (wave_rk_cu/RK_Syn, rk4.cu:20-33,154-257) and the Cerjan
// sponge (apply_cerjan_cu, cerjan.cu:166-200), reading each wavefield word
// once from HBM.
//
// Work decomposition: a block owns a TJ x TK tile of (j,k) columns and
// streams a chunk of i planes (i is the fault-normal, slowest axis).  The
// five planes the x-stencil needs sit in a per-thread register queue; the
// current plane plus its y/z halo is staged in a double-buffered LDS tile,
// so each plane costs one barrier and the next plane's loads are in flight
// while the current plane is computed.  Blocks are numbered so that each
// XCD (and its private L2) receives a contiguous range of work items of one
// i-chunk, which keeps the k-halo rows of neighbouring tiles L2 hits.
//
// Addressing: every global access is a 32-bit byte offset from a
// wave-uniform field base, so one VGPR addresses all 9 wave fields and the
// metric fields of a point (the grid is limited to 2^30 points).
//
// Points of the fault slab (i0-3..i0+3 without i0) keep their RHS in a slab
// buffer so the split-node kernels can overwrite it (fault_dvelo/
// fault_dstrs) before fault_post advances the slab.
//
// This header holds the stage kernels and their launchers; each
// wave_stage_<metric storage>.hip instantiates them for one metric storage
// type (so the three compile in parallel), and wave_stage.hip builds the
// work lists and calls them.
#pragma once
#include "fd_ops.h"
#include <algorithm>
#include <type_traits>
#include <vector>

namespace cgfdm {
namespace wave {
using namespace fd;


constexpr int NTHR = 512;  // threads per block
constexpr int TJ = 64;     // default tile: one wavefront per k-row, j contiguous
constexpr int TK = NTHR / TJ;
constexpr int TJN = 32;    // narrow tile for the absorbing bands along j (32 j x 8 k)
constexpr int NTHRN = 256;  // threads per block of the narrow tiles
constexpr int TKN = NTHRN / TJN;
constexpr int TJB = 20;    // exact-width tiles of the absorbing bands along j when they are at most 20
constexpr int TKB = 12;    // columns wide (20 x 12, 240 threads; the 20-layer PML and sponge)
constexpr int TK6 = 6;     // rows of the 64 x 6 interior tiles (WaveInteriorKernel 2)
constexpr int TK4 = 4;     // rows of the 64 x 4 interior tiles (WaveInteriorKernel 3)
constexpr int kPmlBoxInts = 8;  // ints of one box of the auxiliary update


// Volume arrays are plane-interleaved with padded rows: word (field c,
// padded plane x, column jk = jpad + j + k*py) sits at (x*nf + c)*pyz + jk,
// nf = 9 for wavefields, 13 for the metric (16 in its bfloat16-deviation form); py
// is a multiple of 32 words.  A plane of an array is addressed as one buffer resource
// (base = the plane's first word, range = the plane's bytes) with the lane's
// column byte offset as voffset and the field's offset c*nyz*size as
// soffset: no per-lane 64-bit address arithmetic, a handful of scalar
// registers per plane, and one block touches few memory pages per plane.
// Word 3 of the resource is the gfx9-family default (32-bit data, no swizzle).
constexpr int kBufWord3 = 0x00020000;
typedef __amdgpu_buffer_rsrc_t Rsrc;
template <class T>
__device__ __forceinline__ Rsrc plane_rsrc(const T* a, int plane, uint32_t nf, uint32_t nyz) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(a) + (size_t)plane * nf * nyz, (short)0,
                                           (int)(nf * nyz * (uint32_t)sizeof(T)), kBufWord3);
}
// Cache policy of an access: kReuse for stage-input words that neighbouring
// tiles read again (halo rows and columns, the x-queue warm-up), kStream
// (non-temporal) for words touched once per stage, so they do not push the
// reused rows out of the XCD's L2.
constexpr int kReuse = 0, kStream = 2;
template <int POL = kReuse>
__device__ __forceinline__ float bld(Rsrc r, uint32_t voff, uint32_t soff) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, POL));
}
template <int POL = kStream>
__device__ __forceinline__ void bst(Rsrc r, uint32_t voff, uint32_t soff, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, (int)voff, (int)soff, POL);
}
template <class MT>
__device__ __forceinline__ float bldm(Rsrc r, uint32_t voff, uint32_t soff) {
  if constexpr (sizeof(MT) == 2) {
    const unsigned short v = __builtin_amdgcn_raw_buffer_load_b16(r, (int)voff, (int)soff, kStream);
    return __uint_as_float(((unsigned)v) << 16);
  } else {
    return bld<kStream>(r, voff, soff);
  }
}
// The auxiliary arrays of an absorbing face hold, for each of its planes pi,
// nine fields of pnk x pnj words (pp): word (c, pi, pk, pj) at
// pi*stride + c*pp + pk*pnj + pj.  The two faces of an axis share an array:
// along x the high face's planes follow the low face's, along y and z the
// high face's nine fields follow the low face's within each plane.  The
// plane index is uniform in a block, so one plane of an axis is one buffer
// resource (its low face's base, np nine-field parts long), addressed like a
// plane of the volume arrays, with a lane's side in its byte offset.
__device__ __forceinline__ Rsrc aux_rsrc(const float* a, int pi, uint32_t pp, uint32_t np) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a) + (size_t)pi * np * 9 * pp, (short)0, (int)(np * 9 * pp * 4),
                                           kBufWord3);
}
// A uniform word of an array that no kernel writes (the 1-D profiles): a
// scalar load, which does not queue behind the vector loads in flight.
__device__ __forceinline__ float uni(const float* p, int i) {
  return ((const __attribute__((address_space(4))) float*)p)[i];
}
// The same uniform value, with what is computed from it kept at its use: the
// eight field offsets of each auxiliary array, taken out of the plane loop,
// do not fit the scalar registers and were read back from vector lanes (866
// v_readlane in the loop of the 64 x 4 band tiles).
template <class V>
__device__ __forceinline__ V here(V v) {
  asm volatile("" : "+s"(v));
  return v;
}
// A byte offset past the end of every buffer resource: a load there returns 0
// and a store is dropped, without memory traffic.
constexpr uint32_t kNoWord = 0xfffffff0u;
// Word of field c at padded plane x, column jk (plain loads, off the hot path).
__device__ __forceinline__ float wat(const float* W, int c, int x, uint32_t jk, uint32_t nyz) {
  return W[((size_t)x * 9 + c) * nyz + jk];
}
__device__ __forceinline__ float mat_(const float* M, int c, int x, uint32_t jk, uint32_t nyz, const float*) {
  return M[((size_t)x * 13 + c) * nyz + jk];
}
__device__ __forceinline__ float mat_(const uint16_t* M, int c, int x, uint32_t jk, uint32_t nyz, const float*) {
  return __uint_as_float(((unsigned)M[((size_t)x * 13 + c) * nyz + jk]) << 16);
}
// Metric in bfloat16 with the media words exact (18 16-bit slots per
// plane): the bfloat16 of each metric word's deviation from a reference
// value of its field (ref[c], the midrange of the field over the grid), so
// the rounding scales with the field's variation rather than its size,
// packed two to a 32-bit word (slots 2p and 2p+1 form 32-bit plane p, field
// 2p in the low half).  Slots 0-8 hold the nine metric coefficients, slot 9
// the point's entry in the media palette (lambda, mu, rho of the few
// distinct media of a layered or two-half model, see WaveArgs::pal; 0 when
// the media have no palette), slots 10-15 lambda, mu and rho as three FP32
// planes, slot 16 the Jacobian (its deviation, field 9 of ref), slot 17 0.
struct MetBf16Delta {
  uint16_t h;
};
constexpr uint32_t kMetDeltaSlots = 18;
constexpr uint32_t kMetDeltaJac = 16;  // slot of the Jacobian
template <class MT>
constexpr uint32_t met_nf() {
  return std::is_same<MT, MetBf16Delta>::value ? kMetDeltaSlots : 13u;
}
__device__ __forceinline__ float mat_(const MetBf16Delta* Ms, int c, int x, uint32_t jk, uint32_t nyz, const float* ref) {
  const uint16_t* M = &Ms->h;
  if (c < 10) {  // field c of the pair at slot c & ~1 (c < 9), or the Jacobian in the low half at its slot
    const uint32_t s = c == 9 ? kMetDeltaJac : (uint32_t)(c & ~1);
    const uint32_t u = ((const uint32_t*)(M + ((size_t)x * kMetDeltaSlots + s) * nyz))[jk];
    return __uint_as_float((c < 9 && (c & 1)) ? (u & 0xffff0000u) : (u << 16)) + ref[c];
  }
  return ((const float*)(M + ((size_t)x * kMetDeltaSlots + 10) * nyz))[(size_t)(c - 10) * nyz + jk];
}
// Field c (a metric coefficient 0..8 or a media word 10..12) of a metric
// plane resource r at byte column voff (mpb bytes a field); ref is the
// field's reference value in the deviation form.
template <class MT>
__device__ __forceinline__ float bldmc(Rsrc r, uint32_t voff, int c, uint32_t mpb, float ref) {
  if constexpr (std::is_same<MT, MetBf16Delta>::value) {
    if (c >= 10) return bld<kStream>(r, 2 * voff, (uint32_t)(10 + 2 * (c - 10)) * mpb);  // FP32 word
    const uint32_t u = __float_as_uint(bld<kStream>(r, 2 * voff, (uint32_t)(c & ~1) * mpb));  // pair of c
    return __uint_as_float((c & 1) ? (u & 0xffff0000u) : (u << 16)) + ref;
  }
  return bldm<MT>(r, voff, c * mpb);
}

// RK_Syn combine (rk4.cu:20-33) of field c of the planes rs (S) and rt (T).
// Stage 0 sets the accumulator T = S + (dt/6) h0 beside the stage value
// W1 = S + (dt/2) h0, so T = S + (W1 - S) / 3: stage 1, which reads S and
// W1 anyway, derives it (to FP32 rounding) instead of stage 0 writing it and
// stage 1 reading it, 18 of the 144 wavefield words of a step.  A point
// whose stage-0 value changes after the combine (Cerjan-damped, or on the
// fault plane, where fault2wave rewrites it) keeps the stored accumulator:
// keep_t.  The same point takes the same branch in every stage.
__device__ __forceinline__ float rk_derived_t(float s, float w1) { return s + (w1 - s) * (1.0f / 3.0f); }
__device__ __forceinline__ float rk_combine_b(int irk, float rka, float rkb, float w, float h, Rsrc rs, Rsrc rt,
                                              uint32_t voff, uint32_t soff, bool keep_t) {
  if (irk == 0) {
    if (keep_t) bst(rt, voff, soff, w + rkb * h);
    return w + rka * h;
  }
  if (irk == 3) return bld<kStream>(rt, voff, soff) + rkb * h;
  const float s = bld<kStream>(rs, voff, soff);
  const float t = irk == 1 && !keep_t ? rk_derived_t(s, w) : bld<kStream>(rt, voff, soff);
  bst(rt, voff, soff, t + rkb * h);
  return s + rka * h;
}

template <class MT>
struct WaveArgs {
  const float* __restrict__ Win;
  float* __restrict__ Wout;
  const float* __restrict__ S;
  float* __restrict__ T;
  const MT* __restrict__ met;
  float* __restrict__ slabH;
  float* __restrict__ rhs;
  float* itop;  // what the surface rows need of the free-surface image, [ni][18][nj] (image_top_kernel)
  WaveCold cold;  // absorbing layers and free-surface maps, indexed with constants only
  const int4* __restrict__ work;  // two int4 per block: (j0, k0, first plane, end plane), (j lanes, k rows, first active j lane, first active k row)
  unsigned nyz;                   // words of one field of one plane (py*nz, padded rows)
  int py, jpad;                   // row pitch and front pad of volume rows
  int nwork, ni, nj, nk, ny, ii0;
  float rDH, rka, rkb;
  float mref[10];   // metric reference values (bfloat16-deviation form)
  // bfloat16-deviation form: lambda, mu, rho (and 0) of each media palette
  // entry, or null when the media have no palette (the pipelined kernels
  // then read the FP32 media planes)
  const float4* __restrict__ pal;
  int npal;
  unsigned met_skip;  // bfloat16-deviation form: bit p set when 32-bit metric word p is +-0 on the whole grid
  int irk, freenode, cerjan, fault, rhs_only, pml;
  int aux_fused;  // BAND tiles advance their points' ADE-PML auxiliary fields themselves
};

// The conservative traction vector J (grad xi_ax . sigma) (wave.cu:398-440) of
// a point, from the stage input.
template <class MT>
__device__ __forceinline__ void trac_vec(const WaveArgs<MT>& a, int ax, int x, uint32_t q, float (&o)[3]) {
  const uint32_t nyz = a.nyz;
  const float* W = a.Win;
  const MT* M = a.met;
  const float J = mat_(M, 9, x, q, nyz, a.mref);
  const float txx = wat(W, 3, x, q, nyz), tyy = wat(W, 4, x, q, nyz), tzz = wat(W, 5, x, q, nyz);
  const float txy = wat(W, 6, x, q, nyz), txz = wat(W, 7, x, q, nyz), tyz = wat(W, 8, x, q, nyz);
  const float e0 = mat_(M, 3 * ax, x, q, nyz, a.mref), e1 = mat_(M, 3 * ax + 1, x, q, nyz, a.mref), e2 = mat_(M, 3 * ax + 2, x, q, nyz, a.mref);
  o[0] = (e0 * txx + e1 * txy + e2 * txz) * J;
  o[1] = (e0 * txy + e1 * tyy + e2 * tyz) * J;
  o[2] = (e0 * txz + e1 * tyz + e2 * tzz) * J;
}

// Free surface: the traction-image velocity RHS of the three top rows
// (wave.cu:398-487): DRP derivatives of the traction vectors along each axis,
// the z stencil zero at the surface and odd-mirrored above it, with the PML
// 1/beta of each axis, in planes 3 c + row of itop ([i][18][nj]), row = k -
// (nk-3).  For the top row also what its points need of the velocity maps
// (traction-free condition, wave.cu:207-232): the dip derivative of the
// velocity DzV = matVx2Vz DxV + matVy2Vz DyV in planes 9-11, and its two
// products alone (the source of the x and y faces' auxiliary fields,
// pmlx.cu:185-210) in planes 12-14 and 15-17.  In the stage tiles, short of
// registers, the 18 map words of a point were a chain of 18 memory round
// trips per plane.
// A point's 15 traction vectors are computed where they are used, all loads at
// once: bound by latency, and as a pass of its own, which wrote them for this
// one to read, it cost a launch per stage and a second round trip (ms of tiles
// and image per step at 30 x 80 x 50 0.135 -> 0.124, 100 x 200 x 100 0.449 ->
// 0.436; surface tiles and image at 800 x 1000 x 500 2.07 -> 1.98).
template <int FX, int FY, int FZ, class MT>
__global__ void __launch_bounds__(256) image_top_kernel(WaveArgs<MT> a) {
  const int ni = a.ni, nj = a.nj, nk = a.nk, ny = a.ny;
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)ni * 3 * nj) return;
  const int j = (int)(idx % nj);
  const int row = (int)((idx / nj) % 3);
  const int i = (int)(idx / ((long)nj * 3));
  const int k = nk - 3 + row, ik = 2 - row, x = i + 3;
  const uint32_t col = (uint32_t)a.jpad + (uint32_t)(j + 3) + (uint32_t)(k + 3) * (uint32_t)a.py;
  const MT* M = a.met;
  const uint32_t py = (uint32_t)a.py;
  const float rrhojac = 1.0f / (mat_(M, 12, x, col, a.nyz, a.mref) * mat_(M, 9, x, col, a.nyz, a.mref));
  float rb[3] = {1.0f, 1.0f, 1.0f};
  if (a.pml) {
    rb[0] = 1.0f / a.cold.pB[0][i];
    rb[1] = 1.0f / a.cold.pB[1][j];
    rb[2] = 1.0f / a.cold.pB[2][k];
  }
  const int fl[3] = {FX, FY, FZ};
  float hv[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int ax = 0; ax < 3; ax++) {
    float v[3][7];
#pragma unroll
    for (int l = 0; l < 7; l++) {
      const int xq = ax == 0 ? x + l - 3 : x;
      const int up = ax == 2 ? min(l - 3, 2 - row) : 0;  // rows above the surface: replaced below
      float o[3];
      trac_vec(a, ax, xq, col + (uint32_t)(ax == 1 ? l - 3 : 0) + (uint32_t)up * py, o);
#pragma unroll
      for (int c = 0; c < 3; c++) v[c][l] = o[c];
    }
    if (ax == 2) {
      for (int c = 0; c < 3; c++) {
        if (ik == 0) { v[c][3] = 0.0f; v[c][6] = -v[c][0]; v[c][5] = -v[c][1]; v[c][4] = -v[c][2]; }
        else if (ik == 1) { v[c][4] = 0.0f; v[c][6] = -v[c][2]; v[c][5] = -v[c][3]; }
        else { v[c][5] = 0.0f; v[c][6] = -v[c][4]; }
      }
    }
    for (int c = 0; c < 3; c++) {
      const float d = a.rDH * (fl[ax] > 0 ? drp5<1>(v[c][2], v[c][3], v[c][4], v[c][5], v[c][6])
                                          : drp5<-1>(v[c][0], v[c][1], v[c][2], v[c][3], v[c][4]));
      hv[c] += d * rb[ax];
    }
  }
  float* w = a.itop + (size_t)i * 18 * nj + j;
  for (int c = 0; c < 3; c++) w[(size_t)(c * 3 + row) * nj] = hv[c] * rrhojac;
  if (row == 2) {
    const float* mVx = a.cold.mVx + ((long)(j + 3) + (long)x * ny) * 9;
    const float* mVy = a.cold.mVy + ((long)(j + 3) + (long)x * ny) * 9;
    float dxv[3], dyv[3];
    for (int c = 0; c < 3; c++) {
      const float* v = a.Win + ((size_t)x * 9 + c) * a.nyz + col;
      const long st = 9L * a.nyz;
      dxv[c] = a.rDH * (FX > 0 ? drp5<1>(v[-st], v[0], v[st], v[2 * st], v[3 * st])
                               : drp5<-1>(v[-3 * st], v[-2 * st], v[-st], v[0], v[st]));
      dyv[c] = a.rDH * (FY > 0 ? drp5<1>(v[-1], v[0], v[1], v[2], v[3]) : drp5<-1>(v[-3], v[-2], v[-1], v[0], v[1]));
    }
    for (int r = 0; r < 3; r++) {
      w[(size_t)(9 + r) * nj] = mVx[3 * r] * dxv[0] + mVx[3 * r + 1] * dxv[1] + mVx[3 * r + 2] * dxv[2]
                               + mVy[3 * r] * dyv[0] + mVy[3 * r + 1] * dyv[1] + mVy[3 * r + 2] * dyv[2];
      w[(size_t)(12 + r) * nj] = mVx[3 * r] * dxv[0] + mVx[3 * r + 1] * dxv[1] + mVx[3 * r + 2] * dxv[2];
      w[(size_t)(15 + r) * nj] = mVy[3 * r] * dyv[0] + mVy[3 * r + 1] * dyv[1] + mVy[3 * r + 2] * dyv[2];
    }
  }
}

// Extra auxiliary-field source of the x/y PML faces on the free surface
// (pmlx.cu:185-210, pmly.cu): the z-derivative of velocity eliminated through
// the traction-free condition, component c in 3..8.
__device__ __forceinline__ float pml_fs_term(int c, const float* z1, float ztx, float zty, float ztz, float lam,
                                             float l2m, float mu, float c0) {
  if (c == 3) return c0 * (l2m * ztx * z1[0] + lam * zty * z1[1] + lam * ztz * z1[2]);
  if (c == 4) return c0 * (lam * ztx * z1[0] + l2m * zty * z1[1] + lam * ztz * z1[2]);
  if (c == 5) return c0 * (lam * ztx * z1[0] + lam * zty * z1[1] + l2m * ztz * z1[2]);
  if (c == 6) return c0 * mu * (zty * z1[0] + ztx * z1[1]);
  if (c == 7) return c0 * mu * (ztz * z1[0] + ztx * z1[2]);
  if (c == 8) return c0 * mu * (ztz * z1[1] + zty * z1[2]);
  return 0.0f;
}

// KIND selects the instantiation: 0 interior (no PML, free-surface or Cerjan
// code: the host gives it only points where every absorbing profile is
// trivial), 1 absorbing bands (PML correction, Cerjan), 2 tiles holding the
// free-surface rows (everything).
template <int FX, int FY, int FZ, class MT, int KIND, int TJ_ = TJ, int NT_ = NTHR>
__global__ void __launch_bounds__(NT_, KIND == 2 ? 2 : 4) wave_stage_kernel(WaveArgs<MT> a) {
  constexpr int TJ = TJ_, TK = NT_ / TJ_;  // tile of TJ (j) x TK (k) columns
  constexpr int LJ = TJ + 4, LK = TK + 4;   // LDS tile with halos
  constexpr int NH = 4 * LJ + 4 * TK;       // halo cells of one plane: 4 rows + 4 side cells per row
  static_assert(NH <= NT_, "one halo cell per thread");
  constexpr int HJL = FY > 0 ? 1 : 3;    // halo width below j (the stencil reaches HJL back, 4-HJL forward)
  constexpr int HKL = FZ > 0 ? 1 : 3;
  constexpr int QLO = FX > 0 ? -1 : -3;  // queue holds planes i+QLO .. i+QLO+4
  constexpr int CTR = -QLO;
  __shared__ float lds[2][9][LK][LJ];
  const int item = xcd_remap((int)blockIdx.x, a.nwork);
  const int4 wk = a.work[2 * item], we = a.work[2 * item + 1];
  const int j0 = wk.x, k0 = wk.y, ibeg = wk.z, iend = wk.w;
  const int tj = threadIdx.x, tk = threadIdx.y, tid = tj + tk * TJ;
  const int ni = a.ni, nj = a.nj, nk = a.nk, ny = a.ny;
  const int j = j0 + tj, k = k0 + tk;
  const bool act = tj >= we.z && tj < we.x && tk >= we.w && tk < we.y;
  const bool pml = KIND >= 1 && a.pml, cerjan = KIND >= 1 && a.cerjan;
  const int nxp = ni + 6;  // padded planes
  const uint32_t nyz = a.nyz;
  // Every lane loads (no predicated loads): lanes past the padded array read
  // a clamped in-bounds column whose value no active point ever uses.
  const uint32_t py = a.py, jpad = a.jpad;
  const uint32_t col = jpad + (uint32_t)(min(max(j, -3), nj + 2) + 3) + (uint32_t)(min(max(k, -3), nk + 2) + 3) * py;
  const uint32_t col4 = col << 2;
  const uint32_t mcol = col * (uint32_t)sizeof(MT);
  const uint32_t pb = nyz * 4, mpb = nyz * (uint32_t)sizeof(MT);  // bytes of one field of one plane
  const float* __restrict__ Win = a.Win;

  // this thread's halo cell: 4 full rows of LJ cells, then 4 side cells per row
  int hlk = 0, hlj = 0;
  uint32_t hcol = col;
  if (tid < NH) {
    if (tid < 4 * LJ) {
      const int r = tid / LJ;
      hlk = r < HKL ? r : r + TK;
      hlj = tid % LJ;
    } else {
      const int h2 = tid - 4 * LJ;
      hlk = HKL + h2 / 4;
      const int cc = h2 % 4;
      hlj = cc < HJL ? cc : cc + TJ;
    }
    const int gj = min(max(j0 + hlj - HJL, -3), nj + 2), gk = min(max(k0 + hlk - HKL, -3), nk + 2);
    hcol = jpad + (uint32_t)(gj + 3) + (uint32_t)(gk + 3) * py;
  }
  const uint32_t hcol4 = hcol << 2;

  // ADE-PML: the lane's byte offsets in a plane of its faces' auxiliary arrays
  // (low and high band along y and z, which may overlap; kNoWord outside a
  // band), and which of the four the wavefront has any lane in.  Found out in
  // the plane loop, face by face from the kernel's arguments, the flags, sizes
  // and bases were chains of scalar loads and 61 spilled scalar registers:
  // bands 2.98 -> 1.75 ms per step at 251 x 187 x 143 with WaveBandKernel 0,
  // 1.94 -> 1.05 at 30 x 80 x 50 with 20 layers, which overlap along x.
  float rb2 = 1.0f, rb3 = 1.0f, cjk = 1.0f;
  uint32_t xo4 = kNoWord, yo4[2] = {kNoWord, kNoWord}, zo4[2] = {kNoWord, kNoWord};
  const int N = KIND >= 1 ? a.cold.N : 0;
  const uint32_t xpp = (uint32_t)nk * nj, ypp = (uint32_t)nk * N, zpp = (uint32_t)N * nj;  // words of a field of a face plane
  const uint32_t nyf = KIND >= 1 ? a.cold.on[2] + a.cold.on[3] : 0, nzf = KIND >= 1 ? a.cold.on[4] + a.cold.on[5] : 0;
  if (act && pml) {
    rb2 = 1.0f / a.cold.pB[1][j];
    rb3 = 1.0f / a.cold.pB[2][k];
    xo4 = (uint32_t)(j + k * nj) << 2;
    if (a.cold.on[2] && j < N) yo4[0] = (uint32_t)(j + k * N) << 2;
    if (a.cold.on[3] && j >= nj - N) yo4[1] = ((uint32_t)(j - (nj - N) + k * N) + (a.cold.on[2] ? 9 * ypp : 0u)) << 2;
    if (a.cold.on[4] && k < N) zo4[0] = (uint32_t)(j + k * nj) << 2;
    if (a.cold.on[5] && k >= nk - N) zo4[1] = ((uint32_t)(j + (k - (nk - N)) * nj) + (a.cold.on[4] ? 9 * zpp : 0u)) << 2;
  }
  bool hasy[2], hasz[2];
#pragma unroll
  for (int side = 0; side < 2; side++) {
    hasy[side] = __builtin_amdgcn_ballot_w64(yo4[side] != kNoWord) != 0;
    hasz[side] = __builtin_amdgcn_ballot_w64(zo4[side] != kNoWord) != 0;
  }
  if (act && cerjan) cjk = fminf(a.cold.cj[1][j + 3], a.cold.cj[2][k + 3]);
  const int xend0 = pml && a.cold.on[0] ? N : 0;           // planes of the low x band end here,
  const int xbeg1 = pml && a.cold.on[1] ? ni - N : nxp;    // those of the high one begin here
  float pbx = pml ? uni(a.cold.pB[0], ibeg) : 1.0f;        // beta along x and the sponge factor of plane i
  float cjx = cerjan ? uni(a.cold.cj[0], ibeg + 3) : 1.0f;

  float q[5][9];
#pragma unroll
  for (int m = 0; m < 5; m++) {
    const Rsrc r = plane_rsrc(Win, ibeg + QLO + m + 3, 9, nyz);
#pragma unroll
    for (int c = 0; c < 9; c++) q[m][c] = bld(r, col4, c * pb);
  }
  float hv[9];
  {
    const Rsrc r = plane_rsrc(Win, ibeg + 3, 9, nyz);
#pragma unroll
    for (int c = 0; c < 9; c++) hv[c] = bld(r, hcol4, c * pb);
  }
#pragma unroll
  for (int c = 0; c < 9; c++) lds[0][c][tk + HKL][tj + HJL] = q[CTR][c];
  if (tid < NH) {
#pragma unroll
    for (int c = 0; c < 9; c++) lds[0][c][hlk][hlj] = hv[c];
  }
  __syncthreads();

  typedef const __attribute__((address_space(4))) WaveArgs<MT>* ArgPtr;
  const ArgPtr kargs = (ArgPtr)__builtin_amdgcn_kernarg_segment_ptr();  // the argument a
  for (int i = ibeg; i < iend; ++i) {
    const ArgPtr ap = KIND >= 1 ? here(kargs) : kargs;  // as in wave_interior_kernel
    const int b = (i - ibeg) & 1;
    const bool more = i + 1 < iend;  // uniform per block
    // next plane of the queue and the halo of plane i+1, in flight during the compute
    // (planes clamped in-bounds: past the chunk's end the values go unused)
    float nq[9];
    {
      const Rsrc r = plane_rsrc(Win, min(i + QLO + 8, nxp - 1), 9, nyz);
#pragma unroll
      for (int c = 0; c < 9; c++) nq[c] = bld(r, col4, c * pb);
    }
    {
      const Rsrc r = plane_rsrc(Win, min(i + 4, nxp - 1), 9, nyz);
#pragma unroll
      for (int c = 0; c < 9; c++) hv[c] = bld(r, hcol4, c * pb);
    }
    const float pbxn = pml && more ? uni(a.cold.pB[0], i + 1) : 1.0f;
    const float cjxn = cerjan && more ? uni(a.cold.cj[0], i + 4) : 1.0f;

    if (act) {
      const Rsrc rm = plane_rsrc(ap->met, i + 3, met_nf<MT>(), nyz);
      auto MET = [&](int c) { return bldmc<MT>(rm, mcol, c, mpb, c < 10 ? a.mref[c] : 0.0f); };
      const float xix = MET(0), xiy = MET(1), xiz = MET(2);
      const float etx = MET(3), ety = MET(4), etz = MET(5);
      const float ztx = MET(6), zty = MET(7), ztz = MET(8);
      const float lam = MET(10), mu = MET(11);
      const float rrho = 1.0f / MET(12);
      const float l2m = lam + 2.0f * mu;
      const float rDH = ap->rDH;
      const float rb1 = pml ? 1.0f / pbx : 1.0f;
      const float(*L)[LK][LJ] = lds[b];
      const int lj = tj + HJL, lk = tk + HKL;
      // one-sided DRP difference of field c along each axis (macdrp.h:91-95),
      // without the 1/DH factor (folded into the metric rows below)
      auto Dx = [&](int c) { return drp5<FX>(q[0][c], q[1][c], q[2][c], q[3][c], q[4][c]); };
      auto Dy = [&](int c) {
        return FY > 0 ? drp5<1>(L[c][lk][lj - 1], L[c][lk][lj], L[c][lk][lj + 1], L[c][lk][lj + 2], L[c][lk][lj + 3])
                      : drp5<-1>(L[c][lk][lj - 3], L[c][lk][lj - 2], L[c][lk][lj - 1], L[c][lk][lj], L[c][lk][lj + 1]);
      };
      auto Dz = [&](int c) {
        return FZ > 0 ? drp5<1>(L[c][lk - 1][lj], L[c][lk][lj], L[c][lk + 1][lj], L[c][lk + 2][lj], L[c][lk + 3][lj])
                      : drp5<-1>(L[c][lk - 3][lj], L[c][lk - 2][lj], L[c][lk - 1][lj], L[c][lk][lj], L[c][lk + 1][lj]);
      };
      const bool top = KIND == 2 && ap->freenode && k >= nk - 3;  // uniform per wavefront (one k-row)
      // RHS accumulated derivative by derivative (wave.cu:133-276): each
      // field's derivative adds its momentum / Hooke terms, metric rows
      // pre-scaled by the PML 1/beta of their axis.
      float h[9];
#pragma unroll
      for (int c = 0; c < 9; c++) h[c] = 0.0f;
      {
        const float s1 = rb1 * rDH, s2 = rb2 * rDH, s3 = rb3 * rDH;
        accum_axis(h, Dx, xix * s1, xiy * s1, xiz * s1, rrho, lam, l2m, mu, true);
        accum_axis(h, Dy, etx * s2, ety * s2, etz * s2, rrho, lam, l2m, mu, true);
        accum_axis(h, Dz, ztx * s3, zty * s3, ztz * s3, rrho, lam, l2m, mu, !top);
      }
      if (top) {
        float dzv[3];
        if (k == nk - 1) {  // DzV from the traction-free condition (wave.cu:207-232)
          const uint32_t ij = ((uint32_t)(j + 3) + (uint32_t)(i + 3) * (uint32_t)ny) * 9;
          const float* mVx = ap->cold.mVx;
          const float* mVy = ap->cold.mVy;
          const float dxv[3] = {rDH * Dx(0), rDH * Dx(1), rDH * Dx(2)}, dyv[3] = {rDH * Dy(0), rDH * Dy(1), rDH * Dy(2)};
#pragma unroll
          for (int r = 0; r < 3; r++)
            dzv[r] = mVx[ij + 3 * r] * dxv[0] + mVx[ij + 3 * r + 1] * dxv[1] + mVx[ij + 3 * r + 2] * dxv[2]
                   + mVy[ij + 3 * r] * dyv[0] + mVy[ij + 3 * r + 1] * dyv[1] + mVy[ij + 3 * r + 2] * dyv[2];
        } else if (k == nk - 2) {  // L22 (wave.cu:233-238)
#pragma unroll
          for (int c = 0; c < 3; c++) dzv[c] = rDH * (FZ > 0 ? L[c][lk + 1][lj] - L[c][lk][lj] : L[c][lk][lj] - L[c][lk - 1][lj]);
        } else {  // L24 (wave.cu:239-245)
#pragma unroll
          for (int c = 0; c < 3; c++)
            dzv[c] = rDH * (FZ > 0 ? -C24_1 * L[c][lk][lj] + C24_2 * L[c][lk + 1][lj] - C24_3 * L[c][lk + 2][lj]
                                   : C24_3 * L[c][lk - 2][lj] - C24_2 * L[c][lk - 1][lj] + C24_1 * L[c][lk][lj]);
        }
        const float e0 = ztx * rb3, e1 = zty * rb3, e2 = ztz * rb3;
        h[3] += (l2m * e0 * dzv[0] + lam * e1 * dzv[1] + lam * e2 * dzv[2]);
        h[4] += (lam * e0 * dzv[0] + l2m * e1 * dzv[1] + lam * e2 * dzv[2]);
        h[5] += (lam * e0 * dzv[0] + lam * e1 * dzv[1] + l2m * e2 * dzv[2]);
        h[6] += (e1 * dzv[0] + e0 * dzv[1]) * mu;
        h[7] += (e2 * dzv[0] + e0 * dzv[2]) * mu;
        h[8] += (e2 * dzv[1] + e1 * dzv[2]) * mu;
        {  // the image velocity RHS (image_top_kernel)
          const float* w = ap->itop + ((size_t)i * 18 + (k - (nk - 3))) * nj + j;
#pragma unroll
          for (int c = 0; c < 3; c++) h[c] = w[(size_t)c * 3 * nj];
        }
      }

      // ADE-PML (pmlx.cu:126-210 and the y/z variants): the RHS of a point
      // inside the band of face f gets -aux_f/beta; the auxiliary fields
      // themselves are advanced afterwards by pml_aux_kernel from the same
      // stage input.
      // (a lane without the face adds 0: each face of an axis for all lanes)
      if (pml) {
        auto face = [&](Rsrc r, uint32_t o, uint32_t fb, float rbb) {
          float v[9];
#pragma unroll
          for (int c = 0; c < 9; c++) v[c] = bld(r, o, c * fb);
#pragma unroll
          for (int c = 0; c < 9; c++) h[c] += -v[c] * rbb;
        };
        if (i < xend0) face(aux_rsrc(ap->cold.axY[0], i, xpp, 1), xo4, here(4 * xpp), rb1);
        if (i >= xbeg1) face(aux_rsrc(ap->cold.axY[0], i - xbeg1 + xend0, xpp, 1), xo4, here(4 * xpp), rb1);
        if (hasy[0]) face(aux_rsrc(ap->cold.axY[1], i, ypp, nyf), yo4[0], here(4 * ypp), rb2);
        if (hasy[1]) face(aux_rsrc(ap->cold.axY[1], i, ypp, nyf), yo4[1], here(4 * ypp), rb2);
        if (hasz[0]) face(aux_rsrc(ap->cold.axY[2], i, zpp, nzf), zo4[0], here(4 * zpp), rb3);
        if (hasz[1]) face(aux_rsrc(ap->cold.axY[2], i, zpp, nzf), zo4[1], here(4 * zpp), rb3);
      }

      if (ap->rhs_only) {
#pragma unroll
        for (int c = 0; c < 9; c++) bst(plane_rsrc(ap->rhs, i + 3, 9, nyz), col4, c * pb, h[c]);
      } else if (ap->fault && i >= ap->ii0 - 3 && i <= ap->ii0 + 3 && i != ap->ii0) {
        const Rsrc r = plane_rsrc(ap->slabH, i - (ap->ii0 - 3), 9, nyz);  // slab planes share the layout
#pragma unroll
        for (int c = 0; c < 9; c++) bst(r, col4, c * pb, h[c]);
      } else {
        const float damp = cerjan ? fminf(cjx, cjk) : 1.0f;
        const bool keep_t = damp != 1.0f || (ap->fault && i == ap->ii0);
        const Rsrc rs = plane_rsrc(ap->S, i + 3, 9, nyz), rt = plane_rsrc(ap->T, i + 3, 9, nyz);
        const Rsrc ro = plane_rsrc(ap->Wout, i + 3, 9, nyz);
#pragma unroll
        for (int c = 0; c < 9; c++) {
          const float w = rk_combine_b(ap->irk, ap->rka, ap->rkb, q[CTR][c], h[c], rs, rt, col4, c * pb, keep_t);
          bst(ro, col4, c * pb, w * damp);
        }
      }
    }

    if (more) {  // stage plane i+1 into the other LDS buffer
#pragma unroll
      for (int c = 0; c < 9; c++) lds[b ^ 1][c][tk + HKL][tj + HJL] = q[CTR + 1][c];
      if (tid < NH) {
#pragma unroll
        for (int c = 0; c < 9; c++) lds[b ^ 1][c][hlk][hlj] = hv[c];
      }
    }
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
      for (int c = 0; c < 9; c++) q[m][c] = q[m + 1][c];
#pragma unroll
    for (int c = 0; c < 9; c++) q[4][c] = nq[c];
    pbx = pbxn;
    cjx = cjxn;
    __syncthreads();
  }
}


// Raw metric words of one point (MetricBF16=2: five 32-bit pairs of bfloat16
// deviations, the fifth with the palette entry in its high half, and, when
// the media have no palette, the FP32 lambda, mu, rho; FP32: the 12 words
// xix..ztz, lam, mu, rho; bfloat16: the same 12 as 16-bit words), held
// undecoded while they wait for their plane.
template <class MT>
constexpr int met_raw_n() { return std::is_same<MT, MetBf16Delta>::value ? 8 : 12; }
template <class MT>
__device__ __forceinline__ void met_raw_load(Rsrc r, uint32_t voff, uint32_t mpb, uint32_t (&w)[met_raw_n<MT>()],
                                             bool palette, unsigned skip) {
  if constexpr (std::is_same<MT, MetBf16Delta>::value) {
#pragma unroll
    for (int p = 0; p < 5; p++)  // a word that is +-0 on the whole grid (skip bit p) is not loaded
      w[p] = (skip >> p) & 1u ? 0u : __float_as_uint(bld<kStream>(r, 2 * voff, (uint32_t)(2 * p) * mpb));
    if (palette) {
#pragma unroll
      for (int m = 0; m < 3; m++) w[5 + m] = 0u;
    } else {
#pragma unroll
      for (int m = 0; m < 3; m++) w[5 + m] = __float_as_uint(bld<kStream>(r, 2 * voff, (uint32_t)(10 + 2 * m) * mpb));
    }
  } else if constexpr (sizeof(MT) == 2) {
#pragma unroll
    for (int q = 0; q < 12; q++)
      w[q] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(r, (int)voff, (int)((q < 9 ? q : q + 1) * mpb), kStream) << 16;
  } else {
#pragma unroll
    for (int q = 0; q < 12; q++) w[q] = __float_as_uint(bld<kStream>(r, voff, (uint32_t)(q < 9 ? q : q + 1) * mpb));
  }
}
// Field c (0..8 metric, 10..12 media) of raw metric words; pal is the
// palette in LDS, or null.
template <class MT>
__device__ __forceinline__ float met_raw_get(const uint32_t (&w)[met_raw_n<MT>()], int c, const float* ref,
                                             const float4* pal) {
  if constexpr (std::is_same<MT, MetBf16Delta>::value) {
    if (c >= 10) {
      if (pal) {
        const float4 e = pal[w[4] >> 16];
        return c == 10 ? e.x : c == 11 ? e.y : e.z;
      }
      return __uint_as_float(w[5 + c - 10]);
    }
    const uint32_t u = w[c >> 1];
    return __uint_as_float((c & 1) ? (u & 0xffff0000u) : (u << 16)) + ref[c];
  } else {
    return __uint_as_float(w[c < 9 ? c : c - 1]);
  }
}

// Reads v, so that a load of it is waited for here.
__device__ __forceinline__ void arrived(float v) { asm volatile("" ::"v"(v)); }
__device__ __forceinline__ void arrived(uint32_t v) { asm volatile("" ::"v"(v)); }

// Interior stage kernel with every load of plane i+1 issued before plane i
// is computed: the points of the interior box (no absorbing layer, no free
// surface), where the general kernel's per-plane metric and RK-register
// loads would each cost a memory round trip that the whole block waits for
// at its barrier.  Per plane the block issues, in this order, the halo and
// the new queue plane of plane i+1, the metric of plane i+1, and the S and T
// words of plane i; vector-memory loads return in issue order, so waiting
// for the S and T words at the RK combine leaves nothing outstanding of the
// earlier ones, and those were issued a whole compute phase earlier.  The
// arithmetic is the general kernel's (same operators, same order of the
// sums), so results are identical to it bit for bit.
//
// BAND: the same pipeline on the points of the absorbing layers (the general
// kernel's KIND 1 tiles; no free-surface rows): the RHS of a point inside the
// ADE-PML band of a face gets -aux/beta of that face, and the Cerjan sponge
// damps the new value.  The aux words of plane i are issued with its S and T
// words, one face per axis at most (the host uses this kernel only when the
// two bands of an axis do not overlap), and added after the three axis sums
// in the general kernel's order; 1/beta and the sponge factor of plane i+1
// are fetched during plane i.
//
// With aux_fused a BAND tile also advances the ADE-PML auxiliary fields of
// its points (what pml_aux_kernel does for them, with the same arithmetic),
// one face after another for a point on several.  A kernel of its own for the
// points on several faces read all their words again: 0.55 ms per step at
// 400 x 300 x 200, for 0.1 ms more in the tiles.
//
// TOP: the free-surface rows' terms as well, so that a tile may hold points
// of any kind.
template <int FX, int FY, int FZ, class MT, int TJ_, int NT_, int MINB, bool BAND = false, bool RING = true,
          bool TOP = false>
__global__ void __launch_bounds__(NT_, MINB) wave_interior_kernel(WaveArgs<MT> a) {
  static_assert(!TOP || (BAND && 64 % TJ_ == 0), "free-surface tiles: band terms, whole k rows per wavefront");
  constexpr int TJ = TJ_, TK = NT_ / TJ_;
  constexpr int WR = 64 % TJ_ == 0 ? 64 / TJ_ : TK;  // k rows of a wavefront (of the tile if they do not divide)
  constexpr int LJ = TJ + 4, LK = TK + 4;
  // halo cells of one plane: the 4 k-halo rows over the tile's own columns
  // and 4 j-halo cells per row; the corners of the LDS tile are neither
  // written nor read (the y and z operators reach along one axis only), so
  // each k-halo row costs the cache lines of the tile's own columns alone
  constexpr int NH = 4 * TJ + 4 * TK;
  // a thread has one halo cell; the few cells of a tile that has more of them
  // than threads (64 x 4: 16) are split into words, one per thread: as second
  // cells they took nine registers and nine loads for a sixteenth of the block
  constexpr int NHX = NH > NT_ ? 9 * (NH - NT_) : 0;
  static_assert(NHX <= NT_, "at most one word of the further halo cells per thread");
  constexpr int HJL = FY > 0 ? 1 : 3;
  constexpr int HKL = FZ > 0 ? 1 : 3;
  constexpr int QLO = FX > 0 ? -1 : -3;
  constexpr int CTR = -QLO;
  constexpr int NMW = met_raw_n<MT>();
  // RING: an LDS ring of the planes i .. i + LEAD: plane i + LEAD enters the
  // x-queue during step i, and its y/z halo is loaded in the same step, so
  // that a tile reads its neighbours' edge lines when they load those lines
  // as their own queue plane (still in L2), not LEAD planes later.
  // Otherwise a double buffer of planes i and i + 1 (LEAD 1), whose own
  // values come from the queue: a third of the LDS, for blocks that share a CU.
  constexpr int QLEAD = QLO + 5;  // the queue's newest plane is i + QLEAD
  constexpr int LEAD = RING ? QLEAD : 1;
  constexpr int NS = LEAD + 1;
  __shared__ float lds[NS][9][LK][LJ];
  // the media palette of the bfloat16-deviation form, staged once per block
  __shared__ float4 s_pal[std::is_same<MT, MetBf16Delta>::value ? kMaxMediaPalette : 1];

  const int item = xcd_remap((int)blockIdx.x, a.nwork);
  const int4 wk = a.work[2 * item], we = a.work[2 * item + 1];
  const int j0 = wk.x, k0 = wk.y, ibeg = wk.z, iend = wk.w;
  typedef const __attribute__((address_space(4))) WaveArgs<MT>* ArgPtr;
  const ArgPtr kargs = (ArgPtr)__builtin_amdgcn_kernarg_segment_ptr();  // the argument a
  const int tj = threadIdx.x, tk = threadIdx.y, tid = tj + tk * TJ;
  const int ni = a.ni, nj = a.nj, nk = a.nk;
  const int j = j0 + tj, k = k0 + tk;
  const int ku = k0 + (WR < TK ? __builtin_amdgcn_readfirstlane(tk) : 0);  // first of the wavefront's rows, uniform
  // A lane without a point of the tile computes what its cells give and stores
  // nothing (its stores' offsets are out of range), so that the plane loop
  // branches on uniform values alone; a wavefront without any has a loop of
  // its own.
  const bool act = tj >= we.z && tj < we.x && tk >= we.w && tk < we.y;
  const int nxp = ni + 6;
  const uint32_t nyz = a.nyz;
  const uint32_t py = a.py, jpad = a.jpad;
  const uint32_t col = jpad + (uint32_t)(min(max(j, -3), nj + 2) + 3) + (uint32_t)(min(max(k, -3), nk + 2) + 3) * py;
  const uint32_t col4 = col << 2;
  const uint32_t out4 = act ? col4 : kNoWord;
  // the metric of a point of the tile in every lane
  const uint32_t mcol = (jpad + (uint32_t)(j0 + min(max(tj, we.z), we.x - 1) + 3) +
                         (uint32_t)(k0 + min(max(tk, we.w), we.y - 1) + 3) * py) * (uint32_t)sizeof(MT);
  const uint32_t pb = nyz * 4, mpb = nyz * (uint32_t)sizeof(MT);
  const float* __restrict__ Win = a.Win;
  const int irk = a.irk;

  // LDS place and column of halo cell h: the 4 k-halo rows, then the 4 j-halo
  // cells of each row
  auto halo_cell = [&](int h, int& l, int& m) -> uint32_t {
    if (h < 4 * TJ) {
      const int r = h / TJ;
      l = r < HKL ? r : r + TK;
      m = HJL + h % TJ;
    } else {
      const int h2 = h - 4 * TJ;
      const int cc = h2 % 4;
      l = HKL + h2 / 4;
      m = cc < HJL ? cc : cc + TJ;
    }
    const int gj = min(max(j0 + m - HJL, -3), nj + 2), gk = min(max(k0 + l - HKL, -3), nk + 2);
    return (jpad + (uint32_t)(gj + 3) + (uint32_t)(gk + 3) * py) << 2;
  };
  // this thread's halo cell tid, and its word of the cells from NT_ on
  int hlk = 0, hlj = 0, xl = 0;
  const uint32_t hcol4 = tid < NH ? halo_cell(tid, hlk, hlj) : col4;
  uint32_t xw4 = kNoWord;
  if (NHX > 0 && tid < NHX) {
    int l, m;
    xw4 = halo_cell(NT_ + tid / 9, l, m) + (uint32_t)(tid % 9) * pb;
    xl = (tid % 9 * LK + l) * LJ + m;
  }
  struct Halo {
    float c[9], x;
  };
  auto load_halo = [&](Rsrc r, Halo& v) {
#pragma unroll
    for (int c = 0; c < 9; c++) v.c[c] = bld(r, hcol4, c * pb);
    if (NHX > 0) v.x = bld(r, xw4, 0);
  };
  auto store_halo = [&](float (*L)[LK][LJ], const Halo& v) {
    if (tid < NH) {
#pragma unroll
      for (int c = 0; c < 9; c++) L[c][hlk][hlj] = v.c[c];
    }
    if (NHX > 0 && tid < NHX) (&L[0][0][0])[xl] = v.x;
  };

  // BAND: per lane, the 1/beta of the point's column (j, k) along y and z, the
  // coefficients d/beta and -(alpha + d/beta) of its auxiliary ODEs there,
  // the sponge factor of the column, and its words' byte offsets in the first
  // field of its x, y and z face planes (the high y and z faces follow the
  // low ones within a plane), kNoWord outside the band.  Whether a wavefront
  // has a face along x (its plane), y (its columns) or z (its rows) is
  // uniform, and a face's words are loaded and stored for all of its lanes:
  // those without one read 0 and store nothing.  Under lane masks the loads
  // of the different faces met in the same registers, which cost copies
  // behind waits for the loads in flight.  The uniform descriptors are kernel
  // arguments and every access a buffer access from a uniform plane base:
  // through pointers staged in LDS they were flat accesses, which count as
  // LDS operations too, so that the first LDS read of the compute waited for
  // all loads in flight.
  const bool pml = BAND && a.pml, cerjan = BAND && a.cerjan;
  float rb2 = 1.0f, rb3 = 1.0f, cjk = 1.0f;
  float dy = 0.0f, ay = 0.0f, dz = 0.0f, az = 0.0f;
  const int N = BAND ? a.cold.N : 0;
  const uint32_t xpp = (uint32_t)nk * nj, ypp = (uint32_t)nk * N, zpp = (uint32_t)N * nj;  // words of a field of a face plane
  const uint32_t nyf = BAND ? a.cold.on[2] + a.cold.on[3] : 0, nzf = BAND ? a.cold.on[4] + a.cold.on[5] : 0;
  uint32_t xo4 = kNoWord, yo4 = kNoWord, zo4 = kNoWord;
  bool hasy = false, hasz = false;  // the wavefront has columns in a y band, rows in a z band
  if constexpr (BAND) {
    if (pml) {
      const int ja = j0 + we.z, jb = j0 + we.x;
      hasy = (a.cold.on[2] && ja < N) || (a.cold.on[3] && jb > nj - N);
      hasz = (a.cold.on[4] && ku < N) || (a.cold.on[5] && ku + WR > nk - N);
    }
    if (act && pml) {
      rb2 = 1.0f / a.cold.pB[1][j];
      rb3 = 1.0f / a.cold.pB[2][k];
      dy = a.cold.pD[1][j];
      ay = -(a.cold.pA[1][j] + dy);
      dz = a.cold.pD[2][k];
      az = -(a.cold.pA[2][k] + dz);
      xo4 = (uint32_t)(j + k * nj) << 2;
      if (a.cold.on[2] && j < N) yo4 = (uint32_t)(j + k * N) << 2;
      else if (a.cold.on[3] && j >= nj - N) yo4 = ((uint32_t)(j - (nj - N) + k * N) + (a.cold.on[2] ? 9 * ypp : 0u)) << 2;
      if (a.cold.on[4] && k < N) zo4 = (uint32_t)(j + k * nj) << 2;
      else if (a.cold.on[5] && k >= nk - N) zo4 = ((uint32_t)(j + (k - (nk - N)) * nj) + (a.cold.on[4] ? 9 * zpp : 0u)) << 2;
    }
    if (act && cerjan) cjk = fminf(a.cold.cj[1][j + 3], a.cold.cj[2][k + 3]);
  }
  const int xoff1 = BAND ? (a.cold.on[0] ? N : 0) : 0;  // first plane of the high x face
  // 1/beta of plane i along x and the sponge factor of plane i (uniform)
  auto rb_x = [&](int i) { return pml ? 1.0f / uni(a.cold.pB[0], i) : 1.0f; };
  auto cj_x = [&](int i) { return cerjan ? uni(a.cold.cj[0], i + 3) : 1.0f; };

  if (__builtin_amdgcn_ballot_w64(act) == 0) {  // the cells of the neighbours' stencils alone
    Halo v;
    float own[9];
    auto stage = [&](int plane, int slot) {
      const Rsrc r = plane_rsrc(Win, plane + 3, 9, nyz);
#pragma unroll
      for (int c = 0; c < 9; c++) own[c] = bld(r, col4, c * pb);
      load_halo(r, v);
#pragma unroll
      for (int c = 0; c < 9; c++) lds[slot][c][tk + HKL][tj + HJL] = own[c];
      store_halo(lds[slot], v);
    };
    for (int m = 0; m < LEAD; m++)
      if (ibeg + m < iend) stage(ibeg + m, m);
    if (std::is_same<MT, MetBf16Delta>::value && a.pal != nullptr)
      for (int e = tid; e < a.npal; e += NT_) s_pal[e] = a.pal[e];
    __syncthreads();
    int b = 0;
    for (int i = ibeg; i < iend; ++i) {
      if (i + LEAD < iend) stage(i + LEAD, b == 0 ? NS - 1 : b - 1);
      b = b == NS - 1 ? 0 : b + 1;
      __syncthreads();
    }
    return;
  }

  float q[5][9];
#pragma unroll
  for (int m = 0; m < 5; m++) {
    const Rsrc r = plane_rsrc(Win, ibeg + QLO + m + 3, 9, nyz);
#pragma unroll
    for (int c = 0; c < 9; c++) q[m][c] = bld(r, col4, c * pb);
  }
  // planes ibeg .. ibeg + LEAD - 1 of the ring: own values from the queue,
  // halos loaded here
  Halo hv;
#pragma unroll
  for (int m = 0; m < LEAD; m++) {
    if (ibeg + m < iend) {  // uniform per block
      load_halo(plane_rsrc(Win, ibeg + m + 3, 9, nyz), hv);
#pragma unroll
      for (int c = 0; c < 9; c++) lds[m][c][tk + HKL][tj + HJL] = q[CTR + m][c];
      store_halo(lds[m], hv);
    }
  }
  const bool palette = std::is_same<MT, MetBf16Delta>::value && a.pal != nullptr;  // uniform
  if (palette)
    for (int e = tid; e < a.npal; e += NT_) s_pal[e] = a.pal[e];
  uint32_t mw[NMW];
  const unsigned met_skip = a.met_skip;  // uniform
  met_raw_load<MT>(plane_rsrc(a.met, ibeg + 3, met_nf<MT>(), nyz), mcol, mpb, mw, palette, met_skip);
  float rb1 = 1.0f, cjx = 1.0f;
  if constexpr (BAND) { rb1 = rb_x(ibeg); cjx = cj_x(ibeg); }
  __syncthreads();

  int b = 0;  // ring slot of plane i; plane i + LEAD goes to the slot before it
  for (int i = ibeg; i < iend; ++i) {
    // band tiles read the arguments again in every plane: held in scalar
    // registers across the loop, with the field offsets and the masks of the
    // bands, they spill to vector lanes (444 v_readlane in the loop of the
    // tiles of any kind)
    const ArgPtr ap = BAND ? here(kargs) : kargs;
    const bool more = i + 1 < iend;       // uniform per block
    const bool ahead = i + LEAD < iend;   // uniform per block
    const int bw = b == 0 ? NS - 1 : b - 1;
    // plane i + QLEAD: queue plane, and with RING its halo (clamped
    // in-bounds past the chunk, where the queue plane goes unused); plane
    // i + 1: the halo without RING, and the metric
    float nq[9];
    {
      const Rsrc r = plane_rsrc(Win, min(i + QLEAD + 3, nxp - 1), 9, nyz);
#pragma unroll
      for (int c = 0; c < 9; c++) nq[c] = bld(r, col4, c * pb);
      if (RING && ahead) load_halo(r, hv);
    }
    if (!RING && ahead) load_halo(plane_rsrc(Win, i + 4, 9, nyz), hv);
    uint32_t mwn[NMW];
    met_raw_load<MT>(plane_rsrc(ap->met, min(i + 4, nxp - 1), met_nf<MT>(), nyz), mcol, mpb, mwn, palette, met_skip);
    float rb1n = 1.0f, cjxn = 1.0f;
    if constexpr (BAND) {
      if (more) { rb1n = rb_x(i + 1); cjxn = cj_x(i + 1); }
    }
    // plane i: the step-start (S) and accumulator (T) words of the RK
    // combine; stage 1 derives T from S and the point's stage-0 value
    // unless the point keeps it (rk_combine_b)
    const bool slab = ap->fault && i >= ap->ii0 - 3 && i <= ap->ii0 + 3 && i != ap->ii0;
    const float damp = cerjan ? fminf(cjx, cjk) : 1.0f;
    const bool keep_plane = ap->fault && i == ap->ii0;
    const bool keep_t = damp != 1.0f || keep_plane;
    const bool keep_any = keep_plane || (cerjan && __builtin_amdgcn_ballot_w64(damp != 1.0f) != 0);  // uniform
    const bool rk = !ap->rhs_only && !slab;
    const Rsrc rs = plane_rsrc(ap->S, i + 3, 9, nyz), rt = plane_rsrc(ap->T, i + 3, 9, nyz);
    // (zeros where the stage has no use for them: left unset, the registers
    // were carried from plane to plane, with copies behind a wait for the
    // stores)
    float sv[9], tv[9];
    if (rk && (irk >= 2 || (irk == 1 && keep_any))) {
#pragma unroll
      for (int c = 0; c < 9; c++) tv[c] = bld<kStream>(rt, col4, c * pb);
    } else {
#pragma unroll
      for (int c = 0; c < 9; c++) tv[c] = 0.0f;
    }
    if (rk && (irk == 1 || irk == 2)) {
#pragma unroll
      for (int c = 0; c < 9; c++) sv[c] = bld<kStream>(rs, col4, c * pb);
    } else {
#pragma unroll
      for (int c = 0; c < 9; c++) sv[c] = 0.0f;
    }
    // BAND: the auxiliary values of plane i on the wavefront's faces
    // (pmlx.cu:126-210 and the y/z variants), issued with S and T
    float vx[9], vy[9], vz[9];
    bool inx = false;  // a plane of an x band
    int pix = 0;
    const auto cold = &ap->cold;
    // applies f(resource, byte offset, bytes of a field) to the lane's word
    // of its x, y or z face in the axis's array
    auto on_x = [&](float* arr, auto f) { f(aux_rsrc(arr, pix, xpp, 1), xo4, here(4 * xpp)); };
    auto on_y = [&](float* arr, auto f) { f(aux_rsrc(arr, i, ypp, nyf), yo4, here(4 * ypp)); };
    auto on_z = [&](float* arr, auto f) { f(aux_rsrc(arr, i, zpp, nzf), zo4, here(4 * zpp)); };
    auto ld9 = [](float(&v)[9]) {
      return [&v](Rsrc r, uint32_t o, uint32_t fb) {
#pragma unroll
        for (int c = 0; c < 9; c++) v[c] = bld(r, o, c * fb);
      };
    };
    auto st9 = [](const float(&v)[9]) {
      return [&v](Rsrc r, uint32_t o, uint32_t fb) {
#pragma unroll
        for (int c = 0; c < 9; c++) bst<kReuse>(r, o, c * fb, v[c]);
      };
    };
    if constexpr (BAND) {
      if (pml) {
        if (cold->on[0] && i < N) { inx = true; pix = i; }
        else if (cold->on[1] && i >= ni - N) { inx = true; pix = i - (ni - N) + xoff1; }
        if (inx) on_x(cold->axY[0], ld9(vx));
        if (hasy) on_y(cold->axY[1], ld9(vy));
        if (hasz) on_z(cold->axY[2], ld9(vz));
      }
    }

    {
      auto MET = [&](int c) { return met_raw_get<MT>(mw, c, a.mref, palette ? s_pal : nullptr); };
      const float xix = MET(0), xiy = MET(1), xiz = MET(2);
      const float etx = MET(3), ety = MET(4), etz = MET(5);
      const float ztx = MET(6), zty = MET(7), ztz = MET(8);
      const float lam = MET(10), mu = MET(11);
      const float rrho = 1.0f / MET(12);
      const float l2m = lam + 2.0f * mu;
      const float rDH = ap->rDH;
      const float(*L)[LK][LJ] = lds[b];
      const int lj = tj + HJL, lk = tk + HKL;
      auto Dx = [&](int c) { return drp5<FX>(q[0][c], q[1][c], q[2][c], q[3][c], q[4][c]); };
      auto Dy = [&](int c) {
        return FY > 0 ? drp5<1>(L[c][lk][lj - 1], L[c][lk][lj], L[c][lk][lj + 1], L[c][lk][lj + 2], L[c][lk][lj + 3])
                      : drp5<-1>(L[c][lk][lj - 3], L[c][lk][lj - 2], L[c][lk][lj - 1], L[c][lk][lj], L[c][lk][lj + 1]);
      };
      auto Dz = [&](int c) {
        return FZ > 0 ? drp5<1>(L[c][lk - 1][lj], L[c][lk][lj], L[c][lk + 1][lj], L[c][lk + 2][lj], L[c][lk + 3][lj])
                      : drp5<-1>(L[c][lk - 3][lj], L[c][lk - 2][lj], L[c][lk - 1][lj], L[c][lk][lj], L[c][lk + 1][lj]);
      };
      // TOP: whether the wavefront has surface rows (uniform), the lane's
      // surface row, and word p of its surface words (image_top_kernel)
      const bool top = TOP && ap->freenode && ku + WR > nk - 3;
      const bool last = top && ku + WR > nk - 1;
      const int row = (WR == 1 ? ku : k) - (nk - 3);
      auto top_word = [&](int p, bool mine) {
        return bld(__builtin_amdgcn_make_buffer_rsrc(ap->itop + (size_t)i * 18 * nj, (short)0, 18 * nj * 4, kBufWord3),
                   mine ? (uint32_t)(p * nj + j) << 2 : kNoWord, 0);
      };
      // one step of the auxiliary ODE of the lane's point on its face along
      // axis AX: aux' = -(alpha + d) aux + d * RHS_axis, RHS_axis from the
      // plain derivative along the axis, with the RK4 stage combine; y the
      // values, s and t the step-start and accumulator words
      auto advance = [&](auto AX, auto D, const float(&y)[9], const float(&s)[9], const float(&t)[9], float d1, float ad1, auto on) {
        constexpr int ax = decltype(AX)::value;
        const float rka = ap->rka, rkb = ap->rkb;
        const float e0 = ax == 0 ? xix : ax == 1 ? etx : ztx;
        const float e1 = ax == 0 ? xiy : ax == 1 ? ety : zty;
        const float e2 = ax == 0 ? xiz : ax == 1 ? etz : ztz;
        float dd[9], ah[9], w[9];
#pragma unroll
        for (int c = 0; c < 9; c++) dd[c] = rDH * D(c);
#pragma unroll
        for (int c = 0; c < 9; c++) ah[c] = ad1 * y[c] + d1 * axis_rhs_c(c, dd, e0, e1, e2, rrho, lam, l2m, mu);
        if (TOP && ax < 2 && last) {  // the traction-free term (pmlx.cu:185-210)
          const float c0 = d1 * (ax == 0 ? uni(cold->pB[0], i) : cold->pB[1][nearest_point(j, nj)]);
          float z1[3];
#pragma unroll
          for (int r = 0; r < 3; r++) z1[r] = top_word(12 + 3 * ax + r, row == 2);
#pragma unroll
          for (int c = 3; c < 9; c++) {
            const float v = ah[c] + pml_fs_term(c, z1, ztx, zty, ztz, lam, l2m, mu, c0);
            ah[c] = row == 2 ? v : ah[c];
          }
        }
        if (irk == 0) {  // the accumulator is derived in stage 1 (rk_derived_t)
          on(cold->axS[ax], st9(y));
#pragma unroll
          for (int c = 0; c < 9; c++) w[c] = y[c] + rka * ah[c];
        } else if (irk == 3) {
#pragma unroll
          for (int c = 0; c < 9; c++) w[c] = t[c] + rkb * ah[c];
        } else {
          float tn[9];
          if (irk == 1) {
#pragma unroll
            for (int c = 0; c < 9; c++) tn[c] = rk_derived_t(s[c], y[c]) + rkb * ah[c];
          } else {
#pragma unroll
            for (int c = 0; c < 9; c++) tn[c] = t[c] + rkb * ah[c];
          }
          on(cold->axT[ax], st9(tn));
#pragma unroll
          for (int c = 0; c < 9; c++) w[c] = s[c] + rka * ah[c];
        }
        on(cold->axY[ax], st9(w));
      };
      float h[9];
#pragma unroll
      for (int c = 0; c < 9; c++) h[c] = 0.0f;
      {
        // the general kernel's arithmetic (in the interior beta = 1: rb * rDH = rDH)
        const float s1 = rb1 * rDH, s2 = rb2 * rDH, s3 = rb3 * rDH;
        accum_axis(h, Dx, xix * s1, xiy * s1, xiz * s1, rrho, lam, l2m, mu, true);
        accum_axis(h, Dy, etx * s2, ety * s2, etz * s2, rrho, lam, l2m, mu, true);
        if (!top) {
          accum_axis(h, Dz, ztx * s3, zty * s3, ztz * s3, rrho, lam, l2m, mu, true);
        } else {
          // the top three rows under the free surface (wave.cu:207-245), as
          // the general kernel computes them: DzV of the stress rates from the
          // traction-free condition, L22 or L24, and the velocity RHS of the
          // image.  A wavefront's rows that are no surface rows keep the
          // general sums; by selects, since its rows may be of any of the four
          // kinds.
          float hs[6], tz[3], hv3[3];
          const bool mine = row >= 0 && row < 3;
#pragma unroll
          for (int c = 0; c < 6; c++) hs[c] = h[3 + c];
          accum_axis(h, Dz, ztx * s3, zty * s3, ztz * s3, rrho, lam, l2m, mu, WR > 1);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int c = 0; c < 3; c++) tz[c] = top_word(9 + c, row == 2);
          float dzv[3];
#pragma unroll
          for (int c = 0; c < 3; c++) {
            const float l22 = rDH * (FZ > 0 ? L[c][lk + 1][lj] - L[c][lk][lj] : L[c][lk][lj] - L[c][lk - 1][lj]);
            const float l24 = rDH * (FZ > 0 ? -C24_1 * L[c][lk][lj] + C24_2 * L[c][lk + 1][lj] - C24_3 * L[c][lk + 2][lj]
                                            : C24_3 * L[c][lk - 2][lj] - C24_2 * L[c][lk - 1][lj] + C24_1 * L[c][lk][lj]);
            dzv[c] = row == 2 ? tz[c] : row == 1 ? l22 : l24;
          }
          const float e0 = ztx * rb3, e1 = zty * rb3, e2 = ztz * rb3;
          hs[0] += (l2m * e0 * dzv[0] + lam * e1 * dzv[1] + lam * e2 * dzv[2]);
          hs[1] += (lam * e0 * dzv[0] + l2m * e1 * dzv[1] + lam * e2 * dzv[2]);
          hs[2] += (lam * e0 * dzv[0] + lam * e1 * dzv[1] + l2m * e2 * dzv[2]);
          hs[3] += (e1 * dzv[0] + e0 * dzv[1]) * mu;
          hs[4] += (e2 * dzv[0] + e0 * dzv[2]) * mu;
          hs[5] += (e2 * dzv[1] + e1 * dzv[2]) * mu;
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int c = 0; c < 3; c++) hv3[c] = top_word(3 * c + row, mine);
#pragma unroll
          for (int c = 0; c < 9; c++) {
            const float v = c < 3 ? hv3[c % 3] : hs[(c + 3) % 6];
            h[c] = mine || WR == 1 ? v : h[c];
          }
        }
      }
      if constexpr (BAND) {
        if (pml) {
          // -aux/beta of each face, x then y then z (0 for a lane without it)
          if (inx) {
#pragma unroll
            for (int c = 0; c < 9; c++) h[c] += -vx[c] * rb1;
          }
          if (hasy) {
#pragma unroll
            for (int c = 0; c < 9; c++) h[c] += -vy[c] * rb2;
          }
          if (hasz) {
#pragma unroll
            for (int c = 0; c < 9; c++) h[c] += -vz[c] * rb3;
          }
        }
      }
      // Every load of the plane is waited for here: the youngest are needed
      // now, the others at the plane's end, where a wait for them would be a
      // wait for the stores below as well (they count together, in order).
      // The stores drain during the next plane: 41.7 -> 37.5 ms of interior
      // tiles per step at 800 x 1000 x 500, 2.18 -> 1.76 ms of tiles at
      // 251 x 187 x 143.
#pragma unroll
      for (int c = 0; c < 9; c++) arrived(nq[c]), arrived(hv.c[c]), arrived(sv[c]), arrived(tv[c]);
      if (NHX > 0) arrived(hv.x);
#pragma unroll
      for (int m = 0; m < NMW; m++) arrived(mwn[m]);
      // the first face's step-start and accumulator words, in flight during
      // the RK combine (they take the registers of the stencil's operands)
      const bool fuse = BAND && pml && ap->aux_fused && !ap->rhs_only;
      float as[9], at[9];
      auto ld_st = [&](auto AX, auto on) {
        constexpr int ax = decltype(AX)::value;
        if (irk >= 2) on(cold->axT[ax], ld9(at));
        if (irk == 1 || irk == 2) on(cold->axS[ax], ld9(as));
      };
      constexpr std::integral_constant<int, 0> X{};
      constexpr std::integral_constant<int, 1> Y{};
      constexpr std::integral_constant<int, 2> Z{};
      if (!TOP && fuse) {
        if (inx) ld_st(X, on_x);
        else if (hasy) ld_st(Y, on_y);
        else if (hasz) ld_st(Z, on_z);
      }
      if (ap->rhs_only) {
#pragma unroll
        for (int c = 0; c < 9; c++) bst(plane_rsrc(ap->rhs, i + 3, 9, nyz), out4, c * pb, h[c]);
      } else if (slab) {
        const Rsrc r = plane_rsrc(ap->slabH, i - (ap->ii0 - 3), 9, nyz);
#pragma unroll
        for (int c = 0; c < 9; c++) bst(r, out4, c * pb, h[c]);
      } else {
        // RK_Syn (rk4.cu:20-33); the damping factor is 1 in the interior
        const Rsrc ro = plane_rsrc(ap->Wout, i + 3, 9, nyz);
        const float rka = ap->rka, rkb = ap->rkb;
        // one branch per stage around its nine fields, not one per field
        if (irk == 0) {
          if (keep_any) {
            const uint32_t t4 = keep_t ? out4 : kNoWord;
#pragma unroll
            for (int c = 0; c < 9; c++) bst(rt, t4, c * pb, q[CTR][c] + rkb * h[c]);
          }
#pragma unroll
          for (int c = 0; c < 9; c++) bst(ro, out4, c * pb, (q[CTR][c] + rka * h[c]) * damp);
        } else if (irk == 3) {
#pragma unroll
          for (int c = 0; c < 9; c++) bst(ro, out4, c * pb, (tv[c] + rkb * h[c]) * damp);
        } else {
          float tb[9];
#pragma unroll
          for (int c = 0; c < 9; c++) tb[c] = irk == 2 || keep_t ? tv[c] : rk_derived_t(sv[c], q[CTR][c]);
#pragma unroll
          for (int c = 0; c < 9; c++) {
            bst(rt, out4, c * pb, tb[c] + rkb * h[c]);
            bst(ro, out4, c * pb, (sv[c] + rka * h[c]) * damp);
          }
        }
      }
      if (fuse) {
        if (inx) {
          if (TOP) ld_st(X, on_x);
          const float d1 = uni(cold->pD[0], i);
          advance(X, Dx, vx, as, at, d1, -(uni(cold->pA[0], i) + d1), on_x);
        }
        if (hasy) {
          if (TOP || inx) ld_st(Y, on_y);
          advance(Y, Dy, vy, as, at, dy, ay, on_y);
        }
        if (hasz) {
          if (TOP || inx || hasy) ld_st(Z, on_z);
          advance(Z, Dz, vz, as, at, dz, az, on_z);
        }
      }
    }

    if (ahead) {
#pragma unroll
      for (int c = 0; c < 9; c++) lds[bw][c][tk + HKL][tj + HJL] = RING ? nq[c] : q[CTR + 1][c];
      store_halo(lds[bw], hv);
    }
    b = b == NS - 1 ? 0 : b + 1;
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
      for (int c = 0; c < 9; c++) q[m][c] = q[m + 1][c];
#pragma unroll
    for (int c = 0; c < 9; c++) q[4][c] = nq[c];
#pragma unroll
    for (int m = 0; m < NMW; m++) mw[m] = mwn[m];
    if constexpr (BAND) { rb1 = rb1n; cjx = cjxn; }
    __syncthreads();
  }
}

// ADE-PML auxiliary fields (pmlx.cu:126-210, pmly.cu, pmlz.cu): for every
// point of the band of face f, the plain one-sided derivative along the
// face's axis drives aux' = -(alpha + d/beta) aux + (d/beta) * RHS_axis, plus
// the traction-free term on the free surface for the x/y faces, advanced
// with the same RK4 stage combine as the wavefield.  Runs after the stage
// kernel (which read the old aux values) on the unchanged stage input.  One
// thread per band point, j fastest so aux accesses are contiguous; on x
// faces the band plane index comes next, so the five planes of an
// x-derivative are read by neighbouring blocks and stay in L2.
template <class MT>
struct PmlAuxArgs {
  const float* __restrict__ Win;
  const MT* __restrict__ met;
  // every face's arrays, passed directly (kernel arguments are preloaded):
  // auxiliary value, step start and RK accumulator; per axis the PML
  // profiles; the free-surface velocity maps of the x and y faces.  Picked
  // with constant indices (a runtime index into the argument block would
  // copy it to scratch memory).
  float* Y[6];
  float* S[6];
  float* T[6];
  const float* pA[3];
  const float* pB[3];
  const float* pD[3];
  const float* mat[2];
  // boxes of points to update, kPmlBoxInts ints each: face, then the
  // face-local (start, count) of j, k and i, then the box's first block
  const int* __restrict__ boxes;
  int nbox;
  int flag[3];  // one-sided operator sign along each axis
  int np[3];    // nine-field parts of a plane of each axis's auxiliary arrays
  int N;
  int ni, nj, nk, ny, py, jpad;
  unsigned pyz;
  float rDH, rka, rkb;
  float mref[10];   // metric reference values (bfloat16-deviation form)
  int irk, freenode;
};

template <class T>
__device__ __forceinline__ T pick6(int f, const T (&v)[6]) {
  return f == 0 ? v[0] : f == 1 ? v[1] : f == 2 ? v[2] : f == 3 ? v[3] : f == 4 ? v[4] : v[5];
}
template <class T>
__device__ __forceinline__ T pick3(int x, const T (&v)[3]) { return x == 0 ? v[0] : x == 1 ? v[1] : v[2]; }

// One launch for all absorbing faces: each box of points (a face, or a part
// of one) is served by a contiguous run of blocks, numbered
// XCD-contiguously so that the blocks sharing stencil planes (neighbouring
// band planes on x faces, rows on z faces) share one L2.
template <class MT>
__global__ void __launch_bounds__(256) pml_aux_kernel(PmlAuxArgs<MT> a) {
  const int b = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  // the box of this block (block-uniform loads; a handful of boxes)
  const int* B = a.boxes;
  int q = 0;
  for (int r = 1; r < a.nbox; r++)
    if (b >= B[r * kPmlBoxInts + 7]) q = r;
  const int* bx = B + q * kPmlBoxInts;
  const int f = bx[0], bj0 = bx[1], bnj = bx[2], bk0 = bx[3], bnk = bx[4], bi0 = bx[5], bni = bx[6];
  const int ax = f >> 1, N = a.N, flag = pick3(ax, a.flag);
  const int nn = ax == 0 ? a.ni : ax == 1 ? a.nj : a.nk;
  const int off = (f & 1) ? nn - N : 0;
  const int pnj = ax == 1 ? N : a.nj, pnk = ax == 2 ? N : a.nk;
  const long pp = (long)pnj * pnk;
  const long idx = (long)(b - bx[7]) * 256L + threadIdx.x;
  if (idx >= (long)bnj * bnk * bni) return;
  const int pj = bj0 + (int)(idx % bnj);
  const long t = idx / bnj;
  // j fastest, then the band plane index on x faces (its five x-derivative
  // planes are read by neighbouring blocks), k on the others
  const int pk = bk0 + (ax == 0 ? (int)(t / bni) : (int)(t % bnk));
  const int pi = bi0 + (ax == 0 ? (int)(t % bni) : (int)(t / bnk));
  const long pa = pj + (long)pk * pnj + (long)pi * pick3(ax, a.np) * 9 * pp;  // aux layout (aux_rsrc)
  const int i = pi + (ax == 0 ? off : 0), j = pj + (ax == 1 ? off : 0), k = pk + (ax == 2 ? off : 0);
  const int li = ax == 0 ? i : ax == 1 ? j : k;
  const unsigned pyz = a.pyz;
  const long col = a.jpad + (j + 3) + (long)(k + 3) * a.py;
  const int x = i + 3;
  const float* W = a.Win;
  // neighbour offset (words) along the axis, within one field's plane or across planes
  const long st = ax == 0 ? 9L * pyz : ax == 1 ? 1L : (long)a.py;
  const long base = (long)x * 9 * pyz + col;
  float dd[9];
#pragma unroll
  for (int c = 0; c < 9; c++) {
    const float* w = W + base + (long)c * pyz;
    dd[c] = a.rDH * (flag > 0 ? drp5<1>(w[-st], w[0], w[st], w[2 * st], w[3 * st])
                                : drp5<-1>(w[-3 * st], w[-2 * st], w[-st], w[0], w[st]));
  }
  const MT* M = a.met;
  auto MET = [&](int m) { return mat_(M, m, x, (uint32_t)col, pyz, a.mref); };
  const float e0 = MET(3 * ax), e1 = MET(3 * ax + 1), e2 = MET(3 * ax + 2);
  const float lam = MET(10), mu = MET(11), rrho = 1.0f / MET(12), l2m = lam + 2.0f * mu;
  const float* pAx = pick3(ax, a.pA);
  const float* pBx = pick3(ax, a.pB);
  const float* pDx = pick3(ax, a.pD);
  const float b1 = pBx[li], d1 = pDx[li], ad1 = -(pAx[li] + d1);
  const float c0 = d1 * b1;
  const bool fsx = ax < 2 && a.freenode && k == a.nk - 1;
  float z1[3] = {0.0f, 0.0f, 0.0f}, ztx = 0.0f, zty = 0.0f, ztz = 0.0f;
  if (fsx) {
    const float* mat = ax == 0 ? a.mat[0] : a.mat[1];
    const long ij = ((long)(j + 3) + (long)(i + 3) * a.ny) * 9;
#pragma unroll
    for (int r = 0; r < 3; r++) z1[r] = mat[ij + 3 * r] * dd[0] + mat[ij + 3 * r + 1] * dd[1] + mat[ij + 3 * r + 2] * dd[2];
    ztx = MET(6); zty = MET(7); ztz = MET(8);
  }
  float* Y = pick6(f, a.Y);
  float* S = pick6(f, a.S);
  float* T = pick6(f, a.T);
#pragma unroll
  for (int c = 0; c < 9; c++) {
    const long q = c * pp + pa;
    const float y = Y[q];
    float ah = ad1 * y + d1 * axis_rhs_c(c, dd, e0, e1, e2, rrho, lam, l2m, mu);
    if (fsx && c >= 3) ah += pml_fs_term(c, z1, ztx, zty, ztz, lam, l2m, mu, c0);
    // RK_Syn (rk4.cu:20-33) on the step start S and accumulator T of the
    // auxiliary field, the accumulator of stage 0 derived in stage 1 from S
    // and the stage-0 value (rk_derived_t), as in the band tiles
    float w;
    if (a.irk == 0) {
      S[q] = y;
      w = y + a.rka * ah;
    } else if (a.irk == 3) {
      w = T[q] + a.rkb * ah;
    } else {
      const float s = S[q];
      const float t = a.irk == 1 ? rk_derived_t(s, y) : T[q];
      T[q] = t + a.rkb * ah;
      w = s + a.rka * ah;
    }
    Y[q] = w;
  }
}

// The free-surface image.
template <int FX, int FY, int FZ, class MT>
void launch_image(const WaveArgs<MT>& a, const Ctx& c, hipStream_t s) {
  const long n = (long)c.d.ni * 3 * c.d.nj;
  hipLaunchKernelGGL((image_top_kernel<FX, FY, FZ, MT>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a);
}

template <int FX, int FY, int FZ, class MT>
void launch_wave_t(WaveArgs<MT> a, const Ctx& c, hipStream_t s) {
  // work list order: interior, bands (64-wide tiles), bands (32-wide tiles), free-surface tiles
  const int* n = c.wave_nkind;
  const int o1 = n[0], o2 = o1 + n[1], o3 = o2 + n[2];
  const int4* w = (const int4*)c.wave_work;
  Profiler& pr = const_cast<Ctx&>(c).prof;
  // StageStreams: the interior tiles and the free-surface passes share no
  // words with the bands or with each other (disjoint points, read-only stage
  // input), so they run on side streams, fenced after the work already queued
  // on the solver's stream; the auxiliary update waits for the surface tiles
  // (which read the aux fields) and the caller's next launch for the interior.
  // While kernel classes are timed the launches stay serial, so that each
  // class's events bracket its own kernels only.  A failing event call sets
  // HIP's last error, which the caller's launch check reports.
  const bool par = c.side[0] != nullptr && !c.prof.on;
  hipStream_t si = s, ss = s;
  if (par) {
    (void)hipEventRecord(c.fence[0], s);
    si = c.side[0];
    ss = c.side[1];
    (void)hipStreamWaitEvent(si, c.fence[0], 0);
    (void)hipStreamWaitEvent(ss, c.fence[0], 0);
  }
  if (n[0] > 0) {
    a.work = w; a.nwork = n[0];
    pr.begin(si, PK_STAGE_INTERIOR);
    if (c.wave_tki == TK6)
      hipLaunchKernelGGL((wave_interior_kernel<FX, FY, FZ, MT, TJ, TJ * TK6, 2, false, false>), dim3(a.nwork), dim3(TJ, TK6, 1),
                         0, si, a);
    else if (c.wave_tki == TK4)  // at least 3 waves per SIMD: three blocks per CU (152-161 VGPRs with FP32 metric
      // words, no spills)
      hipLaunchKernelGGL((wave_interior_kernel<FX, FY, FZ, MT, TJ, TJ * TK4, 3, false, false>), dim3(a.nwork),
                         dim3(TJ, TK4, 1), 0, si, a);
    else if (c.wave_pipe && c.wave_ring)
      hipLaunchKernelGGL((wave_interior_kernel<FX, FY, FZ, MT, TJ, NTHR, 2>), dim3(a.nwork), dim3(TJ, TK, 1), 0, si, a);
    else if (c.wave_pipe)
      hipLaunchKernelGGL((wave_interior_kernel<FX, FY, FZ, MT, TJ, NTHR, 2, false, false>), dim3(a.nwork), dim3(TJ, TK, 1), 0,
                         si, a);
    else if (c.wave_tall)
      hipLaunchKernelGGL((wave_stage_kernel<FX, FY, FZ, MT, 0, TJ, 2 * NTHR>), dim3(a.nwork), dim3(TJ, 2 * TK, 1), 0, si, a);
    else
      hipLaunchKernelGGL((wave_stage_kernel<FX, FY, FZ, MT, 0>), dim3(a.nwork), dim3(TJ, TK, 1), 0, si, a);
    pr.end(si);
  }
  if (c.wave_unified) {
    pr.begin(s, PK_STAGE_BAND);
    if (a.freenode) launch_image<FX, FY, FZ, MT>(a, c, s);
    a.work = w + 2 * o1; a.nwork = n[1];
    hipLaunchKernelGGL((wave_interior_kernel<FX, FY, FZ, MT, TJN, NTHRN, 2, true, false, true>), dim3(a.nwork),
                       dim3(TJN, TKN, 1), 0, s, a);
    pr.end(s);
    return;
  }
  if (n[3] > 0) {
    a.work = w + 2 * o3; a.nwork = n[3];
    pr.begin(ss, PK_STAGE_SURFACE);
    if (a.freenode) launch_image<FX, FY, FZ, MT>(a, c, ss);
    if (c.wave_surf_pipe)
      hipLaunchKernelGGL((wave_interior_kernel<FX, FY, FZ, MT, TJ, NTHR, 2, true, true, true>), dim3(a.nwork), dim3(TJ, TK, 1),
                         0, ss, a);
    else
      hipLaunchKernelGGL((wave_stage_kernel<FX, FY, FZ, MT, 2>), dim3(a.nwork), dim3(TJ, TK, 1), 0, ss, a);
    pr.end(ss);
  }
  if (n[1] + n[2] > 0) {
    pr.begin(s, PK_STAGE_BAND);
    if (n[1] > 0) {
      a.work = w + 2 * o1; a.nwork = n[1];
      if (c.wave_band_pipe && c.wave_band_tk == TK4)
        hipLaunchKernelGGL((wave_interior_kernel<FX, FY, FZ, MT, TJ, TJ * TK4, 2, true, false>), dim3(a.nwork), dim3(TJ, TK4, 1),
                           0, s, a);
      else if (c.wave_band_pipe)
        hipLaunchKernelGGL((wave_interior_kernel<FX, FY, FZ, MT, TJ, NTHR, 2, true>), dim3(a.nwork), dim3(TJ, TK, 1), 0, s, a);
      else
        hipLaunchKernelGGL((wave_stage_kernel<FX, FY, FZ, MT, 1>), dim3(a.nwork), dim3(TJ, TK, 1), 0, s, a);
    }
    if (n[2] > 0) {
      a.work = w + 2 * o2; a.nwork = n[2];
      if (c.wave_band_pipe && c.wave_tjn == TJB)
        hipLaunchKernelGGL((wave_interior_kernel<FX, FY, FZ, MT, TJB, TJB * TKB, 2, true>), dim3(a.nwork), dim3(TJB, TKB, 1), 0,
                           s, a);
      else if (c.wave_band_pipe)
        hipLaunchKernelGGL((wave_interior_kernel<FX, FY, FZ, MT, TJN, NTHRN, 2, true>), dim3(a.nwork), dim3(TJN, TKN, 1), 0,
                           s, a);
      else
        hipLaunchKernelGGL((wave_stage_kernel<FX, FY, FZ, MT, 1, TJN, NTHRN>), dim3(a.nwork), dim3(TJN, TKN, 1), 0, s, a);
    }
    pr.end(s);
  }
  if (par) {
    (void)hipEventRecord(c.fence[2], ss);
    (void)hipStreamWaitEvent(s, c.fence[2], 0);
  }
  // the auxiliary fields of the points whose tiles do not advance them: all
  // of them without the fused update, with it those of the free-surface rows
  // k >= ktop when their tiles run the general kernel
  if (a.pml && !a.rhs_only) {
    PmlAuxArgs<MT> p{};
    p.Win = a.Win; p.met = a.met; p.N = c.pml.N;
    p.ni = a.ni; p.nj = a.nj; p.nk = a.nk; p.ny = a.ny; p.py = a.py; p.jpad = a.jpad; p.pyz = a.nyz;
    for (int m = 0; m < 10; m++) p.mref[m] = a.mref[m];
    p.rDH = a.rDH; p.rka = a.rka; p.rkb = a.rkb; p.irk = a.irk; p.freenode = a.freenode;
    p.flag[0] = FX; p.flag[1] = FY; p.flag[2] = FZ;
    for (int ax = 0; ax < 3; ax++) { p.pA[ax] = c.pml.A[ax]; p.pB[ax] = c.pml.B[ax]; p.pD[ax] = c.pml.D[ax]; }
    for (int ax = 0; ax < 3; ax++) p.np[ax] = c.pml.parts(ax);
    p.mat[0] = c.matVx2Vz; p.mat[1] = c.matVy2Vz;
    for (int f = 0; f < 6; f++) { p.Y[f] = c.pml.Y[f]; p.S[f] = c.pml.S[f]; p.T[f] = c.pml.T[f]; }
    // the boxes (wave_work_list): every face whole, or with the fused
    // update the free-surface rows when their tiles run the general kernel
    p.boxes = c.pml_boxes;
    p.nbox = c.pml_nbox;
    const int blocks = c.pml_blocks;
    if (blocks > 0) {
      pr.begin(s, PK_PML_AUX);
      hipLaunchKernelGGL(pml_aux_kernel<MT>, dim3((unsigned)blocks), dim3(256), 0, s, p);
      pr.end(s);
    }
  }
  if (par) {
    (void)hipEventRecord(c.fence[1], si);
    (void)hipStreamWaitEvent(s, c.fence[1], 0);
  }
}

template <class MT>
void launch_wave_dispatch(const WaveArgs<MT>& a, const Ctx& c, int fx, int fy, int fz, hipStream_t s) {
  int key = (fx > 0) * 4 + (fy > 0) * 2 + (fz > 0);
  switch (key) {
    case 0: launch_wave_t<-1, -1, -1, MT>(a, c, s); break;
    case 1: launch_wave_t<-1, -1, 1, MT>(a, c, s); break;
    case 2: launch_wave_t<-1, 1, -1, MT>(a, c, s); break;
    case 3: launch_wave_t<-1, 1, 1, MT>(a, c, s); break;
    case 4: launch_wave_t<1, -1, -1, MT>(a, c, s); break;
    case 5: launch_wave_t<1, -1, 1, MT>(a, c, s); break;
    case 6: launch_wave_t<1, 1, -1, MT>(a, c, s); break;
    default: launch_wave_t<1, 1, 1, MT>(a, c, s); break;
  }
}

// one instantiation per metric storage type, each in its own source file
extern template void launch_wave_dispatch<float>(const WaveArgs<float>&, const Ctx&, int, int, int, hipStream_t);
extern template void launch_wave_dispatch<uint16_t>(const WaveArgs<uint16_t>&, const Ctx&, int, int, int, hipStream_t);
extern template void launch_wave_dispatch<MetBf16Delta>(const WaveArgs<MetBf16Delta>&, const Ctx&, int, int, int,
                                                        hipStream_t);

}  // namespace wave
}  // namespace cgfdm
