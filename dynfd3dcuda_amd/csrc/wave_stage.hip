// Work lists and launches of the wave stage kernels (wave_stage_kernels.h):
// the interior box, absorbing-band and free-surface tiles of one RK stage,
// the XCD-contiguous block numbering, and the per-stage launch.
#include "wave_stage_kernels.h"
#include <cmath>

namespace cgfdm {
using namespace wave;

namespace {

template <class MT>
WaveArgs<MT> make_args(Ctx& c, const StageBufs& b, int irk, bool rhs_only, float* rhs_out) {
  WaveArgs<MT> a{};
  a.Win = b.Win; a.Wout = b.Wout; a.S = b.S; a.T = b.T;
  a.met = (const MT*)c.met;
  a.slabH = c.slabH;
  a.rhs = rhs_out;
  a.itop = c.img_top;
  WaveCold& w = a.cold;
  for (int x = 0; x < 3; x++) { w.pA[x] = c.pml.A[x]; w.pB[x] = c.pml.B[x]; w.pD[x] = c.pml.D[x]; w.cj[x] = c.cj[x]; }
  for (int f = 0; f < 6; f++) { w.auxY[f] = c.pml.Y[f]; w.on[f] = c.pml.on[f]; }
  for (int x = 0; x < 3; x++) {
    const int f = c.pml.on[2 * x] ? 2 * x : 2 * x + 1;  // the axis's first absorbing face
    w.axY[x] = c.pml.Y[f]; w.axS[x] = c.pml.S[f]; w.axT[x] = c.pml.T[f];
  }
  w.mVx = c.matVx2Vz; w.mVy = c.matVy2Vz;
  w.N = c.pml.N;
  bool any = false;
  for (int f = 0; f < 6; f++) any |= c.pml.on[f] != 0;
  a.pml = any ? 1 : 0;
  a.ni = c.d.ni; a.nj = c.d.nj; a.nk = c.d.nk; a.ny = c.d.ny; a.ii0 = c.d.i0 - 3;
  a.nyz = (unsigned)c.d.pyz;
  a.py = c.d.py; a.jpad = c.d.jpad;
  a.rDH = (float)(1.0 / c.p.DH);
  for (int m = 0; m < 10; m++) a.mref[m] = c.met_ref[m];
  a.pal = std::is_same<MT, MetBf16Delta>::value ? (const float4*)c.met_pal : nullptr;
  a.npal = c.met_npal;
  a.met_skip = std::is_same<MT, MetBf16Delta>::value ? c.met_skip : 0u;
  const double RA[4] = {0.5, 0.5, 1.0, 1e10}, RB[4] = {1.0 / 6.0, 1.0 / 3.0, 1.0 / 3.0, 1.0 / 6.0};
  a.rka = (float)(RA[irk] * c.p.DT);
  a.rkb = (float)(RB[irk] * c.p.DT);
  a.irk = irk;
  a.freenode = c.p.FreeSurface ? 1 : 0;
  a.cerjan = c.p.useCerjan ? 1 : 0;
  a.fault = c.p.Rupture ? 1 : 0;
  a.rhs_only = rhs_only ? 1 : 0;
  a.aux_fused = c.pml_fused ? 1 : 0;
  return a;
}

// Tiles [lo, hi) of one axis: the edge band below, tiles of length t
// starting at the interior's first index, the edge band above.  Each
// segment is (start, length, interior?).
// A tile range along one axis: lanes [0, n) of a tile starting at index s,
// of which [o, n) are active.  Low-side band segments end at the interior
// edge, so a partial tile's idle lanes fall on the ghost side (their clamped
// loads all hit the ghost column) rather than on interior points.
struct Seg { int s, n; bool in; int o; };
std::vector<Seg> axis_segments(int n, int lo, int hi, int t) {
  std::vector<Seg> v;
  const int a = std::min(lo, n), b = std::max(a, n - hi);
  const int m = (a + t - 1) / t;
  for (int q = 0; q < m; q++) {
    const int x = a - (m - q) * t;
    v.push_back({x, t, false, std::max(0, -x)});
  }
  for (int x = a; x < b; x += t) v.push_back({x, std::min(t, b - x), true, 0});
  for (int x = b; x < n; x += t) v.push_back({x, std::min(t, n - x), false, 0});
  return v;
}

}  // namespace

const char* const kProfNames[PK_COUNT] = {"stage_interior", "stage_band", "stage_surface", "pml_aux",
                                          "fault_pre", "fault_deriv", "fault_post", "rup_sensor", "fault_rs"};

// First interior column along j: the width of the low absorbing band, or
// with WaveBandRound that width rounded up to whole TJ-wide tiles, so that
// the band's tiles are full width (a 32-wide tile holding 20 band columns
// pays the j halo in whole cache lines for few points, in a launch of its
// own that cannot share those lines with the interior tile beside it).  The
// columns between the band and this edge are then plain points, which the
// band kernel treats like the interior one.
int interior_lo_j(const Params& p) {
  if (wave_unified(p)) return 0;  // tiles from the first column on
  const int band = std::max(p.usePML ? p.PML_N : 0, p.useCerjan ? p.DAMP_N : 0);
  if (p.WaveBandRound == 0) return band;
  return (band + TJ - 1) / TJ * TJ;
}

// Clears the counts of points and (point, face) pairs of the work lists.
static void clear_counts(Ctx& c) {
  for (int kd = 0; kd < 3; kd++) c.wave_points[kd] = 0;
  for (int kd = 0; kd < 4; kd++) c.aux_read_pairs[kd] = c.aux_update_pairs[kd] = 0;
}

// Adds the points of a block, planes [i0, i1) of columns [j0, j1) and rows
// [k0, k1), to the counts of kind kd; update: it advances their auxiliary
// fields.  Every list counts what it pushes, so that a tile missed or listed
// twice shows in the sums.
static void count_block(Ctx& c, int kd, int i0, int i1, int j0, int j1, int k0, int k1, bool update) {
  // points of [lo, hi) along axis ax inside that axis's absorbing bands, once
  // for each of the two where they overlap
  auto in_bands = [&](int ax, int lo, int hi) {
    const int N = c.pml.N, nn = ax == 0 ? c.d.ni : ax == 1 ? c.d.nj : c.d.nk;
    const int a0 = 0, a1 = c.pml.on[2 * ax] ? std::min(N, nn) : 0;
    const int b0 = c.pml.on[2 * ax + 1] ? std::max(nn - N, 0) : nn, b1 = nn;
    auto len = [&](int x0, int x1) { return std::max(0, std::min(x1, hi) - std::max(x0, lo)); };
    return len(a0, a1) + len(b0, b1);
  };
  const long Li = i1 - i0, Lj = j1 - j0, Lk = k1 - k0;
  const long bi = in_bands(0, i0, i1), bj = in_bands(1, j0, j1), bk = in_bands(2, k0, k1);
  const long pairs = bi * Lj * Lk + Li * bj * Lk + Li * Lj * bk;
  c.wave_points[kd] += Li * Lj * Lk;
  c.aux_read_pairs[kd] += pairs;
  if (update) c.aux_update_pairs[kd] += pairs;
}

// Uploads a work list (two int4 per block).
static int put_work(Ctx& c, const std::vector<int4>& all) {
  if (c.wave_work) { (void)hipFree(c.wave_work); c.wave_work = nullptr; }
  if (hipMalloc(&c.wave_work, all.size() * sizeof(int4)) != hipSuccess) return 1;
  if (hipMemcpy(c.wave_work, all.data(), all.size() * sizeof(int4), hipMemcpyHostToDevice) != hipSuccess) return 1;
  c.wave_nwork = (int)all.size() / 2;
  return 0;
}

// Compute units of the current device.
static int cu_count() {
  int cus = 0, dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus <= 0)
    cus = 256;
  return cus;
}

// The interior kernel (WaveInteriorKernel, see wave_work_list): -1 (default)
// picks 3 when the interior launch holds at least 16 rounds of resident 64 x 4
// blocks (three per CU; fewer rounds leave the last ones ragged:
// 1600 x 1000 x 500, 88 k blocks: 90-95 ms of interior per step against
// 96-101 for 1; 400 x 300 x 200, 2 k blocks: 2.50 against 2.16 ms), else 1.
// As the box beside the other tiles, ms per step with 3 and with 1, metric as
// bfloat16 deviations | FP32: 600 x 640 x 500, 19 k blocks, 28.3 and 31.1 | 32.6
// and 31.9; 400 x 300 x 200, 1.5 k blocks, 5.35 and 5.59 | 6.07 and 5.88 (the
// buffers' places in memory alone make 5% between two solvers of a process).
// cols: 64-wide tiles along j, rows along k, planes along i.
static int interior_kernel(const Params& p, long cols, long rows, long planes, int cus) {
  if (p.WaveInteriorKernel >= 0) return p.WaveInteriorKernel;
  return cols * (rows / TK4) * ((planes + 31) / 32) >= 16L * 3 * cus ? 3 : 1;
}

// Planes per block of a launch with one block per CU and few rounds of blocks
// (the ring kernel): it takes its rounds times the planes of a block and about
// two more for its start, and the last round may be nearly empty, so the
// length that takes the least (400 x 300 x 200, 84 tiles of 360 planes: 120
// planes in one round, 2.16 ms of interior per step; 2.37 with 32, 2.92 with
// 90).
static int rounds_chunk(int span, long ntiles, int cus) {
  int len = std::max(span, 1);
  long best = 0;
  for (int n = std::min(len, 8); n <= std::max(span, 1); n++) {
    const long t = (n + 2) * ((ntiles * ((span + n - 1) / n) + cus - 1) / cus);
    if (best == 0 || t < best) { best = t; len = n; }
  }
  return len;
}

// The work list of the unified launch: 32 x 8 tiles over the whole grid, or
// over all of it but the interior box, in chunks of planes; before it the
// box's tiles.  A wavefront's time is the same for a full and for a
// partial tile, and most grids leave less of a 32-wide tile empty than of a
// 64-wide one (ms of tiles per step, 64 x 4 -> 32 x 8: 100 x 200 x 100
// 0.52 -> 0.45, 151 x 211 x 133 1.60 -> 1.42, 200 x 160 x 120 1.30 -> 1.13;
// where 64 x 4 fits better, 97 x 125 x 81, level: 0.37).
static std::vector<int4> unified_work(Ctx& c, int cus) {
  const Params& p = c.p;
  const int ni = c.d.ni, nj = c.d.nj, nk = c.d.nk;
  c.wave_tall = c.wave_pipe = c.wave_ring = c.wave_band_pipe = c.wave_surf_pipe = false;
  c.pml_fused = true;
  c.wave_ktop = nk;
  // the interior box [i0, i1) x [j0, j1) x [k0, k1) in whole 64 x 8 tiles on
  // the 32 x 8 tiles' lattice (a lattice from the low bands' edges has larger
  // boxes, but partial tiles at all four sides: 512 x 384 x 256 11.7 against
  // 10.5 ms per step, 251 x 187 x 143 2.32 against 2.05)
  int i0 = 0, i1 = 0, j0 = 0, j1 = 0, k0 = 0, k1 = 0;
  if (p.WaveUnified == 2 || (p.WaveUnified < 0 && (double)p.NX * p.NY * p.NZ > kBoxPoints)) {
    int lo[3], hi[3];
    for (int ax = 0; ax < 3; ax++) {
      const int damp = p.useCerjan ? p.DAMP_N : 0;
      lo[ax] = std::max(c.pml.on[2 * ax] ? c.pml.N : 0, damp);
      hi[ax] = ax == 2 && p.FreeSurface ? 3 : std::max(c.pml.on[2 * ax + 1] ? c.pml.N : 0, damp);
    }
    i0 = std::min(lo[0], ni);
    i1 = std::max(i0, ni - hi[0]);
    j0 = (lo[1] + TJN - 1) / TJN * TJN;
    j1 = j0 + std::max(0, nj - hi[1] - j0) / TJ * TJ;
    k0 = (lo[2] + TKN - 1) / TKN * TKN;
    k1 = k0 + std::max(0, nk - hi[2] - k0) / TKN * TKN;
    if (i1 == i0 || j1 == j0 || k1 == k0) i1 = i0;
  }
  const long span = i1 - i0;
  std::vector<int4> box;
  if (span > 0) {
    c.wave_pipe = true;
    c.wave_ring = interior_kernel(p, (j1 - j0) / TJ, k1 - k0, span, cus) == 1;
    c.wave_tki = c.wave_ring ? (int)TK : (int)TK4;
    const int len = c.wave_ring ? rounds_chunk((int)span, (long)(j1 - j0) / TJ * ((k1 - k0) / TK), cus) : std::min((int)span, 32);
    for (int i = i0; i < i1; i += len)
      for (int k = k0; k < k1; k += c.wave_tki)
        for (int j = j0; j < j1; j += TJ) {
          box.push_back(make_int4(j, k, i, std::min(i1, i + len)));
          box.push_back(make_int4(TJ, c.wave_tki, 0, 0));
          count_block(c, 0, i, std::min(i1, i + len), j, j + TJ, k, k + c.wave_tki, false);
        }
  }
  // the other tiles: all of them on the planes outside the box, those around
  // it on its planes
  const long tiles = (long)((nj + TJN - 1) / TJN) * ((nk + TKN - 1) / TKN);
  const long around = tiles - (long)(j1 - j0) / TJN * ((k1 - k0) / TKN);
  auto blocks = [&](int n) {
    auto cut = [&](long planes) { return (planes + n - 1) / n; };
    return span > 0 ? tiles * (cut(i0) + cut(ni - i1)) + around * cut(span) : tiles * cut(ni);
  };
  int len = p.WaveBandIChunk;
  if (len <= 0) {
    // planes per block: a block takes about its planes and one more for its
    // start, the launch its blocks spread over the resident ones (two per CU)
    // and the last of them; shorter chunks for grids that would leave CUs
    // idle (151 x 211 x 133: 1.41 ms of tiles per step against 1.62 with 20
    // planes; 200 x 160 x 120: 1.13 against 1.35)
    double best = 0.0;
    for (int n = std::min(ni, 2); n <= std::min(ni, 20); n++) {
      const double t = (n + 1.0) * ((double)blocks(n) / (2.0 * cus) + 1.0);
      if (len <= 0 || t < best) { best = t; len = n; }
    }
  }
  std::vector<int4> rest;
  auto add = [&](int a, int b, bool whole) {
    for (int i = a; i < b; i += len)
      for (int k = 0; k < nk; k += TKN)
        for (int j = 0; j < nj; j += TJN) {
          if (!whole && j >= j0 && j < j1 && k >= k0 && k < k1) continue;
          const int ie = std::min(b, i + len), w = std::min((int)TJN, nj - j), h = std::min((int)TKN, nk - k);
          rest.push_back(make_int4(j, k, i, ie));
          rest.push_back(make_int4(w, h, 0, 0));
          count_block(c, 1, i, ie, j, j + w, k, k + h, true);
        }
  };
  if (span > 0) {
    add(0, i0, true);
    add(i0, i1, false);
    add(i1, ni, true);
  } else {
    add(0, ni, true);
  }
  for (int l = 0; l < 4; l++) c.wave_nkind[l] = 0;
  c.wave_nkind[0] = (int)box.size() / 2;
  c.wave_nkind[1] = (int)rest.size() / 2;
  c.pml_nbox = c.pml_blocks = 0;
  box.insert(box.end(), rest.begin(), rest.end());
  return box;
}

// True when the two ADE-PML bands of every axis are disjoint (2 N <= the axis
// length), which the pipelined kernels' one face per axis and point needs.
static bool bands_disjoint(const Params& p) {
  if (!p.usePML) return true;
  return 2 * p.PML_N <= p.NX && 2 * p.PML_N <= p.NY && (p.FreeSurface || 2 * p.PML_N <= p.NZ);
}

// One launch of tiles of any kind instead of one per kind, and beside it, with
// a box, the interior kernel on the interior tiles: WaveUnified 1 (without the
// box) or 2 (with it), or -1 (default) without any of the per-kind launch
// options: 1 up to kBoxPoints points, 2 up to kPerKindPoints, one launch per
// kind above.  WaveInteriorKernel 1 or 3 with WaveUnified 2 names the box's
// kernel.  Each launch ends with CUs idle while its last blocks run, and
// the launches of a stage run one after another, so small grids take one;
// the box's kernel streams interior points at twice the rate, which pays
// for a second launch, and the many blocks of a large grid make the tiles of
// each kind's own shape the better choice.  ms per step with one launch, with
// the box, and per kind:
//   97 x 125 x 81    0.36   0.43   1.52
//   200 x 160 x 120  1.32   1.31
//   251 x 187 x 143  2.15   2.05   2.83
//   400 x 300 x 200  6.20   5.91   6.00
//   512 x 384 x 256  11.1   10.5   12.2
//   560 x 640 x 440         23.3   25.6
//   640 x 512 x 400         25.1   27.3
//   600 x 640 x 500         27.9   30.7
//   700 x 750 x 500         39.3   38.5
//   800 x 1000 x 500 71.8   57.1   55.8
// (with FP32 metric words 560 x 640 x 440 25.9 and 31.4, 600 x 640 x 500 30.8
// and 33.1, 700 x 750 x 500 44.2 and 44.1)
bool wave_unified(const Params& p) {
  if (p.WaveUnified == 0 || !bands_disjoint(p)) return false;
  const bool box_kernel = p.WaveUnified == 2 && (p.WaveInteriorKernel == 1 || p.WaveInteriorKernel == 3);
  if ((p.WaveInteriorKernel != -1 && !box_kernel) || p.WaveBandKernel != -1 || p.WaveSurfaceKernel != 1 || p.WaveSurfaceTiles != 1 ||
      p.WaveTallInterior || p.WaveBandRound || !p.PmlAuxFused || p.StageStreams || p.WaveIChunk || p.WaveTopIChunk)
    return false;
  return p.WaveUnified > 0 || (double)p.NX * p.NY * p.NZ <= kPerKindPoints;
}

// With one launch per kind the interior box excludes every face band where a
// PML profile or the Cerjan sponge is non-trivial and the three free-surface
// rows; its tiles start at the box edge so that no interior tile straddles a
// band.  Interior items come first, then the edge items; each list is
// chunk-major so that one XCD's contiguous share covers neighbouring tiles.
std::vector<int4> wave_work_list(Ctx& c, int cus, std::vector<int>& boxes) {
  boxes.clear();
  clear_counts(c);
  const Params& p = c.p;
  const int n3[3] = {c.d.ni, c.d.nj, c.d.nk};
  c.wave_unified = wave_unified(p);
  if (c.wave_unified) return unified_work(c, cus);
  const bool freenode = p.FreeSurface != 0;
  int lo[3], hi[3];
  for (int ax = 0; ax < 3; ax++) {
    lo[ax] = ax == 1 ? interior_lo_j(p) : std::max(c.pml.on[2 * ax] ? c.pml.N : 0, p.useCerjan ? p.DAMP_N : 0);
    hi[ax] = std::max(c.pml.on[2 * ax + 1] ? c.pml.N : 0, p.useCerjan && (ax < 2 || !freenode) ? p.DAMP_N : 0);
  }
  // WaveSurfaceTiles: the free-surface tiles are exactly the top TK rows
  // (full tiles) and the interior's k remainder joins the low band instead;
  // their j tiles are laid out on their own, line-aligned and full width
  const bool surf = freenode && p.WaveSurfaceTiles != 0;
  if (freenode) hi[2] = std::max(hi[2], surf ? TK : 3);
  // the interior box holds whole tiles along j and k: a remainder joins the
  // high-side band (or the free-surface tiles), whose kernels treat any point
  // (WaveTallInterior: interior tiles of 2 TK rows in blocks of 2 NTHR
  // threads, which re-read the k halo rows for twice as many points)
  const bool tall = p.WaveTallInterior != 0;
  c.wave_tall = tall;
  // WaveInteriorKernel: 0 the general kernel on the interior tiles, 1 the
  // pipelined interior kernel (64 x 8 tiles, LDS plane ring, one block per
  // CU), 2 the pipelined kernel on 64 x 6 tiles (384 threads, two blocks per
  // CU), 3 on 64 x 4 tiles (256 threads, three blocks per CU), 4 on 64 x 8
  // tiles with an LDS double buffer instead of the ring
  const int wik = interior_kernel(p, std::max(0, n3[1] - lo[1] - hi[1]) / TJ, std::max(0, n3[2] - lo[2] - hi[2]),
                                  std::max(0, n3[0] - lo[0] - hi[0]), cus);
  c.wave_pipe = !tall && wik >= 1;
  c.wave_ring = wik == 1;
  // WaveBandKernel 1: the pipelined kernel on the band tiles too, which adds
  // the aux terms of one face per axis: used when the two ADE-PML bands of
  // every axis are disjoint (2 N <= the axis length)
  const bool disjoint = bands_disjoint(p);
  // -1 (automatic): 64 x 4 band tiles beside the 64 x 4 interior tiles of a
  // large grid, 64 x 8 ones on a grid too small for those (400 x 300 x 200:
  // bands 3.28 against 3.35 ms per step)
  const int wbk = p.WaveBandKernel >= 0 ? p.WaveBandKernel : wik == 3 ? 2 : 1;
  c.wave_band_pipe = wbk >= 1 && disjoint;
  c.wave_band_tk = c.wave_band_pipe && wbk == 2 ? TK4 : TK;  // 2: 64 x 4 band tiles, two blocks per CU
  // WaveSurfaceKernel 1: the pipelined kernel on the free-surface tiles too
  // (with the band terms and, with PmlAuxFused, the auxiliary fields)
  c.wave_surf_pipe = disjoint && p.WaveSurfaceKernel >= 1;
  // PmlAuxFused 1: the pipelined band and free-surface tiles advance their
  // points' auxiliary fields; pml_aux_kernel runs on the free-surface rows
  // when those run the general kernel, and on everything with the general
  // band kernel
  c.pml_fused = c.wave_band_pipe && p.PmlAuxFused != 0;
  const int tki = tall ? 2 * TK : (c.wave_pipe && wik == 2) ? TK6 : (c.wave_pipe && wik == 3) ? TK4 : TK;  // interior tile rows
  c.wave_tki = tki;
  for (int ax = 1; ax < 3; ax++) {
    const int t = ax == 1 ? TJ : tki, e = n3[ax] - lo[ax] - hi[ax];
    if (e > t) (ax == 2 && surf ? lo[ax] : hi[ax]) += e % t;
  }
  const std::vector<Seg> sj = axis_segments(n3[1], lo[1], hi[1], TJ);
  const std::vector<Seg> sk = axis_segments(n3[2], lo[2], hi[2], TK);
  const std::vector<Seg> ski = tki != TK ? axis_segments(n3[2], lo[2], hi[2], tki) : sk;  // interior tiles' rows
  const std::vector<Seg>& sji = sj;
  const int nk = n3[2];
  auto is_top = [&](const Seg& b) { return freenode && b.s + b.n > nk - 3; };
  std::vector<Seg> sjt = sj;  // j tiles of the free-surface rows
  if (surf) {
    sjt.clear();
    const int s0 = lo[1] - 32 * ((lo[1] + 31) / 32);  // j = s0 starts a 128-byte line
    for (int x = s0; x < n3[1]; x += TJ) sjt.push_back({x, std::min(TJ, n3[1] - x), false, std::max(0, -x)});
  }
  int tiles[3] = {0, 0, 0};
  for (const Seg& b : sk)
    for (const Seg& a : sj)
      if (!is_top(b)) tiles[a.in && b.in ? 0 : 1]++;
  for (const Seg& b : sk)
    if (is_top(b)) tiles[2] += (int)sjt.size();
  int tiles_in = 0;  // interior blocks per chunk
  for (const Seg& b : ski)
    for (const Seg& a : sji) tiles_in += a.in && b.in;
  const int ni = n3[0], ia = std::min(lo[0], ni), ib = std::max(ia, ni - hi[0]);
  // planes per block of each kind: short chunks (several thousand blocks per
  // launch) balance the CUs better than the longer chunks would save on the
  // 4-plane warm-up of the x-queue; the few free-surface tiles take at least
  // 4 planes too (shorter chunks re-read the warm-up planes for 1-2 planes
  // of work; 0.58 against 0.52 ms per step on 400 x 300 x 200)
  auto chunk = [&](int span, int ntiles, int target, int minlen) {
    span = std::max(span, 1);
    const int chunks = std::max(1, std::min(span, (target + std::max(ntiles, 1) - 1) / std::max(ntiles, 1)));
    return std::max((span + chunks - 1) / chunks, std::min(minlen, span));
  };
  // The pipelined interior kernel streams 32 planes per block: its loads
  // overlap the compute, so a longer chunk mostly saves warm-up planes
  // (1600 x 1000 x 500: 97.7 ms of interior per step against 106.2 for the
  // ~300-plane chunks of a 4096-block target and 104.5 for 16 planes;
  // 400 x 300 x 200: 2.44 against 2.70 ms for ~8 planes).
  const int ich_in = p.WaveIChunk > 0 ? p.WaveIChunk
                     : c.wave_ring   ? rounds_chunk(ib - ia, tiles_in, cus)
                     : c.wave_pipe   ? std::min(std::max(ib - ia, 1), 32)
                                     : chunk(ib - ia, tiles_in, tall ? 2048 : 4096, 4);
  // band tiles stream 20 planes (1600 x 1000 x 500: 23.4 ms per step against
  // 24.6, 25.0 and 32.9 for 16, 32 and 48 planes and 29.6 for the ~4 planes
  // of an 8192-block target; 400 x 300 x 200: 2.55 against 2.68 ms)
  const int ich_band = p.WaveBandIChunk > 0 ? p.WaveBandIChunk : std::min(std::max(ni, 1), 20);
  const int ich_top = p.WaveTopIChunk > 0 ? p.WaveTopIChunk : chunk(ni, tiles[2], 2048, 4);
  // lists: 0 interior, 1 absorbing bands (64-wide tiles), 2 absorbing bands
  // of at most 32 columns along j (32 x 16 tiles, half the idle lanes),
  // 3 tiles holding free-surface rows
  std::vector<int4> lists[4];
  auto push = [&](int list, const Seg& a, const Seg& b, int i0, int i1) {
    lists[list].push_back(make_int4(a.s, b.s, i0, i1));
    lists[list].push_back(make_int4(a.n, b.n, a.o, b.o));
    const int kd = list == 0 ? 0 : list == 3 ? 2 : 1;
    // the fused update in the band tiles and the pipelined free-surface tiles
    count_block(c, kd, i0, i1, a.s + a.o, a.s + a.n, b.s + b.o, b.s + b.n, c.pml_fused && (kd == 1 || (kd == 2 && c.wave_surf_pipe)));
  };
  const auto narrow = [&](const Seg& a) { return !a.in && a.n - a.o <= TJN; };
  // bands of at most TJB columns get tiles exactly TJB wide (with the
  // pipelined band kernel), so that a 20-column band keeps every lane busy
  // (a 32-wide tile idles 12 of its 32; 1600 x 1000 x 500: 2.8 ms per stage
  // for the 32 M points of the two j bands against 2.4 ms for the 48 M
  // points of the 64-wide band tiles); wider narrow bands get TJN x TKN tiles
  int wmax = 0;
  for (const Seg& a : sj)
    if (narrow(a)) wmax = std::max(wmax, a.n - a.o);
  const bool exact = c.wave_band_pipe && wmax > 0 && wmax <= TJB;
  const int tjn = exact ? TJB : TJN, tkn = exact ? TKB : TKN;
  c.wave_tjn = tjn;
  // the same active columns in a tjn-wide tile: anchored at the interior
  // edge on the low side, at the band start on the high side
  const auto narrowed = [&](const Seg& a) {
    const int w = a.n - a.o;
    return a.o > 0 ? Seg{a.s + a.n - tjn, tjn, false, tjn - w} : Seg{a.s, w, false, 0};
  };
  int ktop = nk;  // first row of the free-surface tiles
  for (const Seg& b : sk)
    if (is_top(b)) ktop = std::min(ktop, b.s);
  c.wave_ktop = ktop;
  for (int i0 = ia; i0 < ib; i0 += ich_in)
    for (const Seg& b : ski) for (const Seg& a : sji) if (a.in && b.in) push(0, a, b, i0, std::min(ib, i0 + ich_in));
  // band tiles of TK rows, or of TK4 rows with WaveBandKernel 2 (the rows
  // from ktop up are the free-surface tiles')
  const std::vector<Seg> skb = c.wave_band_tk == TK4 ? axis_segments(n3[2], lo[2], hi[2], TK4) : sk;
  for (int i0 = 0; i0 < ni; i0 += ich_band)
    for (const Seg& b : skb)
      for (const Seg& a : sj) {
        const int i1 = std::min(ni, i0 + ich_band);
        if (b.s >= ktop || narrow(a)) continue;
        if (!(a.in && b.in)) { push(1, a, b, i0, i1); continue; }
        // interior tile: only the parts of [i0, i1) outside [ia, ib)
        if (i0 < ia) push(1, a, b, i0, std::min(i1, ia));
        if (i1 > ib) push(1, a, b, std::max(i0, ib), i1);
      }
  for (int i0 = 0; i0 < ni; i0 += ich_band)
    for (int k0 = 0; k0 < ktop; k0 += tkn)
      for (const Seg& a : sj)
        if (narrow(a)) push(2, narrowed(a), Seg{k0, std::min(tkn, ktop - k0), false, 0}, i0, std::min(ni, i0 + ich_band));
  for (int i0 = 0; i0 < ni; i0 += ich_top)
    for (const Seg& b : sk)
      if (is_top(b))
        for (const Seg& a : sjt) push(3, a, b, i0, std::min(ni, i0 + ich_top));
  // boxes of the auxiliary-update kernel: every absorbing face whole; with
  // the fused update only the points the tiles leave to it, the rows from
  // ktop up when their tiles run the general kernel
  {
    const int N = c.pml.N;
    std::vector<int>& bx = boxes;
    int blocks = 0;
    // box in face-local (j, k, i) coordinates
    auto add = [&](int f, int j0, int nj_, int k0, int nk_, int i0, int ni_) {
      if (nj_ <= 0 || nk_ <= 0 || ni_ <= 0) return;
      bx.insert(bx.end(), {f, j0, nj_, k0, nk_, i0, ni_, blocks});
      blocks += (int)(((long)nj_ * nk_ * ni_ + 255) / 256);
      c.aux_update_pairs[3] += (long)nj_ * nk_ * ni_;
    };
    for (int f = 0; f < 6; f++) {
      if (!c.pml.on[f] || (c.pml_fused && c.wave_surf_pipe)) continue;
      // per axis the face's first point and the one past its last; of a layer
      // wider than the axis only the points of the grid
      int p0[3], p1[3];
      for (int ax = 0; ax < 3; ax++) {
        const bool own = ax == f / 2;
        p0[ax] = own && (f & 1) ? std::max(N - n3[ax], 0) : 0;
        p1[ax] = !own ? n3[ax] : (f & 1) ? N : std::min(N, n3[ax]);
      }
      if (c.pml_fused) p0[2] = std::max(p0[2], ktop - (f == 5 ? nk - N : 0));
      add(f, p0[1], p1[1] - p0[1], p0[2], p1[2] - p0[2], p0[0], p1[0] - p0[0]);
    }
    c.pml_nbox = (int)bx.size() / kPmlBoxInts;
    c.pml_blocks = blocks;
  }
  std::vector<int4> all;
  for (int l = 0; l < 4; l++) {
    all.insert(all.end(), lists[l].begin(), lists[l].end());
    c.wave_nkind[l] = (int)lists[l].size() / 2;
  }
  return all;
}

// Builds and uploads the stage-kernel work lists and allocates the
// free-surface buffer.
int upload_wave_work(Ctx& c) {
  if (c.p.FreeSurface && !c.img_top) {  // the image stencil reaches six rows down (NZ >= 7)
    if (hipMalloc(&c.img_top, sizeof(float) * 18 * (size_t)c.d.ni * c.d.nj) != hipSuccess) return 1;
    c.allocations.push_back(c.img_top);
  }
  std::vector<int> boxes;
  const std::vector<int4> all = wave_work_list(c, cu_count(), boxes);
  if (c.pml_boxes) { (void)hipFree(c.pml_boxes); c.pml_boxes = nullptr; }
  if (!boxes.empty()) {
    if (hipMalloc(&c.pml_boxes, boxes.size() * sizeof(int)) != hipSuccess) return 1;
    if (hipMemcpy(c.pml_boxes, boxes.data(), boxes.size() * sizeof(int), hipMemcpyHostToDevice) != hipSuccess) return 1;
  }
  return put_work(c, all);
}

void launch_wave_stage(Ctx& c, const StageBufs& b, int irk, int fx, int fy, int fz, bool rhs_only, float* rhs_out) {
  if (c.p.MetricBF16 == 2) {
    WaveArgs<MetBf16Delta> a = make_args<MetBf16Delta>(c, b, irk, rhs_only, rhs_out);
    launch_wave_dispatch(a, c, fx, fy, fz, c.stream);
  } else if (c.p.MetricBF16) {
    WaveArgs<uint16_t> a = make_args<uint16_t>(c, b, irk, rhs_only, rhs_out);
    launch_wave_dispatch(a, c, fx, fy, fz, c.stream);
  } else {
    WaveArgs<float> a = make_args<float>(c, b, irk, rhs_only, rhs_out);
    launch_wave_dispatch(a, c, fx, fy, fz, c.stream);
  }
}

}  // namespace cgfdm
