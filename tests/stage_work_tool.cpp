// Test helper: the stage kernels' work list for a parameter set, as the
// solver builds it at setup (wave_work_list), without a GPU.
//   stage_work_tool <compute units> KEY=VALUE...
// prints "what value..." lines, then one "item" line per block (list, first
// column, row and plane, end plane, columns and rows of the tile, first active
// column and row), one "box" line per box of the auxiliary-update kernel, and
// for the columns -64 .. nj+63 the profile index that a lane there reads.
#include "cgfdm_internal.h"
#include <cstdio>
#include <cstdlib>
#include <cstring>

using namespace cgfdm;

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  Ctx c;
  for (int a = 2; a < argc; a++) {
    const char* eq = std::strchr(argv[a], '=');
    if (!eq || c.p.set(std::string(argv[a], eq - argv[a]), std::atof(eq + 1))) {
      std::fprintf(stderr, "bad argument %s\n", argv[a]);
      return 2;
    }
  }
  c.p.derive();
  c.d.ni = c.p.ni; c.d.nj = c.p.nj; c.d.nk = c.p.nk;
  c.pml.N = c.p.PML_N;
  for (int f = 0; f < 6; f++) c.pml.on[f] = c.p.usePML && (f < 5 || !c.p.FreeSurface);
  std::vector<int> boxes;
  const std::vector<int4> w = wave_work_list(c, std::atoi(argv[1]), boxes);
  std::printf("unified %d\nring %d\npipe %d\ntki %d\ntjn %d\nband_tk %d\nband_pipe %d\nsurf_pipe %d\nfused %d\n", (int)c.wave_unified,
              (int)c.wave_ring, (int)c.wave_pipe, c.wave_tki, c.wave_tjn, c.wave_band_tk, (int)c.wave_band_pipe,
              (int)c.wave_surf_pipe, (int)c.pml_fused);
  std::printf("points %ld %ld %ld\n", c.wave_points[0], c.wave_points[1], c.wave_points[2]);
  std::printf("read %ld %ld %ld %ld\n", c.aux_read_pairs[0], c.aux_read_pairs[1], c.aux_read_pairs[2], c.aux_read_pairs[3]);
  std::printf("update %ld %ld %ld %ld\n", c.aux_update_pairs[0], c.aux_update_pairs[1], c.aux_update_pairs[2], c.aux_update_pairs[3]);
  size_t q = 0;
  for (int l = 0; l < 4; l++)
    for (int n = 0; n < c.wave_nkind[l]; n++, q += 2)
      std::printf("item %d %d %d %d %d %d %d %d %d\n", l, w[q].x, w[q].y, w[q].z, w[q].w, w[q + 1].x, w[q + 1].y, w[q + 1].z, w[q + 1].w);
  if (q != w.size()) return 1;
  for (size_t b = 0; b + 8 <= boxes.size(); b += 8) {
    std::printf("box");
    for (int v = 0; v < 8; v++) std::printf(" %d", boxes[b + v]);
    std::printf("\n");
  }
  std::printf("column");
  for (int j = -64; j < c.d.nj + 64; j++) std::printf(" %d", nearest_point(j, c.d.nj));
  std::printf("\n");
  return 0;
}
