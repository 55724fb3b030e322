// Prints how 3D grids step (plan3d.h): for "nx ny nz" lines on the input, the
// z chunks of the separable form and of whole rows (0: not that form) and the
// default tile without and with a body, for FP32 and for 16-bit storage.  With
// an argument: the most planes of a chunk for all of them as one batch.
#include <cstdio>

#include "../../freeflow_amd/csrc/plan3d.h"

int main(int argc, char**) {
  int nx, ny, nz;
  std::vector<ff::Grid3> all;
  while (std::scanf("%d %d %d", &nx, &ny, &nz) == 3) {
    const ff::Grid3 g{nx, ny, nz};
    all.push_back(g);
    if (argc > 1) continue;
    const size_t plane = (size_t)(g.cells() + 255) / 256 * 256;
    std::printf("%d", ff::sep3d_chunks(g, plane));
    for (size_t elem : {4, 2})
      std::printf(" %d %d %d", ff::rows3d_chunks(g, plane, 10, elem), ff::default_tile3(g, plane, 10, elem, false),
                  ff::default_tile3(g, plane, 10, elem, true));
    std::printf("\n");
  }
  if (argc > 1) std::printf("%d\n", ff::batch_chunk_planes(all));
  return 0;
}
