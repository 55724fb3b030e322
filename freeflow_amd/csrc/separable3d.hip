// separable3d.hip -- 3D stream+collide launch of a domain stepped on its own:
// the separable form (separable3d.h) or whole rows (rows3d.h) where their
// rules say so, else the tiles (kernels3d.hip).

#include "ff_internal.h"
#include "rows3d.h"
#include "separable3d.h"
#include "stencil.h"

namespace ff {

template <bool PERIODIC>
__global__ void __launch_bounds__(kSepThreads, 5)
    k_sep3d(const float* __restrict__ in, float* __restrict__ out, const uint8_t* __restrict__ flags, int nx, int ny,
            int nz, size_t plane, float omega, int tiles_x, int tiles_y, int chunks, int ntiles) {
  const int t = xcd_tile(blockIdx.x, ntiles);
  if (t < 0) return;
  sep3d_tile<PERIODIC>(in, out, flags, nx, ny, nz, plane, omega, tiles_x, tiles_y, chunks, t);
}

void plan3d(Domain& d) {
  const Grid3 g{d.nx, d.ny, d.nz};
  d.sep_chunks = sep3d_chunks(g, d.plane);
  d.row_chunks = rows3d_chunks(g, d.plane, storage_planes(d.storage, 3), storage_bytes(d.storage));
}

// The form of the domain's next step (FF_FORM_*) and the tile that it takes
// where it has tiles.
int stream_form(const Domain& d, int* tile) {
  if (d.dim == 2) {
    *tile = d.tile2;
    return FF_FORM_TILES;
  }
  *tile = tile3_of(d, d.has_boundary && d.ne > 0);
  return sep3d_plan(d) ? FF_FORM_SEPARABLE : (rows3d_plan(d) ? FF_FORM_ROWS : FF_FORM_TILES);
}

int launch_bulk3d(Domain& d, const void* in, void* out) {
  const int chunks = sep3d_plan(d);
  if (!chunks) {
    const int rows = rows3d_plan(d);
    return rows ? launch_rows3d(d, in, out, rows) : launch_bulk3d_tiles(d, in, out);
  }
  const int tx = (d.nx + kSepTX - 1) / kSepTX, ty = (d.ny + kSepTY - 1) / kSepTY, nt = tx * ty * chunks;
  const auto k = (d.options & FF_OPT_PERIODIC) ? k_sep3d<true> : k_sep3d<false>;
  launch_timed(k, dim3(xcd_grid(nt)), dim3(kSepThreads), d.stream, d.tev0, d.tev1, (const float*)in, (float*)out,
               d.flags, d.nx, d.ny, d.nz, d.plane, d.omega, tx, ty, chunks, nt);
  FF_HIP(hipGetLastError());
  return FF_OK;
}

}  // namespace ff
