// rows3d.hip -- 3D stream+collide launch with tiles of whole rows (rows3d.h).

#include "ff_internal.h"
#include "rows3d.h"
#include "stencil.h"

namespace ff {

template <typename S, bool PERIODIC, bool FAST>
__global__ void __launch_bounds__(kRowsThreads, 4)
    k_rows3d(const S* __restrict__ in, S* __restrict__ out, const uint8_t* __restrict__ flags, int nx, int ny, int nz,
             size_t plane, float omega, int tiles_x, int tiles_y, int chunks, int ntiles) {
  __shared__ Rows3Lds lds;
  const int t = xcd_tile(blockIdx.x, ntiles);
  if (t < 0) return;
  rows3d_tile<S, PERIODIC, FAST>(in, out, flags, nx, ny, nz, plane, omega, tiles_x, tiles_y, chunks, t, lds);
}

template <typename S>
static int rows3d_typed(Domain& d, const void* in, void* out, int chunks) {
  const int tx = (d.nx + kRowsTX - 1) / kRowsTX, ty = (d.ny + kRowsTY - 1) / kRowsTY, nt = tx * ty * chunks;
  const bool per = d.options & FF_OPT_PERIODIC, fast = d.options & FF_OPT_FAST_MATH;
  const auto k = per ? (fast ? k_rows3d<S, true, true> : k_rows3d<S, true, false>)
                     : (fast ? k_rows3d<S, false, true> : k_rows3d<S, false, false>);
  launch_timed(k, dim3(xcd_grid(nt)), dim3(kRowsThreads), d.stream, d.tev0, d.tev1, (const S*)in, (S*)out, d.flags,
               d.nx, d.ny, d.nz, d.plane, d.omega, tx, ty, chunks, nt);
  FF_HIP(hipGetLastError());
  return FF_OK;
}

int launch_rows3d(Domain& d, const void* in, void* out, int chunks) {
  switch (d.storage) {
    case FF_STORAGE_F32: return rows3d_typed<float>(d, in, out, chunks);
    case FF_STORAGE_F16: return rows3d_typed<__half>(d, in, out, chunks);
    case FF_STORAGE_F16U: return rows3d_typed<h16u>(d, in, out, chunks);
    default: return rows3d_typed<__hip_bfloat16>(d, in, out, chunks);
  }
}

}  // namespace ff
