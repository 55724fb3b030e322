// rows3d.h -- D3Q27 stream+collide tile of whole 64-cell rows, for domains
// without a body whose grid fills the chip with them (rows3d_chunks).
//
// The arithmetic is that of the staged columns of stencil.h (recon3 and
// collide3 in either form), so the results are the same bit for bit.
// Bounce-back walls are left to the columns.
#pragma once

#include "ff_internal.h"
#include "hermite.h"
#include "separable3d.h"
#include "stencil.h"

namespace ff {

// Tile: 64 x 6 cells marching along z, one wave per row and two waves for the
// rows below and above, which also take the columns left and right of the
// tile (a plane ahead).  x neighbours are the wave's own lanes (DPP), y
// neighbours pass nine populations each way through a double-buffered LDS
// plane, z neighbours wait in registers: one barrier a plane, 100 VGPRs and
// 57 KB of LDS, two blocks a CU.
// The staged columns are bound by the lines between L2 and L1, not by their
// arithmetic: a copy that reads 32x12 tiles with their halo in 16 bits takes
// 143 us at 256x192x160 (14 rows of three 128-byte lines for 384 cells), as
// long as the whole step, and 70 us in rows of 64 with the side columns.
// 256x192x160: FP16 fast 147 -> 113 us (split velocity 177 -> 139), FP32
// reference order 189 -> 163; 250x150x150: 102 -> 78, 144 -> 110, 173 -> 141.
// Rows of 8 (96 VGPRs, 5 spilled) 146 us in FP16.
constexpr int kRowsThreads = 64 * (kRowsTY + 2);

// The domain's whole rows: their z chunks, or 0 if it steps with the tiles.
inline int rows3d_plan(const Domain& d) {
  if (d.dim != 3 || !d.rows3 || (d.has_boundary && d.ne > 0) || d.walls3) return 0;
  return d.row_chunks;
}

// Stored moments of a cell, `r` from the start of a z-plane on, moment planes
// `pb` bytes apart, the lane's byte offset `off` (kNoCell: dropped).  `load`
// leaves the moments as stored, so that nothing waits for them before they
// are used; `value` decodes, `store` encodes: for the 16-bit formats with the
// rounding and scaling of Store<S> (on a register copy).  h16u has the low
// halves of the velocity behind the ten.
template <typename S> struct RowIo {
  static constexpr bool kLow = std::is_same<S, h16u>::value;
  static constexpr int kRaw = kLow ? 13 : 10;
  using Raw = unsigned short;
  static __device__ __forceinline__ void load(BufRsrc r, unsigned off, unsigned pb, Raw* m) {
#pragma unroll
    for (int q = 0; q < kRaw; q++) m[q] = __builtin_amdgcn_raw_buffer_load_b16(r, (int)off, (int)(q * pb), 0);
  }
  static __device__ __forceinline__ void value(const Raw* r, float* m) {
#pragma unroll
    for (int q = 0; q < 10; q++) {
      S v[10];
      __builtin_memcpy(&v[0], &r[q], 2);
      if constexpr (kLow)
        if (q >= 1 && q <= 3) __builtin_memcpy(&v[9], &r[q + 9], 2);
      m[q] = Store<S>::template load<3>(v, q, 1);
    }
  }
  static __device__ __forceinline__ void store(BufRsrc r, unsigned off, unsigned pb, const float* m) {
#pragma unroll
    for (int q = 0; q < 10; q++) {
      S v[10];
      Raw b;
      Store<S>::template store<3>(v, q, m[q], 1);
      __builtin_memcpy(&b, &v[0], 2);
      __builtin_amdgcn_raw_buffer_store_b16(b, r, (int)off, (int)(q * pb), 0);
      if constexpr (kLow)
        if (q >= 1 && q <= 3) {
          __builtin_memcpy(&b, &v[9], 2);
          __builtin_amdgcn_raw_buffer_store_b16(b, r, (int)off, (int)((q + 9) * pb), 0);
        }
    }
  }
};
template <> struct RowIo<float> {
  static constexpr int kRaw = 10;
  using Raw = float;
  static __device__ __forceinline__ void load(BufRsrc r, unsigned off, unsigned pb, Raw* m) {
#pragma unroll
    for (int q = 0; q < 10; q++) m[q] = sep_load(r, off, pb, q);
  }
  static __device__ __forceinline__ void value(const Raw* r, float* m) {
#pragma unroll
    for (int q = 0; q < 10; q++) m[q] = r[q];
  }
  static __device__ __forceinline__ void store(BufRsrc r, unsigned off, unsigned pb, const float* m) {
#pragma unroll
    for (int q = 0; q < 10; q++) sep_store(r, off, pb, q, m[q]);
  }
};

// positions of direction i among the nine that share its c_x, its c_y
__host__ __device__ constexpr int xclass_index(int i) {
  int n = 0;
  for (int j = 0; j < i; j++) n += D3::cx(j) == D3::cx(i) ? 1 : 0;
  return n;
}
__host__ __device__ constexpr int yclass_index(int i) {
  int n = 0;
  for (int j = 0; j < i; j++) n += D3::cy(j) == D3::cy(i) ? 1 : 0;
  return n;
}

struct Rows3Lds {
  // pulled in x: the nine c_y = +1 populations of the row below and the nine
  // c_y = -1 ones of the row above each row
  float up[2][9][kRowsTY][64], dn[2][9][kRowsTY][64];
  // the nine c_x = +1 populations of the cell left and the nine c_x = -1 ones
  // of the cell right of each row, -1 to TY
  float side[2][2][kRowsTY + 2][kSepSide];
};

template <typename S, bool PERIODIC, bool FAST>
__device__ __forceinline__ void bulk3d_rows(const S* __restrict__ in, S* __restrict__ out,
                                            const uint8_t* __restrict__ flags, int nx, int ny, int nz, size_t plane,
                                            float omega, int bx, int by, int z0, int zend, Rows3Lds& lds) {
  constexpr int TY = kRowsTY;
  using Io = RowIo<S>;
  using Raw = typename Io::Raw;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = (int)(threadIdx.x & 63u);
  const int x0 = bx * kRowsTX, y0 = by * TY;
  const size_t nxy = (size_t)nx * ny;
  const unsigned pb = (unsigned)(plane * sizeof(S));  // bytes of a moment plane
  auto src_x = [&](int gx) { return PERIODIC ? ((gx % nx) + nx) % nx : min(nx - 1, max(0, gx)); };
  auto src_y = [&](int gy) { return PERIODIC ? ((gy % ny) + ny) % ny : min(ny - 1, max(0, gy)); };
  // planes z0 - 1 to zend (one wrap at most), numbered from 0; past the last one it is taken again
  const int np = zend - z0 + 2;
  auto plane_at = [&](int i) {
    const int gz = z0 - 1 + min(i, np - 1);
    return (unsigned)(PERIODIC ? (gz < 0 ? gz + nz : (gz >= nz ? gz - nz : gz)) : min(nz - 1, max(0, gz))) * nxy;
  };
  auto load = [&](int i, unsigned off, Raw* m) { Io::load(buf_rsrc(in + plane_at(i)), off, pb, m); };
  auto recon = [&](const Raw* r, float* f) {
    float m[10];
    Io::value(r, m);
    if constexpr (FAST) recon3_fast(m, f);
    else recon3_all(m, f);
  };
  // the row's populations pulled in x (f in and out), and those that its neighbour rows pull
  auto row_stage = [&](float* f, int buf, int row, bool to_up, bool to_down) {
    float el[9], er[9];
#pragma unroll
    for (int k = 0; k < 9; k++) {
      el[k] = lds.side[buf][0][row + 1][k];
      er[k] = lds.side[buf][1][row + 1][k];
    }
#pragma unroll
    for (int i = 0; i < 27; i++) {
      if (D3::cx(i) > 0) f[i] = lane_before(el[xclass_index(i)], f[i]);
      if (D3::cx(i) < 0) f[i] = lane_after(er[xclass_index(i)], f[i]);
      if (D3::cy(i) > 0 && to_up) lds.up[buf][yclass_index(i)][row + 1][lane] = f[i];
      if (D3::cy(i) < 0 && to_down) lds.dn[buf][yclass_index(i)][row - 1][lane] = f[i];
    }
  };
  if (wave < TY) {
    const int x = x0 + lane, y = y0 + wave;
    const bool inside = x < nx && y < ny;
    const unsigned src = (unsigned)(src_y(y) * nx + src_x(x));
    const unsigned cell = inside ? (unsigned)(y * nx + x) : 0u;  // in its plane
    Raw m[Io::kRaw];
    uint8_t fl = 0, fout = 0;
    load(0, src * sizeof(S), m);
    // c_z = +1 of the plane below the output's and of the output's own plane,
    // c_z = 0 of the output's plane
    float below[9], up[9], mid[9];
#pragma unroll
    for (int k = 0; k < 9; k++) below[k] = up[k] = mid[k] = 0.0f;
    auto put_results = [&](S* to_plane, unsigned to, const float* o) { Io::store(buf_rsrc(to_plane), to, pb, o); };
    {
      // as many (dropped) stores as a pass ends with: the wait for the moments
      // at its top then counts them out in the first pass too
      const float none[10] = {};
      put_results(out, kNoCell, none);
    }
    S* out_plane = out + (size_t)z0 * nxy;
    __syncthreads();  // the side columns of the first plane
    for (int i = 0; i < np; i++) {
      const int K = i & 1;
      float f[27];
      recon(m, f);
      const uint8_t fz = fl;
      load(i + 1, src * sizeof(S), m);
      fl = __builtin_amdgcn_raw_buffer_load_b8(buf_rsrc(flags + plane_at(i + 1)), (int)cell, 0, 0);
      row_stage(f, K, wave, wave + 1 < TY, wave >= 1);
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 27; k++) {
        if (D3::cy(k) > 0) f[k] = lds.up[K][yclass_index(k)][wave][lane];
        if (D3::cy(k) < 0) f[k] = lds.dn[K][yclass_index(k)][wave][lane];
        f[k] = clamp0(f[k]);
      }
      float p[27], o[10];
#pragma unroll
      for (int k = 0; k < 27; k++) {
        const int j = zclass_index(k);
        p[k] = D3::cz(k) > 0 ? below[j] : (D3::cz(k) < 0 ? f[k] : mid[j]);
      }
      if constexpr (FAST) collide3_fast(p, omega, o);
      else collide3(p, omega, o);
      // output plane z0 + i - 2, from the third plane on
      const unsigned to = (i >= 2 && inside && is_updated(fout)) ? (unsigned)(cell * sizeof(S)) : kNoCell;
      put_results(out_plane, to, o);
      if (i >= 2) out_plane += nxy;
      fout = fz;  // the flag of this pass's plane, the next output
#pragma unroll
      for (int k = 0; k < 27; k++) {
        const int j = zclass_index(k);
        if (D3::cz(k) > 0) {
          below[j] = up[j];
          up[j] = f[k];
        } else if (D3::cz(k) == 0) {
          mid[j] = f[k];
        }
      }
    }
  } else {
    const bool upper = wave == TY + 1;  // row TY and the right column, or row -1 and the left column
    const int row = upper ? TY : -1;
    const unsigned off = (unsigned)(src_y(y0 + row) * nx + src_x(x0 + lane)) * sizeof(S);
    const int srow = min(lane, TY + 1);  // side cell of this lane: row srow - 1
    const unsigned soff =
        (unsigned)(src_y(y0 + srow - 1) * nx + src_x(upper ? x0 + kRowsTX : x0 - 1)) * sizeof(S);
    auto side = [&](const Raw* r, int buf) {
      float f[27];
      recon(r, f);
      if (lane < TY + 2) {
#pragma unroll
        for (int i = 0; i < 27; i++) {
          if (upper && D3::cx(i) < 0) lds.side[buf][1][lane][xclass_index(i)] = f[i];
          if (!upper && D3::cx(i) > 0) lds.side[buf][0][lane][xclass_index(i)] = f[i];
        }
      }
    };
    Raw m[Io::kRaw], ms[Io::kRaw];
    load(0, soff, ms);
    load(0, off, m);
    side(ms, 0);
    load(1, soff, ms);
    __syncthreads();
    for (int i = 0; i < np; i++) {
      const int K = i & 1;
      float f[27];
      recon(m, f);
      load(i + 1, off, m);
      row_stage(f, K, row, !upper, upper);
      side(ms, K ^ 1);  // the side columns of the next plane
      load(i + 2, soff, ms);
      __syncthreads();
    }
  }
}

// Tile t of a domain's tiles_x x tiles_y x chunks grid.
template <typename S, bool PERIODIC, bool FAST>
__device__ __forceinline__ void rows3d_tile(const S* in, S* out, const uint8_t* flags, int nx, int ny, int nz,
                                            size_t plane, float omega, int tiles_x, int tiles_y, int chunks, int t,
                                            Rows3Lds& lds) {
  const int bx = t % tiles_x, by = (t / tiles_x) % tiles_y, bz = t / (tiles_x * tiles_y);
  const int z0 = (int)((long long)bz * nz / chunks), zend = (int)((long long)(bz + 1) * nz / chunks);
  bulk3d_rows<S, PERIODIC, FAST>(in, out, flags, nx, ny, nz, plane, omega, bx, by, z0, zend, lds);
}

}  // namespace ff
