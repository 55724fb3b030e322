// separable3d.h -- D3Q27 stream+collide in moment space, one axis at a time
// (the fast form of FP32 domains without a body and without bounce-back walls).
//
// The update needs only ten moments of the 27 pulled populations, and both
// the reconstruction and the pull are products over the axes: a population is
//   f(cx, cy, cz) = w(cx) w(cy) w(cz) sum_abc A_abc H_a(cx) H_b(cy) H_c(cz),
// with H_0 = 1, H_1 = c, H_2 = c^2 - 1/3 and the 17 coefficients A of orders
// up to three that the moment set has (LbmUtilsFunc.cu's third-order terms).
// Pulling along x and taking the x-moments a' = 0, 1, 2 turns the columns
// (b, c) of A into S_a'(b, c); the same along y gives T_a'b'(c) and along z
// the moments U_a'b'c'.  With w = (1, 4, 1) / 6 and the second-order
// coefficients kept divided by 3, one axis of one column is
//   F+ = A0 + 2 A2 + A1, F- = A0 + 2 A2 - A1, F0 = A0 - A2,
//   M0 = 4 F0 + F+(x-1) + F-(x+1), M1 = F+(x-1) - F-(x+1), M2 = F+(x-1) + F-(x+1)
// (6 times the moment).  No population is formed: about 250 instead of 420
// operations a cell, and 18 instead of 27 values exchanged through LDS.
//
// The reference clamps every pulled population at zero (FsiCoupling3D.cu:
// 209-285).  A cell whose populations are positive by the triangle inequality
// (sep_bound) needs no clamp; a wave with any other cell forms its cells'
// populations, and a cell with a negative one goes on with the columns of the
// clamped ones (sep_clamp), all nine of them.
// Columns are sums over a cell's populations, so one that is infinite or larger
// by orders than the others takes them with it, and they would reach all 26
// neighbours.  Blocks that meet such a cell (not tame) redo the cells around
// it from single populations (sep_redo).
#pragma once

#include "ff_internal.h"
#include "hermite.h"
#include "plan3d.h"

namespace ff {

// Column index of (b, c): 3 c + b.
constexpr int kSepCols = 9;

// The 17 coefficients; second-order factors divided by 3.
struct SepCoef {
  float r, x, y, z, xx, yy, zz, xy, yz, xz, xxy, xyy, xxz, xzz, yyz, yzz, xyz;
};

__device__ __forceinline__ SepCoef sep_coef(const float* m) {
  SepCoef A;
  const float rho = m[0], ux = m[1], uy = m[2], uz = m[3];
  const float pxx = m[4], pyy = m[5], pzz = m[6], pxy = m[7], pyz = m[8], pxz = m[9];
  const float r3 = 3.0f * rho, r15 = 1.5f * rho, r9 = 9.0f * rho;
  A.r = rho;
  A.x = r3 * ux;
  A.y = r3 * uy;
  A.z = r3 * uz;
  A.xx = r15 * pxx;
  A.yy = r15 * pyy;
  A.zz = r15 * pzz;
  A.xy = r9 * pxy;
  A.yz = r9 * pyz;
  A.xz = r9 * pxz;
  // 4.5 rho (u_b D_a + 2 P_ab u_a), D_a = P_aa - 2 u_a^2
  const float Dx = fmaf(-2.0f * ux, ux, pxx), Dy = fmaf(-2.0f * uy, uy, pyy), Dz = fmaf(-2.0f * uz, uz, pzz);
  const float hx = 1.5f * A.x, hy = 1.5f * A.y, hz = 1.5f * A.z;
  A.xxy = fmaf(hy, Dx, A.xy * ux);
  A.xyy = fmaf(hx, Dy, A.xy * uy);
  A.xxz = fmaf(hz, Dx, A.xz * ux);
  A.xzz = fmaf(hx, Dz, A.xz * uz);
  A.yyz = fmaf(hz, Dy, A.yz * uy);
  A.yzz = fmaf(hy, Dz, A.yz * uz);
  // 27 rho (P_xy u_z + P_yz u_x + P_xz u_y - 2 u_x u_y u_z)
  A.xyz = 3.0f * fmaf(A.xy, uz, fmaf(A.yz, ux, fmaf(A.xz, uy, (-4.0f * hx) * (uy * uz))));
  return A;
}

// By the triangle inequality, with s = sum |u_a|, p = sum |P_aa|, q = sum |P_ab|
// (a < b), |H_1| <= 1 and |H_2| <= 2/3, the terms of a population besides rho
// are at most rho times
//   first order 3 s, second order 3 p + 9 q,
//   third order sum over a != b of 9 |u_b D_a + 2 P_ab u_a| <= 9 s p + 18 s q + 4.5 s^3
//   (sum u_a^2 |u_b| <= s^3 / 4) and 27 (s q + 2 s^3 / 27).
// positive: every population of the cell is, with a margin far above the
// rounding of this sum.  tame: none exceeds rho by more than 256 times (a fluid
// has s below 1, p and q about s^2).  Both false for NaN and where rho overflows
// the columns.
struct SepBound {
  bool positive, tame;
};
__device__ __forceinline__ SepBound sep_bound(const float* m) {
  const float s = fabsf(m[1]) + fabsf(m[2]) + fabsf(m[3]);
  const float p = fabsf(m[4]) + fabsf(m[5]) + fabsf(m[6]);
  const float q = fabsf(m[7]) + fabsf(m[8]) + fabsf(m[9]);
  const float third = fmaf(9.0f, p, fmaf(45.0f, q, 6.5f * s * s));
  const float t = fmaf(3.0f, s + p, fmaf(9.0f, q, s * third));
  const bool finite = fabsf(m[0]) < 1e30f;
  return {t < 0.999f && m[0] > 0.0f && finite, t < 256.0f && finite};
}

// F-, F0, F+ along x of the nine columns of a cell.
struct SepX {
  float p[kSepCols], m[kSepCols], c[kSepCols];
};

// (values in, so that outputs may be the same variables)
__device__ __forceinline__ void sep_axis(float a0, float a1, float a2, float& p, float& m, float& c) {
  const float e = fmaf(2.0f, a2, a0);
  p = e + a1;
  m = e - a1;
  c = a0 - a2;
}

// F+ (s = 1) or F- (s = -1) alone.
__device__ __forceinline__ void sep_face(const SepCoef& A, float s, float* f) {
  f[0] = fmaf(s, A.x, fmaf(2.0f, A.xx, A.r));
  f[1] = fmaf(s, A.xy, fmaf(2.0f, A.xxy, A.y));
  f[2] = fmaf(s, A.xyy, A.yy);
  f[3] = fmaf(s, A.xz, fmaf(2.0f, A.xxz, A.z));
  f[4] = fmaf(s, A.xyz, A.yz);
  f[5] = A.yyz;
  f[6] = fmaf(s, A.xzz, A.zz);
  f[7] = A.yzz;
  f[8] = 0.0f;
}

__device__ __forceinline__ void sep_columns(const SepCoef& A, SepX& X) {
  sep_axis(A.r, A.x, A.xx, X.p[0], X.m[0], X.c[0]);
  sep_axis(A.y, A.xy, A.xxy, X.p[1], X.m[1], X.c[1]);
  X.p[2] = A.yy + A.xyy;
  X.m[2] = A.yy - A.xyy;
  X.c[2] = A.yy;
  sep_axis(A.z, A.xz, A.xxz, X.p[3], X.m[3], X.c[3]);
  X.p[4] = A.yz + A.xyz;
  X.m[4] = A.yz - A.xyz;
  X.c[4] = A.yz;
  X.p[5] = X.m[5] = X.c[5] = A.yyz;
  X.p[6] = A.zz + A.xzz;
  X.m[6] = A.zz - A.xzz;
  X.c[6] = A.zz;
  X.p[7] = X.m[7] = X.c[7] = A.yzz;
  X.p[8] = X.m[8] = X.c[8] = 0.0f;
}

// Inverse of sep_axis.
__device__ __forceinline__ void sep_inverse(float fp, float fm, float fc, float& a0, float& a1, float& a2) {
  const float e = 0.5f * (fp + fm);
  a1 = 0.5f * (fp - fm);
  a2 = (e - fc) * (1.0f / 3.0f);
  a0 = fc + a2;
}

// Columns of one c_x (a row of SepX) with its nine populations (divided by
// their weights) clamped at zero; unchanged if none is negative.
__device__ __forceinline__ void sep_clamp(float* col) {
  float f[3][3];  // [c_y: +, -, 0][c], then [c_z: +, -, 0]
#pragma unroll
  for (int c = 0; c < 3; c++) sep_axis(col[3 * c], col[3 * c + 1], col[3 * c + 2], f[0][c], f[1][c], f[2][c]);
  bool ok = true;
#pragma unroll
  for (int y = 0; y < 3; y++) {
    sep_axis(f[y][0], f[y][1], f[y][2], f[y][0], f[y][1], f[y][2]);
#pragma unroll
    for (int z = 0; z < 3; z++) {
      ok = ok && f[y][z] >= 0.0f;  // false for NaN, which the clamp turns into 0
      f[y][z] = fmaxf(0.0f, f[y][z]);
    }
  }
  if (ok) return;
#pragma unroll
  for (int y = 0; y < 3; y++) sep_inverse(f[y][0], f[y][1], f[y][2], f[y][0], f[y][1], f[y][2]);
#pragma unroll
  for (int c = 0; c < 3; c++) sep_inverse(f[0][c], f[1][c], f[2][c], col[3 * c], col[3 * c + 1], col[3 * c + 2]);
}

// value of the lane before / after this one in the wave; `edge` where there is none
__device__ __forceinline__ float lane_before(float edge, float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(edge), __float_as_int(v), 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ float lane_after(float edge, float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(edge), __float_as_int(v), 0x130, 0xf, 0xf, false));
}

// Relaxation of the ten moments U (216 times the raw sums) and normalisation:
// the tail of collide3_fast divided through by rho (Collision,
// LbmUtilsFunc.cu:337-414, F = 0).
struct SepU {
  float r, x, y, z, xx, yy, zz, xy, yz, xz;
};
__device__ __forceinline__ void sep_collide(const SepU& U, float omega, float* out) {
  // v_rcp_f32 (1 ulp) and one Newton step, and 1/216 in two parts: an error
  // of either would be the same in every cell and step and add up over a run
  // (1.5e-8 of the mass and up to 6e-8 of the momentum a step).
  const float inv1 = __builtin_amdgcn_rcpf(U.r);
  const float inv = fmaf(inv1, fmaf(-U.r, inv1, 1.0f), inv1);
  const float ux = U.x * inv, uy = U.y * inv, uz = U.z * inv;
  const float third = 1.0f / 3.0f, omw = 1.0f - omega;
  const float qxx = U.xx * inv, qyy = U.yy * inv, qzz = U.zz * inv;
  const float tq = (qxx + qyy + qzz) * third;
  const float xx = ux * ux, yy = uy * uy, zz = uz * uz;
  const float e = (xx + yy + zz) * third;
  const float wux = omega * ux, wuy = omega * uy, w = omw * inv;
  constexpr float c216 = 1.0f / 216.0f, c216_lo = (float)(1.0 / 216.0 - (double)c216);
  out[0] = fmaf(U.r, c216, U.r * c216_lo);
  out[1] = ux;
  out[2] = uy;
  out[3] = uz;
  out[4] = fmaf(omw, qxx - tq, fmaf(omega, xx - e, e));
  out[5] = fmaf(omw, qyy - tq, fmaf(omega, yy - e, e));
  out[6] = fmaf(omw, qzz - tq, fmaf(omega, zz - e, e));
  out[7] = fmaf(w, U.xy, wux * uy);
  out[8] = fmaf(w, U.yz, wuy * uz);
  out[9] = fmaf(w, U.xz, wux * uz);
}

// Buffer accesses to a moment buffer: `r` describes it from the start of a
// z-plane of cells on, a moment plane adds a scalar offset, the lane a 32-bit
// byte offset; an offset of kNoCell is out of range, so that the lane's
// access is dropped.  Every lane then takes part in every access, with no
// branch around it: the wait for a plane's moments counts the younger loads
// and stores exactly (behind a branch it had to wait for all of them).
constexpr unsigned kNoCell = 0xFFFFFFFFu;
using BufRsrc = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ BufRsrc buf_rsrc(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)0xFFFFFFFF, 0x00027000);
}

__device__ __forceinline__ float sep_load(BufRsrc r, unsigned off, unsigned pb, int q) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (int)off, (int)(q * pb), 0));
}
__device__ __forceinline__ void sep_store(BufRsrc r, unsigned off, unsigned pb, int q, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, (int)off, (int)(q * pb), 0);
}

// Tile: 64 x 8 cells marching along z, one wave per row of 64 cells, and two
// waves for the rows below and above, which also take the columns left and
// right of the tile (a plane ahead).  The x neighbours are the wave's own
// lanes (DPP), the y neighbours pass F+- of nine (a', c) columns through a
// double-buffered LDS plane, the z neighbours are the previous and next
// plane's values in registers: one barrier a plane, 76 KB of LDS and 92
// VGPRs, so that two blocks share a CU.
// Bound by VALU issue (48 us of a 256x128x128 FP32 step without its loads and
// stores, at two blocks a CU) beside HBM (a copy with the same access pattern
// takes 70-75 us): 82-88 us against 102 us of the staged columns, 33 against
// 46 us on 128^3.  Measured and not kept:
// two planes of moments in flight (110-127 VGPRs, one block a CU less: 88 us),
// rows of 4 or 6 (91-97 us), non-temporal loads (halo rows miss L2: 97-106 us),
// stores a plane later (no change once their count is exact), the side columns
// of three planes at a time by one wave (97 us: the others wait for it).
constexpr int kSepThreads = 64 * (kSepTY + 2);
constexpr int kSepSide = 12;  // nine columns padded for 16-byte reads

// The domain's separable form: its z chunks, or 0 if it steps with the tiles.
// A body or a wall keeps the tiles: their boundary cells and bounce-back work
// on populations, and results with a body do not depend on which cells have
// links.  16-bit storage keeps them too: there another rounding in FP32 turns
// stored values by whole 16-bit roundings, which after 500 steps has moved a
// run by more than FP32 results may move (2e-5 of it at 256x192x160 in FP16;
// 110 against 147 us a step).
inline int sep3d_plan(const Domain& d) {
  if (d.dim != 3 || d.storage != FF_STORAGE_F32 || !(d.options & FF_OPT_FAST_MATH) || (d.has_boundary && d.ne > 0) ||
      d.walls3)
    return 0;
  return d.sep_chunks;
}

// The update of cell (x, y, z) from single populations, in the reference's
// order, if it pulls from a cell that is not tame; its own thread has stored
// the columns' result before.
template <bool PERIODIC>
__device__ __forceinline__ void sep_redo(const float* __restrict__ in, float* __restrict__ out, int nx, int ny, int nz,
                                         size_t plane, float omega, int x, int y, int z) {
  const auto source = [](int g, int n) { return PERIODIC ? (g < 0 ? g + n : (g >= n ? g - n : g)) : min(n - 1, max(0, g)); };
  float p[27];
  bool tame = true;
#pragma unroll
  for (int i = 0; i < 27; i++) {
    const int sx = source(x - D3::cx(i), nx), sy = source(y - D3::cy(i), ny), sz = source(z - D3::cz(i), nz);
    const float* src = in + ((size_t)sz * ny + sy) * nx + sx;
    float m[10];
#pragma unroll
    for (int q = 0; q < 10; q++) m[q] = src[q * plane];
    tame = tame && sep_bound(m).tame;
    p[i] = clamp0(recon3_pop(m, i));
  }
  if (tame) return;
  float o[10];
  collide3(p, omega, o);
  float* dst = out + ((size_t)z * ny + y) * nx + x;
#pragma unroll
  for (int q = 0; q < 10; q++) dst[q * plane] = o[q];
}

template <bool PERIODIC>
__device__ __forceinline__ void sep3d_column(const float* __restrict__ in, float* __restrict__ out,
                                             const uint8_t* __restrict__ flags, int nx, int ny, int nz, size_t plane,
                                             float omega, int bx, int by, int z0, int zend) {
  constexpr int TY = kSepTY;
  // F+ of the row below and F- of the row above each row: [buffer][a'][row][lane], c = 0, 1 and c = 2
  __shared__ float2 s_p[2][3][TY][64], s_m[2][3][TY][64];
  __shared__ float s_p2[2][3][TY][64], s_m2[2][3][TY][64];
  __shared__ __align__(16) float s_side[2][2][TY + 2][kSepSide];  // [buffer][left, right][row + 1][column]
  __shared__ int s_wild[2];  // a cell that is not tame was met; each cleared by one of the two last waves
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = (int)(threadIdx.x & 63u);
  const int x0 = bx * kSepTX, y0 = by * TY;
  const size_t nxy = (size_t)nx * ny;
  const unsigned pb = (unsigned)(plane * sizeof(float));  // bytes of a moment plane
  auto src_x = [&](int gx) { return PERIODIC ? ((gx % nx) + nx) % nx : min(nx - 1, max(0, gx)); };
  auto src_y = [&](int gy) { return PERIODIC ? ((gy % ny) + ny) % ny : min(ny - 1, max(0, gy)); };
  // Planes run from z0 - 1 to zend (one wrap at most); `i` counts them from 0,
  // past the last one it is taken again.
  const int np = zend - z0 + 2;
  auto plane_at = [&](int i) {
    const int gz = z0 - 1 + min(i, np - 1);
    return (unsigned)(PERIODIC ? (gz < 0 ? gz + nz : (gz >= nz ? gz - nz : gz)) : min(nz - 1, max(0, gz))) * nxy;
  };
  auto load = [&](int i, unsigned off, float* m) {
    const BufRsrc r = buf_rsrc(in + plane_at(i));
#pragma unroll
    for (int q = 0; q < 10; q++) m[q] = sep_load(r, off, pb, q);
  };
  // The x stage of a row from its cells' moments and the side columns of its
  // plane, and the y faces of the row: F+ to the row above, F- to the row
  // below (rows of the tile); hc: F0 along y.  The columns are taken by c,
  // each group finished before the next, which keeps the registers few.
  auto row_stage = [&](const float* m, int buf, int row, float (*hc)[3], auto&& refill) {
    const bool up = row + 1 < TY, down = row >= 1;  // wave-uniform
    float el[kSepSide], er[kSepSide];
#pragma unroll
    for (int k = 0; k < kSepSide; k += 4) {
      *reinterpret_cast<float4*>(el + k) = *reinterpret_cast<const float4*>(&s_side[buf][0][row + 1][k]);
      *reinterpret_cast<float4*>(er + k) = *reinterpret_cast<const float4*>(&s_side[buf][1][row + 1][k]);
    }
    // the ninth column (2, 2) is zero unless a clamp acted on a cell or on a side cell
    const SepBound bound = sep_bound(m);
    const bool plain = bound.positive && el[8] == 0.0f && er[8] == 0.0f;
    const bool nine = !__all(plain), wild = !__all(bound.tame);
    const SepCoef A = sep_coef(m);
    SepX X;
    sep_columns(A, X);
    refill();  // the moments are used: their registers take the next plane's
    if (nine) {
      if (wild) s_wild[0] = 1;
      sep_clamp(X.p);
      sep_clamp(X.m);
      sep_clamp(X.c);
    }
    float hp[2][3], hm[2][3];  // [c & 1][a']
#pragma unroll
    for (int c = 0; c < 3; c++) {
      float Sx[3][3];  // [b][a']
#pragma unroll
      for (int b = 0; b < 3; b++) {
        const int k = 3 * c + b;
        if (k == 8 && !nine) {
          Sx[b][0] = Sx[b][1] = Sx[b][2] = 0.0f;
        } else {
          const float p = lane_before(el[k], X.p[k]), n = lane_after(er[k], X.m[k]);
          Sx[b][2] = p + n;
          Sx[b][1] = p - n;
          Sx[b][0] = fmaf(4.0f, X.c[k], Sx[b][2]);
        }
      }
#pragma unroll
      for (int a = 0; a < 3; a++) sep_axis(Sx[0][a], Sx[1][a], Sx[2][a], hp[c & 1][a], hm[c & 1][a], hc[c][a]);
      if (c == 1) {
#pragma unroll
        for (int a = 0; a < 3; a++) {
          if (up) s_p[buf][a][row + 1][lane] = make_float2(hp[0][a], hp[1][a]);
          if (down) s_m[buf][a][row - 1][lane] = make_float2(hm[0][a], hm[1][a]);
        }
      } else if (c == 2) {
#pragma unroll
        for (int a = 0; a < 3; a++) {
          if (up) s_p2[buf][a][row + 1][lane] = hp[0][a];
          if (down) s_m2[buf][a][row - 1][lane] = hm[0][a];
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (wave < TY) {
    const int x = x0 + lane, y = y0 + wave;
    const bool inside = x < nx && y < ny;
    const unsigned src = (unsigned)(src_y(y) * nx + src_x(x));
    const unsigned cell = inside ? (unsigned)(y * nx + x) : 0u;  // in its plane
    float m[10];
    uint8_t fl = 0, fout = 0;
    load(0, src * sizeof(float), m);
    // z stage state of the columns (a', b') = 00, 10, 01, 20, 11, 02:
    // F+ of the plane below the current one, and 4 F0 + F+ of the two planes
    // that the pending output already has
    float kp1[6], zc[6], kp2[3];
#pragma unroll
    for (int k = 0; k < 6; k++) kp1[k] = zc[k] = 0.0f;
    kp2[0] = kp2[1] = kp2[2] = 0.0f;
    // The loop's results go out at the end of a pass; as many (dropped) stores
    // here let the wait for the moments at the top of every pass count them
    // out, the first pass included, instead of waiting for their write-back.
    auto put_results = [&](float* to_plane, unsigned to, const float* o) {
      const BufRsrc r = buf_rsrc(to_plane);
#pragma unroll
      for (int q = 0; q < 10; q++) sep_store(r, to, pb, q, o[q]);
    };
    {
      const float none[10] = {};
      put_results(out, kNoCell, none);
    }
    float* out_plane = out + (size_t)z0 * nxy;
    __syncthreads();  // the side columns of the first plane
    for (int i = 0; i < np; i++) {
      const int K = i & 1;
      float hc[3][3];  // [c][a']
      const uint8_t fz = fl;
      row_stage(m, K, wave, hc, [&] {
        load(i + 1, src * sizeof(float), m);
        fl = __builtin_amdgcn_raw_buffer_load_b8(buf_rsrc(flags + plane_at(i + 1)), (int)cell, 0, 0);
      });
      __syncthreads();
      // z stage of column k = (a', b') from its y moments t (c = 0, 1, 2):
      // returns U_a'b'0 of the output plane, with F+ below and F- above it for
      // the other c', and advances the state
      auto z_stage = [&](int k, const float* t, float& below, float& above) {
        float p, n, c;
        sep_axis(t[0], t[1], t[2], p, n, c);
        const float u = zc[k] + n;
        above = n;
        if (k < 3) {
          below = kp2[k];
          kp2[k] = kp1[k];
        }
        zc[k] = fmaf(4.0f, c, kp1[k]);
        kp1[k] = p;
        return u;
      };
      SepU U;  // of output plane z0 + i - 2 (from the third plane on)
      float b0, b1, b2, n0, n1, n2, unused;
      float2 p01[3], m01[3];
      float p2[3], m2[3];
#pragma unroll
      for (int a = 0; a < 3; a++) {  // F+ of the row below, F- of the row above
        p01[a] = s_p[K][a][wave][lane];
        m01[a] = s_m[K][a][wave][lane];
        p2[a] = s_p2[K][a][wave][lane];
        m2[a] = s_m2[K][a][wave][lane];
      }
#pragma unroll
      for (int a = 0; a < 3; a++) {
        const float hp[3] = {p01[a].x, p01[a].y, p2[a]}, hm[3] = {m01[a].x, m01[a].y, m2[a]};
        float t0[3], t1[3], t2[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
          t2[c] = hp[c] + hm[c];
          t1[c] = hp[c] - hm[c];
          t0[c] = fmaf(4.0f, hc[c][a], t2[c]);
        }
        if (a == 0) {
          U.r = z_stage(0, t0, b0, n0);
          U.y = z_stage(2, t1, b2, n2);
          U.yy = z_stage(5, t2, unused, unused);
        } else if (a == 1) {
          U.x = z_stage(1, t0, b1, n1);
          U.xy = z_stage(4, t1, unused, unused);
        } else {
          U.xx = z_stage(3, t0, unused, unused);
        }
      }
      U.z = b0 - n0;
      U.zz = b0 + n0;
      U.xz = b1 - n1;
      U.yz = b2 - n2;
      float o[10];
      sep_collide(U, omega, o);
      const unsigned to = (i >= 2 && inside && is_updated(fout)) ? (unsigned)(cell * sizeof(float)) : kNoCell;
      put_results(out_plane, to, o);
      if (i >= 2) out_plane += nxy;
      fout = fz;  // the flag of this step's plane, the next output
    }
    if ((s_wild[0] || s_wild[1]) && inside) {  // set before the last barrier
      for (int z = z0; z < zend; z++)
        if (is_updated(flags[(size_t)z * nxy + cell])) sep_redo<PERIODIC>(in, out, nx, ny, nz, plane, omega, x, y, z);
    }
  } else {
    const bool upper = wave == TY + 1;  // row TY and the right column, or row -1 and the left column
    const int row = upper ? TY : -1;
    const unsigned off = (unsigned)(src_y(y0 + row) * nx + src_x(x0 + lane)) * sizeof(float);
    const int srow = min(lane, TY + 1);  // side cell of this lane: row srow - 1
    const unsigned soff = (unsigned)(src_y(y0 + srow - 1) * nx + src_x(upper ? x0 + 64 : x0 - 1)) * sizeof(float);
    const float sg = upper ? -1.0f : 1.0f;  // F- of the right column, F+ of the left
    auto side = [&](const float* m, int buf, auto&& refill) {
      const SepBound bound = sep_bound(m);
      const bool clamp = !__all(bound.positive), wild = !__all(bound.tame);
      const SepCoef A = sep_coef(m);
      float f[kSepCols];
      sep_face(A, sg, f);
      refill();
      if (clamp) {
        if (wild) s_wild[upper] = 1;
        sep_clamp(f);
      }
      if (lane < TY + 2) {
        float* d = s_side[buf][upper ? 1 : 0][lane];
#pragma unroll
        for (int k = 0; k < kSepCols; k++) d[k] = f[k];
      }
    };
    float m[10], ms[10];
    s_wild[upper] = 0;
    load(0, soff, ms);
    load(0, off, m);
    side(ms, 0, [&] { load(1, soff, ms); });
    __syncthreads();
    for (int i = 0; i < np; i++) {
      const int K = i & 1;
      float hc[3][3];
      row_stage(m, K, row, hc, [&] { load(i + 1, off, m); });
      __builtin_amdgcn_sched_barrier(0);
      side(ms, K ^ 1, [&] { load(i + 2, soff, ms); });  // the side column of the next plane
      __syncthreads();
    }
  }
}

// Tile t of a domain's tiles_x x tiles_y x chunks grid.
template <bool PERIODIC>
__device__ __forceinline__ void sep3d_tile(const float* in, float* out, const uint8_t* flags, int nx, int ny, int nz,
                                           size_t plane, float omega, int tiles_x, int tiles_y, int chunks, int t) {
  const int bx = t % tiles_x, by = (t / tiles_x) % tiles_y, bz = t / (tiles_x * tiles_y);
  const int z0 = (int)((long long)bz * nz / chunks), zend = (int)((long long)(bz + 1) * nz / chunks);
  sep3d_column<PERIODIC>(in, out, flags, nx, ny, nz, plane, omega, bx, by, z0, zend);
}

}  // namespace ff
