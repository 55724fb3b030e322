// links_body.h -- device bodies of the boundary-cell, element-sum and finish
// phases, shared by the per-domain kernels (links.hip) and the batched
// kernels (batch.hip).  Each body takes its block index within the domain's
// part of the grid explicitly.
#pragma once

#include "ff_internal.h"
#include "geometry.h"
#include "hermite.h"

namespace ff {

// Virtual lanes of the per-body wrench sum (finish_last_body).
constexpr int kSumLanes = 256;


// ---------------------------------------------------------------- boundary cells
// First barycentric of a (slot, direction) whose link was not applied this
// step.  Applied 3D links can carry a slightly negative barycentric (the
// triangle test accepts u + v <= 1 + 1e-6), so the marker is far outside.
constexpr float kLinkUnused = -1.0e30f;

// Full update of every cell that owns a keyed link, one lane per lattice
// direction: the per-direction logic of mrDeformableSolver2DKernel_Shrd
// (FsiCoupling2D.cu:154-224) / mrDeformableSolver3DKernel_ShrdM
// (FsiCoupling3D.cu:194-285), moving-wall value from the single-population
// reconstruction, momentum-exchange force (FsiCoupling2D.cu:193-214,
// FsiCoupling3D.cu:243-271).  Overwrites the bulk kernel's value for the cell.
// Population i of a cell from its moments m: the reference's rounding
// (recon2_pop / recon3_pop, with the FP16 tile staging in 2D when STAGE),
// or under FAST the reference's all-FP32 single-population form in 2D.
template <int DIM, bool STAGE, bool FAST>
__device__ __forceinline__ float cell_pop(const float* m, int i) {
  if constexpr (DIM == 2) {
    if constexpr (FAST) {
      return recon2_at(m[0], m[1], m[2], m[3], m[5], m[4], i);
    } else {
      const float f = recon2_pop(m[0], m[1], m[2], m[3], m[5], m[4], i);
      if constexpr (STAGE) return __half2float(to_half_rn(f));
      return f;
    }
  } else {
    return recon3_pop(m, i);
  }
}

template <int DIM, int NT>
struct CellsLds {
  static constexpr int CPB = NT / (DIM == 2 ? 16 : 32);
  float sp[CPB][DIM == 2 ? 9 : 27];
  int s_slot[NT], s_cell[NT], s_wn[NT / 64], s_upd[CPB];
};

// The result is written to the cell's side-buffer row (la.sb), not to the
// output moments: the stream-collide tiles of the same launch also write the
// cell, and the element-sum launch copies the side buffer over them.
// Each block scans la.bc_span (<= NT) link-table slots at a time (grid
// stride nblk * bc_span), compacts the occupied ones in LDS and updates those
// cells CPB at a time.
template <int DIM, typename S, bool STAGE, bool PERIODIC, int NT, bool FAST = false>
__device__ __forceinline__ void bcells_body(const S* __restrict__ in, const LinkArgs& la, int blk, int nblk,
                                            CellsLds<DIM, NT>& lds) {
  constexpr int Q = DIM == 2 ? 9 : 27;
  constexpr int K = Q - 1;
  constexpr int NM = DIM == 2 ? 6 : 10;
  constexpr int LPC = DIM == 2 ? 16 : 32;  // lanes per cell
  constexpr int CPB = NT / LPC;            // cells per block
  constexpr int NW = NT / 64;
  auto& sp = lds.sp;
  auto& s_slot = lds.s_slot;
  auto& s_cell = lds.s_cell;
  auto& s_wn = lds.s_wn;
  auto& s_upd = lds.s_upd;
  const unsigned gen = step_gen(la);
  const unsigned tag = step_tag(la);
  const float* v = la.v[gen & 1];
  const float* u = la.u[gen & 1];
  const int lc = threadIdx.x / LPC, dir = threadIdx.x % LPC;
  const unsigned long long* cells = table_cells(la, tag);
  const unsigned long long* keys = table_keys<DIM>(la, tag);
  const int span = la.bc_span;
  for (int base = blk * span; base < la.cap; base += nblk * span) {
    // occupied slots of this chunk, in slot order
    const int s = base + (int)threadIdx.x;
    const bool scan = (int)threadIdx.x < span && s < la.cap;
    const unsigned long long ent = scan ? cells[s] : 0ull;
    const bool occ = scan && (unsigned)(ent >> 32) == tag;
    const unsigned long long m = __ballot(occ);
    const int w = (int)(threadIdx.x >> 6);
    if ((threadIdx.x & 63u) == 0) s_wn[w] = (int)__popcll(m);
    __syncthreads();
    int off = 0, count = 0;
#pragma unroll
    for (int i = 0; i < NW; i++) {
      off += i < w ? s_wn[i] : 0;
      count += s_wn[i];
    }
    if (occ) {
      const int r = off + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
      s_slot[r] = s;
      s_cell[r] = (int)(uint32_t)ent;
    }
    __syncthreads();
    for (int c0 = 0; c0 < count; c0 += CPB) {
      const int t = c0 + lc;
      int cell = 0;
      if (t < count && dir < Q) {
        const int slot = s_slot[t];
        cell = s_cell[t];
        const int x = cell % la.nx, y = (cell / la.nx) % la.ny, z = DIM == 3 ? cell / (la.nx * la.ny) : 0;
        const int dx = DIM == 2 ? D2::cx(dir) : D3::cx(dir);
        const int dy = DIM == 2 ? D2::cy(dir) : D3::cy(dir);
        const int dz = DIM == 2 ? 0 : D3::cz(dir);
        const int inv = DIM == 2 ? D2::inv(dir) : D3::inv(dir);
        const int x1 = x - dx, y1 = y - dy, z1 = z - dz;
        const bool notCross = x1 >= 0 && x1 < la.nx && y1 >= 0 && y1 < la.ny && z1 >= 0 && z1 < la.nz;
        const int xw = (x1 + la.nx) % la.nx, yw = (y1 + la.ny) % la.ny, zw = (z1 + la.nz) % la.nz;
        int sx, sy, sz;  // pull source: clamped halo (reference) or periodic
        if (PERIODIC) {
          sx = xw; sy = yw; sz = zw;
        } else {
          sx = min(la.nx - 1, max(0, x1));
          sy = min(la.ny - 1, max(0, y1));
          sz = min(la.nz - 1, max(0, z1));
        }
        const size_t sc = ((size_t)sz * la.ny + sy) * la.nx + sx;
        const size_t li = (size_t)slot * K + (dir - 1);
        // every load that depends only on the cell index is issued up front
        const uint8_t fup = la.flags[((size_t)zw * la.ny + yw) * la.nx + xw];
        const uint32_t key = dir > 0 ? lt_key(keys, li, tag) : 0xFFFFFFFFu;
        float mc[NM], mn[NM];
#pragma unroll
        for (int q = 0; q < NM; q++) {
          mc[q] = Store<S>::template load<DIM>(in + q * la.plane + cell, q, la.plane);
          mn[q] = Store<S>::template load<DIM>(in + q * la.plane + sc, q, la.plane);
        }
        // the lane needs two populations: the pulled one and the cell's own opposite one
        const float fn_dir = cell_pop<DIM, STAGE, FAST>(mn, dir);
        const float fc_inv = cell_pop<DIM, STAGE, FAST>(mc, inv);
        // direction 0 pulls from the cell itself: its flag is the cell's own,
        // kept for the collision after the barrier (a load there would come
        // after this block's link stores and wait for their write-back)
        if (dir == 0) s_upd[lc] = is_updated(fup) ? 1 : 0;
        float pop = 0.0f;
        bool done = false;
        bool linked = false;
        if (DIM == 3 && is_wall3(fup)) {  // 3D keeps flag bounce-back (FsiCoupling3D.cu:209-222)
          pop = fmaxf(0.0f, fc_inv);
          done = true;
        }
        if (!done && dir > 0 && notCross && (DIM == 3 || !is_wall2(fup)) && key != 0xFFFFFFFFu) {
          const int elem = (int)(key & 0xFFFFu);
          Hit h;
          bool hit;
          if constexpr (DIM == 2) {
            hit = hit_elem2(v, la.e, elem, (float)x * la.cl, (float)y * la.cl, (float)xw * la.cl, (float)yw * la.cl, h);
          } else {
            const float p1[3] = {(float)x * la.cl, (float)y * la.cl, (float)z * la.cl};
            const float p2[3] = {(float)xw * la.cl, (float)yw * la.cl, (float)zw * la.cl};
            hit = hit_elem3(v, la.e, elem, p1, p2, h);
          }
          if (hit) {
            done = true;
            const float fin = fmaxf(0.0f, fc_inv);
            float uw[3] = {0.f, 0.f, 0.f};
            float fout;
            if constexpr (DIM == 2) {
              // getVelocityAt<2> (:173-180), then `ux *= ct / cl` (FsiCoupling2D.cu:200-201)
              const uint32_t v1 = la.e[2 * elem], v2 = la.e[2 * elem + 1];
              uw[0] = u[2 * v1] * h.b[0] + u[2 * v2] * h.b[1];
              uw[1] = u[2 * v1 + 1] * h.b[0] + u[2 * v2 + 1] * h.b[1];
              uw[0] = uw[0] * (la.ct / la.cl);
              uw[1] = uw[1] * (la.ct / la.cl);
              const float pixx = mc[3] + uw[0] * uw[0] - mc[1] * mc[1];
              const float piyy = mc[4] + uw[1] * uw[1] - mc[2] * mc[2];
              const float pixy = mc[5] + uw[1] * uw[0] - mc[1] * mc[2];
              fout = recon2_at(mc[0], uw[0], uw[1], pixx, pixy, piyy, dir);
            } else {
              // getVelocityAt<3> (:385-398), then `u * ct / cl` (FsiCoupling3D.cu:244)
              const uint32_t v1 = la.e[3 * elem], v2 = la.e[3 * elem + 1], v3 = la.e[3 * elem + 2];
#pragma unroll
              for (int c = 0; c < 3; c++)
                uw[c] = ((u[3 * v1 + c] * h.b[0] + u[3 * v2 + c] * h.b[1] + u[3 * v3 + c] * h.b[2]) * la.ct) / la.cl;
              float ms[10];
              ms[0] = mc[0];
              ms[1] = uw[0];
              ms[2] = uw[1];
              ms[3] = uw[2];
              ms[4] = mc[4] + uw[0] * uw[0] - mc[1] * mc[1];
              ms[5] = mc[5] + uw[1] * uw[1] - mc[2] * mc[2];
              ms[6] = mc[6] + uw[2] * uw[2] - mc[3] * mc[3];
              ms[7] = mc[7] + uw[0] * uw[1] - mc[1] * mc[2];
              ms[8] = mc[8] + uw[1] * uw[2] - mc[2] * mc[3];
              ms[9] = mc[9] + uw[0] * uw[2] - mc[1] * mc[3];
              fout = recon3_at(ms, dir);
            }
            pop = fout;
            linked = true;
            const float cc[3] = {(float)dx, (float)dy, (float)dz};
#pragma unroll
            for (int c = 0; c < DIM; c++) {
              la.lf[li * DIM + c] = (fin * (-cc[c] - uw[c]) - fout * (cc[c] - uw[c])) * la.cf;
              la.lb[li * DIM + c] = h.b[c];
              la.lh[li * DIM + c] = h.hit[c];
            }
          }
        }
        // after every load of the lane: a store before the hit test's loads
        // would make their wait include its write-back
        if (dir > 0 && !linked) la.lb[li * DIM] = kLinkUnused;
        if (!done) pop = fmaxf(0.0f, fn_dir);
        sp[lc][dir] = pop;
      }
      __syncthreads();
      if (t < count && dir == 0 && s_upd[lc]) {
        float p[Q];
#pragma unroll
        for (int i = 0; i < Q; i++) p[i] = sp[lc][i];
        float o[NM];
        if constexpr (DIM == 2 && FAST) collide2_fast(p, la.omega, o);
        else if constexpr (DIM == 2) collide2(p, la.omega, o);
        else if constexpr (FAST) collide3_fast(p, la.omega, o);
        else collide3(p, la.omega, o);
        float* row = la.sb + (size_t)s_slot[t] * NM;
#pragma unroll
        for (int q = 0; q < NM; q++) row[q] = o[q];
      }
      __syncthreads();
    }
  }
}

// ---------------------------------------------------------------- finalize
struct FinalArgs {
  const int* elem_body;
  const double* body_ref;
  int n_bodies;
  double* elem_acc;
  double* wrench;
  double* hist;
  double* power;       // per body, latest step
  double* power_hist;  // ring of hist_cap steps (with hist)
  int hist_cap;
  const int* bptr;
  const int* bidx;
  const int* vptr;
  const int* vinc;
  float* vforce;
  float* proxy_forces;
  int wave;
  const float* rest;
  const float* s;
  const int* vbody;
  const double* wpar;
  int wave_fast;  // FP32 kinematics (fast math)
  double dt;
  float* vn[2];
  float* un[2];
  void* buf;
  const OutletCell* outlets;
  int n_outlets;
  int outlet_blocks;
  int copy_blocks;  // copy-back blocks of the sums launch
  int kin_blocks;   // stream launch extras: kinematics blocks, then fin_blocks
  int fin_blocks;   // of a deferred finish (vertex blocks + 1) of step fin_gen
  unsigned fin_gen;
};

// Block size of the element-sum launch (elements_per_block).
constexpr int kSumBlock = 256;
static_assert(kSumBlock == kBlock3, "a block of the element sums and of the detection takes the same triangles");

// Host: the FinalArgs of a domain (outlets written into `out`, next-step
// kinematics into vn/un, per-vertex forces optionally added to proxy_forces).
FinalArgs make_final_args(Domain& d, void* out, float* vn0, float* vn1, float* un0, float* un1, float* proxy_forces);
// Host: grid sizes of the boundary-cell and copy-back parts of a step.
int boundary_cell_blocks(const Domain& d, int span);
int copyback_blocks(const Domain& d, int fb, int per_thread);

// Travelling wave along the body axis:
//   y = y_rest + A s sin(theta), v_y = -2 pi f A s cos(theta),
//   theta = 2 pi (s L/lambda - f t) + phi,  t = g dt at step g.
// par holds per body the four FP64 parameters (A, f, phi, L/lambda)
// followed by eight FP32 values derived from them on the host
// (wave_fp32_params); with fast32 the phase is reduced in cycles in FP32:
// f t mod 1 comes from g times (f dt) held as a float pair hi + lo, the
// product's rounding error recovered with an FMA, so the phase error stays
// about 1e-7 cycle for any g below 2^24.
template <int DIM>
__device__ __forceinline__ void wave_vertex(const float* rest, const float* s, const int* vbody, const double* par,
                                            int fast32, int k, unsigned g, double dt, float* v, float* vel) {
  // every input is read before the first store: a read issued after a store
  // (which may alias it, for the compiler) waits for that store's write-back
  const int b = vbody[k];
  float r[DIM];
#pragma unroll
  for (int c = 0; c < DIM; c++) r[c] = rest[k * DIM + c];
  const float sk32 = s[k];
  float y, vy;
  if (fast32) {
    const float* q = (const float*)(par + kWaveParStride * b + 4);
    const float A = q[0], kl = q[1], phic = q[2], hi = q[3], lo = q[4], vamp = q[5];
    const float gf = (float)g;
    const float pr = gf * hi;
    const float er = fmaf(gf, hi, -pr);
    const float tc = (pr - floorf(pr)) + fmaf(gf, lo, er);  // f t mod 1 (up to a whole cycle)
    float cyc = fmaf(sk32, kl, -tc) + phic;
    cyc -= rintf(cyc);
    float sn, cs;
    sincospif(2.0f * cyc, &sn, &cs);
    const float as = A * sk32;
    y = fmaf(as, sn, r[1]);
    vy = -vamp * sk32 * cs;
  } else {
    const double* p = par + kWaveParStride * b;
    const double A = p[0], f = p[1], phi = p[2], kl = p[3];
    const double sk = (double)sk32;
    const double t = (double)g * dt;
    const double two_pi = 6.283185307179586;
    const double th = two_pi * (sk * kl - f * t) + phi;
    double sn, cs;
    sincos(th, &sn, &cs);
    y = (float)((double)r[1] + A * sk * sn);
    vy = (float)(-two_pi * f * A * sk * cs);
  }
#pragma unroll
  for (int c = 0; c < DIM; c++) {
    v[k * DIM + c] = c == 1 ? y : r[c];
    vel[k * DIM + c] = c == 1 ? vy : 0.0f;
  }
}

// Next-step kinematics for one block of vertices (stream launch): the vertex
// buffers of the next step are not read during this step.
// FAST kernels take the FP32 kinematics (FF_OPT_FAST_MATH always sets wave_fast).
template <int DIM, int FB, bool FAST = false>
__device__ __forceinline__ void wave_block_body(const LinkArgs& la, const FinalArgs& fa, int blk) {
  const int k = blk * FB + threadIdx.x;
  if (k < la.nv) {
    const unsigned g = step_gen(la);
    wave_vertex<DIM>(fa.rest, fa.s, fa.vbody, fa.wpar, FAST ? 1 : fa.wave_fast, k, g, fa.dt, fa.vn[(g + 1) & 1],
                     fa.un[(g + 1) & 1]);
  }
}

// Detection of the next step's links (tag + 1, the next step's vertex
// positions) into the other link table.
template <int DIM, bool BATCHED>
__device__ __forceinline__ void detect_next_body(const LinkArgs& la, int blk, DetLds<DIM>& lds, int epb) {
  const unsigned gen = step_gen(la);
  detect_block<DIM, BATCHED>(la, (long long)blk, step_tag(la) + 1u, la.v[(gen + 1u) & 1u], lds, epb);
}

// ---------------------------------------------------------------- element sums
// v of lane + N of the same DPP row (16 lanes), 0 beyond its end.
template <int N>
__device__ __forceinline__ double row_down(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, 0x100 | N, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), 0x100 | N, 0xf, 0xf, true);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
// Lane 0 of every row ends with the row's sums (a fixed tree).
template <int M>
__device__ __forceinline__ void row_sums(double* a) {
#pragma unroll
  for (int k = 0; k < M; k++) a[k] += row_down<8>(a[k]);
#pragma unroll
  for (int k = 0; k < M; k++) a[k] += row_down<4>(a[k]);
#pragma unroll
  for (int k = 0; k < M; k++) a[k] += row_down<2>(a[k]);
#pragma unroll
  for (int k = 0; k < M; k++) a[k] += row_down<1>(a[k]);
}

// Bit l set: direction l + 1 of the slot holds a key of this generation that
// names element `etag` (the winner of the link).
template <int DIM>
__device__ __forceinline__ unsigned links_of_element(const unsigned long long* keys, int slot, unsigned tag,
                                                     unsigned etag) {
  constexpr int K = DIM == 2 ? 8 : 26;
  // a row of keys is K * 8 bytes, a multiple of 16, in a 256-byte aligned table
  const ulonglong2* row = reinterpret_cast<const ulonglong2*>(keys + (size_t)slot * K);
  unsigned m = 0;
#pragma unroll
  for (int l = 0; l < K; l += 2) {
    const ulonglong2 w = row[l / 2];
    if ((unsigned)(w.x >> 32) == tag && (~(unsigned)w.x & 0xFFFFu) == etag) m |= 1u << l;
    if ((unsigned)(w.y >> 32) == tag && (~(unsigned)w.y & 0xFFFFu) == etag) m |= 2u << l;
  }
  return m;
}

// Row sums of a block's kBlock3 / kRow rows.
using SumPart = double[kBlock3 / kRow][kRow];

// Sum of one segment's links by LANES = kRow lanes, or the block where a
// window is large (elements_per_block): each lane takes up to two
// window cells per pass (its own table probes and key rows in flight
// together), then the links of those cells that name this element, in
// direction order; a fixed tree folds the lanes.  The pass is a chain of
// dependent loads (vertices -> table -> keys -> links) at every step's end, and
// with many domains it is bound by instruction issue: one (cell, direction)
// task per lane loaded every link's force and geometry before knowing whose
// it was, and folded one element per wave.
template <int LANES>
__device__ __forceinline__ void elem_sum2(const LinkArgs& la, const FinalArgs& fa, int elem, int lane, SumPart& part) {
  constexpr int K = 8, STRIDE = elem_stride_v<2>, U = 2;
  const unsigned gen = step_gen(la), tag = step_tag(la);
  const float* v = dev_global(la.v[gen & 1]);
  const float* u = dev_global(la.u[gen & 1]);
  const u32x2 ends = load2(dev_global(la.e) + 2 * (size_t)elem);
  const int body = fa.elem_body ? dev_global(fa.elem_body)[elem] : 0;
  const f32x2 pa = load2(v + 2 * (size_t)ends.x), pb = load2(v + 2 * (size_t)ends.y);
  const f32x2 ua = load2(u + 2 * (size_t)ends.x), ub = load2(u + 2 * (size_t)ends.y);
  const double rx = dev_global(fa.body_ref)[2 * body], ry = dev_global(fa.body_ref)[2 * body + 1];
  const int n[2] = {la.nx, la.ny};
  int lo[2], hi[2];
  seg_window(pa, pb, la.cl, n, lo, hi);
  const int wx = hi[0] - lo[0] + 1, wy = hi[1] - lo[1] + 1;
  const int ncell = (wx > 0 && wy > 0) ? wx * wy : 0;
  double acc[STRIDE];
#pragma unroll
  for (int a = 0; a < STRIDE; a++) acc[a] = 0.0;
  const unsigned etag = (unsigned)elem & 0xFFFFu;
  const uint8_t* flags = dev_global(la.flags);
  const unsigned long long* cells = table_cells(la, tag);
  const unsigned long long* keys = table_keys<2>(la, tag);
  const float* lf = dev_global(la.lf);
  const float* lb = dev_global(la.lb);
  const float* lh = dev_global(la.lh);
  for (int k0 = lane; k0 < ncell; k0 += LANES * U) {
    int cell[U];
    unsigned home[U];
    unsigned long long cur[U];
    bool upd[U];
#pragma unroll
    for (int w = 0; w < U; w++) {
      const int k = k0 + w * LANES;
      upd[w] = false;
      if (k < ncell) {
        const int j = k / wx;
        cell[w] = (lo[1] + j) * la.nx + lo[0] + (k - j * wx);
        home[w] = lt_home(la.cap, cell[w]);
        cur[w] = cells[home[w]];
        upd[w] = is_updated(flags[cell[w]]);
      }
    }
    int slot[U];
#pragma unroll
    for (int w = 0; w < U; w++) slot[w] = upd[w] ? lt_resolve(cells, la.cap, tag, cell[w], home[w], cur[w]) : -1;
    unsigned m = 0;
#pragma unroll
    for (int w = 0; w < U; w++)
      if (slot[w] >= 0) m |= links_of_element<2>(keys, slot[w], tag, etag) << (w * K);
    while (m) {  // two links at a time
      size_t li[2];
      f32x2 F[2], B[2], H[2];
      bool use[2];
#pragma unroll
      for (int w = 0; w < 2; w++) {
        use[w] = m != 0;
        if (use[w]) {
          const int b = __ffs((int)m) - 1;
          m &= m - 1;
          li[w] = 2 * ((size_t)(b < K ? slot[0] : slot[1]) * K + (b & (K - 1)));
          F[w] = load2(lf + li[w]);
          B[w] = load2(lb + li[w]);
          H[w] = load2(lh + li[w]);
        }
      }
#pragma unroll
      for (int w = 0; w < 2; w++) {
        if (!use[w] || B[w].x == kLinkUnused) continue;
        acc[0] += (double)(F[w].x * B[w].x);  // addForceAt products
        acc[1] += (double)(F[w].y * B[w].x);
        acc[2] += (double)(F[w].x * B[w].y);
        acc[3] += (double)(F[w].y * B[w].y);
        acc[4] += (double)F[w].x;
        acc[5] += (double)F[w].y;
        acc[6] += ((double)H[w].x - rx) * (double)F[w].y - ((double)H[w].y - ry) * (double)F[w].x;
      }
    }
  }
  row_sums<STRIDE - 1>(acc);
  if constexpr (LANES > kRow) {  // lane 0 of every row has its sums: fold the rows alike
    if (lane % kRow == 0) {
#pragma unroll
      for (int a = 0; a < STRIDE - 1; a++) part[lane / kRow][a] = acc[a];
    }
    __syncthreads();
    if (lane < kRow) {
#pragma unroll
      for (int a = 0; a < STRIDE - 1; a++) acc[a] = part[lane][a];
    }
    row_sums<STRIDE - 1>(acc);
  }
  if (lane == 0) {
    // the element's power: its vertex shares against the velocities the step used
    acc[STRIDE - 1] =
        -(acc[0] * (double)ua.x) - acc[1] * (double)ua.y - acc[2] * (double)ub.x - acc[3] * (double)ub.y;
    double2* row = reinterpret_cast<double2*>(dev_global(fa.elem_acc) + (size_t)elem * STRIDE);
#pragma unroll
    for (int a = 0; a < STRIDE; a += 2) row[a / 2] = make_double2(acc[a], acc[a + 1]);
  }
}

// Sum of one triangle's links by NT threads: a window of some 4^3 to 7^3
// cells, one cell per thread and pass, its 26 keys read as one row.  The cells
// belong to the kBlock3 threads of a block in turn, whose rows of 16 are folded
// by a fixed tree and their sums in row order; a wave (NT = 64) takes the
// block's four waves one after the other, so the sums are the same bits.
// One wave per triangle with (cell, direction) tasks walked the window of a
// triangle of a sphere of 320 in a serial chain of some 150 loads, which set
// the launch's time (76 us in a 160x96x96 domain).
template <int NT>
__device__ __forceinline__ void elem_sum3(const LinkArgs& la, const FinalArgs& fa, int elem, SumPart& part) {
  constexpr int K = 26, STRIDE = elem_stride_v<3>, M = STRIDE - 1, NROW = kBlock3 / kRow;
  static_assert(M <= kRow, "one lane of a row per sum");
  const int tid = (int)threadIdx.x & (NT - 1);
  const unsigned gen = step_gen(la), tag = step_tag(la);
  const float* v = dev_global(la.v[gen & 1]);
  const int n[3] = {la.nx, la.ny, la.nz};
  int lo[3], hi[3];
  elem_window<3>(v, dev_global(la.e), elem, la.cl, n, lo, hi);
  const int wx = hi[0] - lo[0] + 1, wy = hi[1] - lo[1] + 1, wz = hi[2] - lo[2] + 1;
  const int ncell = (wx > 0 && wy > 0 && wz > 0) ? wx * wy * wz : 0;
  const int body = fa.elem_body ? dev_global(fa.elem_body)[elem] : 0;
  double ref[3];
#pragma unroll
  for (int c = 0; c < 3; c++) ref[c] = dev_global(fa.body_ref)[body * 3 + c];
  const unsigned etag = (unsigned)elem & 0xFFFFu;
  const uint8_t* flags = dev_global(la.flags);
  const unsigned long long* cells = table_cells(la, tag);
  const unsigned long long* keys = table_keys<3>(la, tag);
  const float* lf = dev_global(la.lf);
  const float* lb = dev_global(la.lb);
  const float* lh = dev_global(la.lh);
  const int lane = tid % kRow, nq = min(kBlock3 / NT, max(1, (ncell + NT - 1) / NT));
  for (int q = 0; q < nq; q++) {
    double acc[M];
#pragma unroll
    for (int a = 0; a < M; a++) acc[a] = 0.0;
    for (int k = q * NT + tid; k < ncell; k += kBlock3) {
      const int i = lo[0] + k % wx, j = lo[1] + (k / wx) % wy, z = lo[2] + k / (wx * wy);
      const int cell = (z * la.ny + j) * la.nx + i;
      const unsigned home = lt_home(la.cap, cell);
      const unsigned long long cur = cells[home];
      if (!is_updated(flags[cell])) continue;
      const int slot = lt_resolve(cells, la.cap, tag, cell, home, cur);
      if (slot < 0) continue;
      for (unsigned m = links_of_element<3>(keys, slot, tag, etag); m; m &= m - 1) {
        const size_t li = ((size_t)slot * K + (__ffs((int)m) - 1)) * 3;
        float F[3], B[3], H[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
          F[c] = lf[li + c];
          B[c] = lb[li + c];
          H[c] = lh[li + c];
        }
        if (B[0] == kLinkUnused) continue;
#pragma unroll
        for (int jv = 0; jv < 3; jv++)
#pragma unroll
          for (int c = 0; c < 3; c++) acc[jv * 3 + c] += (double)(F[c] * B[jv]);  // addForceAt products
        double r[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
          acc[9 + c] += (double)F[c];
          r[c] = (double)H[c] - ref[c];
        }
        acc[12] += r[1] * (double)F[2] - r[2] * (double)F[1];
        acc[13] += r[2] * (double)F[0] - r[0] * (double)F[2];
        acc[14] += r[0] * (double)F[1] - r[1] * (double)F[0];
      }
    }
    row_sums<M>(acc);
    if (lane == 0) {
#pragma unroll
      for (int a = 0; a < M; a++) part[(q * NT + tid) / kRow][a] = acc[a];
    }
  }
  group_sync<NT>();
  if (tid < kRow) {
    double t = 0.0;
    if (lane < M) {
#pragma unroll
      for (int r = 0; r < NROW; r++)
        if (NT == kBlock3 || r < nq * (NT / kRow)) t += part[r][lane];  // the other rows have no cell: zero
    }
    // the element's power: its vertex shares against the velocities the step used
    double pw = 0.0;
    if (lane < 9) {
      const size_t vid = dev_global(la.e)[(size_t)elem * 3 + lane / 3];
      pw = -t * (double)dev_global(la.u[gen & 1])[vid * 3 + lane % 3];
    }
    row_sums<1>(&pw);
    double* out = dev_global(fa.elem_acc) + (size_t)elem * STRIDE;
    if (lane < M) out[lane] = t;
    if (lane == 0) out[STRIDE - 1] = pw;
  }
}

// LDS of a block of the element-sum launch.
template <int DIM>
union SumsLds {
  DetLds<DIM> det;
  SumPart part[DIM == 2 ? 1 : kBlock3 / 64];
};

// Second launch of a boundary step, kSumBlock threads per block.  The first
// `neb` blocks sum links per element (fixed order, FP64) into elem_acc.
// Then outlet blocks: outlet cells of the freshly written buffer
// (mrApplyOutlet2DKernel / mrApplyOutlet3DKernel; a neighbour that is a
// boundary cell is read from its side-buffer row, which the copy-back of this
// launch writes).  Then copy-back blocks: boundary-cell rows into the output.
// Any further blocks detect the next step's links.
// `epb` elements a block, a constant in a kernel for one domain, `neb` blocks.
template <int DIM, typename S, int FB, bool BATCHED>
__device__ __forceinline__ void elem_sums_body(const LinkArgs& la, const FinalArgs& fa, int blk, void* out,
                                               SumsLds<DIM>& lds, int epb, int neb) {
  static_assert(FB == kSumBlock, "element sums and detection are written for kSumBlock threads");
  constexpr int NM = DIM == 2 ? 6 : 10;
  if (blk >= neb + fa.outlet_blocks + fa.copy_blocks) {
    detect_next_body<DIM, BATCHED>(la, blk - neb - fa.outlet_blocks - fa.copy_blocks, lds.det, epb);
    return;
  }
  if (blk >= neb + fa.outlet_blocks) {
    const unsigned tag = step_tag(la);
    const int b = blk - neb - fa.outlet_blocks;
    const int nb = fa.copy_blocks;
    const unsigned long long* cells = table_cells(la, tag);
    S* o = (S*)out;
    for (int slot = b * FB + threadIdx.x; slot < la.cap; slot += nb * FB) {
      const unsigned long long ent = cells[slot];
      if ((unsigned)(ent >> 32) != tag) continue;
      const int cell = (int)(uint32_t)ent;
      if (!is_updated(la.flags[cell])) continue;
      // the whole row is loaded before the first store: a load issued after a
      // store (which may alias it, for the compiler) waits for that store's
      // write-back
      const float* row = la.sb + (size_t)slot * NM;
      float r[NM];
#pragma unroll
      for (int q = 0; q < NM; q++) r[q] = row[q];
#pragma unroll
      for (int q = 0; q < NM; q++) Store<S>::template store<DIM>(o + q * la.plane + cell, q, r[q], la.plane);
    }
    return;
  }
  if (blk >= neb) {
    const int t = (blk - neb) * FB + threadIdx.x;
    if (t >= fa.n_outlets) return;
    S* buf = (S*)out;
    const OutletCell c = fa.outlets[t];
    if (la.flags[c.nb] != kFluid) return;
    const unsigned tag = step_tag(la);
    const int nslot = la.ne > 0 ? lt_find(table_cells(la, tag), la.cap, tag, c.nb) : -1;
    const float up = nslot >= 0 ? la.sb[(size_t)nslot * NM + c.comp]
                                : Store<S>::template load<DIM>(buf + c.comp * la.plane + c.nb, c.comp, la.plane);
    if ((c.sign > 0 && up > 0.0f) || (c.sign < 0 && up < 0.0f))
      Store<S>::template store<DIM>(buf + c.comp * la.plane + c.cell, c.comp, up, la.plane);
    Store<S>::template store<DIM>(buf + c.pcomp * la.plane + c.cell, c.pcomp, up * up, la.plane);
    return;
  }
  if constexpr (DIM == 2) {
    const int elem = blk * (FB / kRow) + (int)threadIdx.x / kRow;
    if (epb == 1) elem_sum2<FB>(la, fa, blk, (int)threadIdx.x, lds.part[0]);
    else if (elem < la.ne) elem_sum2<kRow>(la, fa, elem, (int)threadIdx.x % kRow, lds.part[0]);
  } else if (epb == 1) {
    elem_sum3<kBlock3>(la, fa, blk, lds.part[0]);
  } else {
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int elem = blk * (FB / 64) + wave;
    if (elem < la.ne) elem_sum3<64>(la, fa, elem, lds.part[wave]);
  }
}

// Vertex blocks sum their incident element shares in CSR order (the
// per-vertex forces addForceAt accumulates); the last block folds element
// sums into body wrenches with a fixed tree (ring slot of step `gen`) and,
// for batched domains, advances gen and tag.
template <int DIM, int FB>
__device__ __forceinline__ void finish_vertex_body(const LinkArgs& la, const FinalArgs& fa, int blk) {
  constexpr int NT = DIM == 2 ? 1 : 3;
  constexpr int STRIDE = elem_stride_v<DIM>;
  const int vtx = blk * FB + threadIdx.x;
  if (vtx >= la.nv) return;
  // the forces being added to are read first, beside the element shares: an
  // interleaved read-add-write chain makes every read wait for the previous
  // write's write-back (the two arrays may alias, for the compiler)
  float fv[DIM], fp[DIM];
#pragma unroll
  for (int c = 0; c < DIM; c++) {
    fv[c] = fa.vforce[vtx * DIM + c];
    fp[c] = fa.proxy_forces ? fa.proxy_forces[vtx * DIM + c] : 0.0f;
  }
  double f[DIM];
#pragma unroll
  for (int c = 0; c < DIM; c++) f[c] = 0.0;
  for (int k = fa.vptr[vtx]; k < fa.vptr[vtx + 1]; k++) {
    const int code = fa.vinc[k];
    const int e = code >> 2, end = code & 3;
#pragma unroll
    for (int c = 0; c < DIM; c++) f[c] += fa.elem_acc[(size_t)e * STRIDE + end * DIM + c];
  }
#pragma unroll
  for (int c = 0; c < DIM; c++) fa.vforce[vtx * DIM + c] = fv[c] + (float)f[c];
  if (fa.proxy_forces) {
#pragma unroll
    for (int c = 0; c < DIM; c++) fa.proxy_forces[vtx * DIM + c] = fp[c] + (float)f[c];
  }
}

// LDS of finish_last_body: the wrench's channels and the power of each lane.
template <int DIM>
struct FinishLds {
  double s_red[DIM + (DIM == 2 ? 1 : 3) + 1][kSumLanes];
};

template <int DIM, int FB>
__device__ __forceinline__ void finish_last_body(const LinkArgs& la, const FinalArgs& fa, unsigned gen, bool advance,
                                                 FinishLds<DIM>& lds) {
  constexpr int NT = DIM == 2 ? 1 : 3;
  constexpr int STRIDE = elem_stride_v<DIM>;
  constexpr int NW = DIM + NT;
  // The sums run over kSumLanes virtual lanes (lane v: elements v, v + kSumLanes,
  // ... of the body, then a fixed tree), whatever the block size FB, so a
  // body's wrench is the same FP64 number from every launch shape.  Channels:
  // the wrench (NW), then the power.
  constexpr int V = kSumLanes, NC = NW + 1;
  auto& s_red = lds.s_red;
  for (int bd = 0; bd < fa.n_bodies; bd++) {
    for (int v = threadIdx.x; v < V; v += FB) {
      double a[NC];
#pragma unroll
      for (int c = 0; c < NC; c++) a[c] = 0.0;
      for (int k = fa.bptr[bd] + v; k < fa.bptr[bd + 1]; k += V) {
        const double* ea = fa.elem_acc + (size_t)fa.bidx[k] * STRIDE + DIM * DIM;
#pragma unroll
        for (int c = 0; c < NC; c++) a[c] += ea[c];
      }
#pragma unroll
      for (int c = 0; c < NC; c++) s_red[c][v] = a[c];
    }
    __syncthreads();
    for (int w = V / 2; w > 0; w >>= 1) {
      for (int v = threadIdx.x; v < w; v += FB)
#pragma unroll
        for (int c = 0; c < NC; c++) s_red[c][v] += s_red[c][v + w];
      __syncthreads();
    }
    if (threadIdx.x == 0) {
      fa.power[bd] = s_red[NW][0];
      if (fa.power_hist) fa.power_hist[(size_t)((gen - 1) % (unsigned)fa.hist_cap) * fa.n_bodies + bd] = s_red[NW][0];
    }
    if ((int)threadIdx.x < NW) {
      fa.wrench[bd * NW + threadIdx.x] = s_red[threadIdx.x][0];
      if (fa.hist)
        fa.hist[((size_t)((gen - 1) % (unsigned)fa.hist_cap) * fa.n_bodies + bd) * NW + threadIdx.x] =
            s_red[threadIdx.x][0];
    }
    __syncthreads();
  }
  if (advance && threadIdx.x == 0) {  // batched domains: the device keeps gen and tag
    la.st->gen = gen + 1;
    la.st->tag = la.st->tag + 1;
  }
}

// Extra blocks of the stream launch of a boundary step: next-step
// kinematics (kin_blocks), then, when the previous step's finish was
// deferred to this launch, its vertex blocks and wrench block (fin_blocks).
// The previous step's element sums are complete (earlier launch) and this
// step's are not started (later launch).
template <int DIM, int NT, bool FAST = false>
__device__ __forceinline__ void stream_extra_body(const LinkArgs& la, const FinalArgs& fa, int blk,
                                                  FinishLds<DIM>& lds) {
  if (blk < fa.kin_blocks) {
    wave_block_body<DIM, NT, FAST>(la, fa, blk);
    return;
  }
  blk -= fa.kin_blocks;
  if (blk < fa.fin_blocks - 1) finish_vertex_body<DIM, NT>(la, fa, blk);
  else finish_last_body<DIM, NT>(la, fa, fa.fin_gen, false, lds);
}

// LDS of a stream launch: its blocks are tiles, boundary-cell blocks or
// extras, and share it.  (Each with its own, a 3D launch had 17 KB more and
// held one box or two 16x12x8 columns a CU instead of two or four: 160x96x96
// around a sphere 125 us against 74 with boxes, 55 against 45 with columns.)
template <int DIM, int NT, class TILE>
union StepLds {
  TILE tile;
  CellsLds<DIM, NT> cells;
  FinishLds<DIM> finish;
};

}  // namespace ff
