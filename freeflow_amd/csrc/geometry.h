// geometry.h -- link/element predicates and the generation-tagged link table.
//
// Predicates restate SolidGeometryProxy_Device.cuh (line_intersect :89-124,
// intersectAtIndex<2> :211-227, line_triangle_intersect :306-341,
// getBoundingBox :198-209, :424-440, depthIndexCompact :79-85).  They take the
// same discrete decisions as the reference only without FMA contraction and
// with IEEE division/square root, which is how every unit including this file
// is compiled.
//
// Link table: open addressing keyed by cell.  Entries carry the step's
// generation in their upper 32 bits, so entries of earlier steps read as
// empty and the table never needs clearing:
//   cell word : (gen << 32) | cell
//   key word  : (gen << 32) | ~depthIndexCompact   (atomicMax keeps the
//               current generation and, within it, the smallest key)
#pragma once

#include <cfloat>
#include <stdint.h>

#include "hermite.h"

namespace ff {

__device__ __forceinline__ unsigned mix32(unsigned h) {
  h ^= h >> 16;
  h *= 0x85ebca6bu;
  h ^= h >> 13;
  h *= 0xc2b2ae35u;
  h ^= h >> 16;
  return h;
}

// Generation and tag of the step being run (see LinkArgs).
__device__ __forceinline__ unsigned step_gen(const LinkArgs& la) { return la.dev_state ? la.st->gen : la.gen; }
__device__ __forceinline__ unsigned step_tag(const LinkArgs& la) { return la.dev_state ? la.st->tag : la.tag; }

// A pointer read from a record in device memory (the batch's domain table) is
// not known to be global to the compiler, which then addresses it generically
// (flat instructions, which also count against the LDS wait counter).  Passed
// through an integer into the global address space, every access derived from
// it is a global one; a pointer that is a kernel argument is unchanged.
template <typename T>
__device__ __forceinline__ T* dev_global(T* p) {
  return (T*)(__attribute__((address_space(1))) T*)reinterpret_cast<unsigned long long>(p);
}

// Two adjacent 4-byte values in one load.  A caller's own boundary arrays
// (ff_step_proxy) are only 4-byte aligned, and these types say so.
typedef float f32x2 __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2), aligned(4)));
__device__ __forceinline__ f32x2 load2(const float* p) { return *reinterpret_cast<const f32x2*>(p); }
__device__ __forceinline__ u32x2 load2(const uint32_t* p) { return *reinterpret_cast<const u32x2*>(p); }

// Two link tables alternate by tag parity: the next step's links are detected
// into one while the current step's are read from the other.
__device__ __forceinline__ unsigned long long* table_cells(const LinkArgs& la, unsigned tag) {
  return dev_global(la.cells) + (size_t)(tag & 1u) * la.cap;
}
template <int DIM>
__device__ __forceinline__ unsigned long long* table_keys(const LinkArgs& la, unsigned tag) {
  return dev_global(la.keys) + (size_t)(tag & 1u) * la.cap * (DIM == 2 ? 8 : 26);
}

// Slot of `cell` under generation `gen`, entering it if absent.  The cells of
// a generation are found again by scanning the slots for its tag (no list, so
// no counter that every detecting lane would serialise on).
__device__ __forceinline__ int lt_claim(unsigned long long* cells, int cap, unsigned gen, int cell, int* overflow) {
  const unsigned long long want = ((unsigned long long)gen << 32) | (unsigned)cell;
  unsigned h = mix32((unsigned)cell) & (unsigned)(cap - 1);
  for (int probe = 0; probe < cap; probe++) {
    unsigned long long cur = cells[h];
    while ((unsigned)(cur >> 32) != gen) {  // stale or never used: try to claim
      const unsigned long long prev = atomicCAS(&cells[h], cur, want);
      if (prev == cur) return (int)h;
      cur = prev;
    }
    if (cur == want) return (int)h;
    h = (h + 1) & (unsigned)(cap - 1);
  }
  atomicOr(overflow, 1);
  return -1;
}

__device__ __forceinline__ unsigned lt_home(int cap, int cell) { return mix32((unsigned)cell) & (unsigned)(cap - 1); }

// Slot of `cell` or -1; `h` is its home slot and `cur` that slot's word (the
// caller loads it, so the loads of several cells are in flight together).
__device__ __forceinline__ int lt_resolve(const unsigned long long* cells, int cap, unsigned gen, int cell, unsigned h,
                                          unsigned long long cur) {
  const unsigned long long want = ((unsigned long long)gen << 32) | (unsigned)cell;
  for (int probe = 0; probe < cap; probe++) {
    if (cur == want) return (int)h;
    if ((unsigned)(cur >> 32) != gen) return -1;
    h = (h + 1) & (unsigned)(cap - 1);
    cur = cells[h];
  }
  return -1;
}

__device__ __forceinline__ int lt_find(const unsigned long long* cells, int cap, unsigned gen, int cell) {
  const unsigned h = lt_home(cap, cell);
  return lt_resolve(cells, cap, gen, cell, h, cells[h]);
}

__device__ __forceinline__ void lt_offer_key(unsigned long long* keys, size_t idx, unsigned gen, uint32_t key) {
  atomicMax(&keys[idx], ((unsigned long long)gen << 32) | (unsigned)(~key));
}
// 0xFFFFFFFF when the link has no key in this generation.
__device__ __forceinline__ uint32_t lt_key(const unsigned long long* keys, size_t idx, unsigned gen) {
  const unsigned long long v = keys[idx];
  return (unsigned)(v >> 32) == gen ? ~(uint32_t)v : 0xFFFFFFFFu;
}

// depthIndexCompact (:79-85)
__device__ __forceinline__ uint32_t depth_key(float depth, int elem) {
  return (((uint32_t)(depth * 32768.0f)) << 16) | (uint32_t)(uint16_t)elem;
}

// line_intersect (:89-124): link p1->p2 against segment p3-p4; depth = 1 - t
// in (0,1) or -1.  Only the segment's x-extent is tested (:117), so exactly
// vertical segments never hit.
__device__ __forceinline__ float seg_link(float x1, float y1, float x2, float y2, float x3, float y3, float x4,
                                          float y4, float& xo, float& yo) {
  const float a1 = (x1 - x2) * (y3 - y4) - (y1 - y2) * (x3 - x4);
  const float b1 = (x4 - x2) * (y3 - y4) - (y4 - y2) * (x3 - x4);
  if (fabsf(a1) <= 0.0f) return -1.0f;
  const float t1 = b1 / a1;
  if (t1 <= 0.0f || t1 >= 1.0f) return -1.0f;
  xo = t1 * x1 + (1.0f - t1) * x2;
  if ((x3 - xo) * (x4 - xo) < 0.0f) {
    yo = t1 * y1 + (1.0f - t1) * y2;
    return (float)(1.0 - (double)t1);
  }
  return -1.0f;
}

// Superset, without a division, of "t1 = b1 / a1 lies in (0, 1)" (the line
// test of seg_link): the quotient is positive only if b1 is nonzero with a1's
// sign, and rounds below 1 only if |b1| < |a1| (rounding is monotone and 1 is
// representable); NaN operands compare false here and fail there.
__device__ __forceinline__ bool seg_link_may_hit(float x1, float y1, float x2, float y2, float x3, float y3, float x4,
                                                 float y4) {
  const float a1 = (x1 - x2) * (y3 - y4) - (y1 - y2) * (x3 - x4);
  const float b1 = (x4 - x2) * (y3 - y4) - (y4 - y2) * (x3 - x4);
  return fabsf(b1) < fabsf(a1) && b1 != 0.0f && (b1 > 0.0f) == (a1 > 0.0f);
}

struct Hit {
  float depth;
  float b[3];
  float hit[3];
};

// intersectAtIndex<2>: barycentrics from glm::distance (:220-221).
// Segment endpoints (p3, p4) given by value.
__device__ __forceinline__ bool hit_seg2(float p3x, float p3y, float p4x, float p4y, float p1x, float p1y, float p2x,
                                         float p2y, Hit& h) {
  float xo = 0.f, yo = 0.f;
  const float d = seg_link(p1x, p1y, p2x, p2y, p3x, p3y, p4x, p4y, xo, yo);
  if (!(d > 0.0f && d < 1.0f)) return false;
  h.depth = d;
  h.hit[0] = xo;
  h.hit[1] = yo;
  h.hit[2] = 0.0f;
  const float ax = p4x - xo, ay = p4y - yo, bx = p4x - p3x, by = p4y - p3y;
  h.b[0] = sqrtf(ax * ax + ay * ay) / sqrtf(bx * bx + by * by);
  h.b[1] = 1.0f - h.b[0];
  h.b[2] = 0.0f;
  return true;
}

__device__ __forceinline__ bool hit_elem2(const float* v, const uint32_t* e, int elem, float p1x, float p1y, float p2x,
                                          float p2y, Hit& h) {
  const uint32_t s = e[2 * elem], t = e[2 * elem + 1];
  return hit_seg2(v[2 * s], v[2 * s + 1], v[2 * t], v[2 * t + 1], p1x, p1y, p2x, p2y, h);
}

// line_triangle_intersect (:306-341) with the NumericUtils 1e-6 tolerances;
// glm::normalize = v * (1 / sqrt(dot(v, v))).  The triangle's own quantities
// (edges, unit normal, Gram terms) are formed once per element.
struct Tri3 {
  float v0[3], e1[3], e2[3], n[3];
  float d00, d01, d11, den;
};

__device__ __forceinline__ Tri3 tri3(const float* v, const uint32_t* e, int elem) {
  float tv[3][3];
#pragma unroll
  for (int j = 0; j < 3; j++)
#pragma unroll
    for (int k = 0; k < 3; k++) tv[j][k] = v[e[3 * elem + j] * 3 + k];
  Tri3 T;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    T.v0[k] = tv[0][k];
    T.e1[k] = tv[1][k] - tv[0][k];
    T.e2[k] = tv[2][k] - tv[0][k];
  }
  const float c[3] = {T.e1[1] * T.e2[2] - T.e2[1] * T.e1[2], T.e1[2] * T.e2[0] - T.e2[2] * T.e1[0],
                      T.e1[0] * T.e2[1] - T.e2[0] * T.e1[1]};
  const float cs = 1.0f / sqrtf(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
#pragma unroll
  for (int k = 0; k < 3; k++) T.n[k] = c[k] * cs;
  T.d00 = T.e1[0] * T.e1[0] + T.e1[1] * T.e1[1] + T.e1[2] * T.e1[2];
  T.d01 = T.e1[0] * T.e2[0] + T.e1[1] * T.e2[1] + T.e1[2] * T.e2[2];
  T.d11 = T.e2[0] * T.e2[0] + T.e2[1] * T.e2[1] + T.e2[2] * T.e2[2];
  T.den = T.d00 * T.d11 - T.d01 * T.d01;
  return T;
}

// The plane parameter of the link p1 -> p1 + dd is num / den with
// num = n . (v0 - p1) and den = n . dd.
__device__ __forceinline__ float tri3_num(const Tri3& T, const float* p1) {
  const float a[3] = {T.v0[0] - p1[0], T.v0[1] - p1[1], T.v0[2] - p1[2]};
  return T.n[0] * a[0] + T.n[1] * a[1] + T.n[2] * a[2];
}
__device__ __forceinline__ float tri3_den(const Tri3& T, const float* dd) {
  return T.n[0] * dd[0] + T.n[1] * dd[1] + T.n[2] * dd[2];
}

// The rest of the test for a link whose plane parameter t passed 0 <= t <= 1
// (or is NaN): parallel-link rejection, then the barycentric inside test.
__device__ __forceinline__ bool tri3_finish(const Tri3& T, const float* p1, const float* dd, float t, Hit& h) {
  const float ds = 1.0f / sqrtf(dd[0] * dd[0] + dd[1] * dd[1] + dd[2] * dd[2]);
  const float d[3] = {dd[0] * ds, dd[1] * ds, dd[2] * ds};
  if (fabsf(T.n[0] * d[0] + T.n[1] * d[1] + T.n[2] * d[2]) <= 1e-6f) return false;
  const float ip[3] = {p1[0] + t * dd[0], p1[1] + t * dd[1], p1[2] + t * dd[2]};
  const float w[3] = {ip[0] - T.v0[0], ip[1] - T.v0[1], ip[2] - T.v0[2]};
  const float d20 = w[0] * T.e1[0] + w[1] * T.e1[1] + w[2] * T.e1[2];
  const float d21 = w[0] * T.e2[0] + w[1] * T.e2[1] + w[2] * T.e2[2];
  const float u0 = (T.d11 * d20 - T.d01 * d21) / T.den;
  const float v0 = (T.d00 * d21 - T.d01 * d20) / T.den;
  if (u0 >= 0.0f - 1e-6f && v0 >= 0.0f - 1e-6f && u0 + v0 <= 1.0f + 1e-6f) {
    h.depth = t;
    h.b[0] = 1.0f - u0 - v0;
    h.b[1] = u0;
    h.b[2] = v0;
    h.hit[0] = ip[0];
    h.hit[1] = ip[1];
    h.hit[2] = ip[2];
    return true;
  }
  return false;
}

// Link p1 -> p2 against a triangle: every test of the reference, the plane
// parameter first (a conjunction of the same predicates on the same values).
__device__ __forceinline__ bool hit_tri3(const Tri3& T, const float* p1, const float* p2, Hit& h) {
  const float dd[3] = {p2[0] - p1[0], p2[1] - p1[1], p2[2] - p1[2]};
  const float t = tri3_num(T, p1) / tri3_den(T, dd);
  if (t < 0.0f || t > 1.0f) return false;
  return tri3_finish(T, p1, dd, t, h);
}

__device__ __forceinline__ bool hit_elem3(const float* v, const uint32_t* e, int elem, const float* p1, const float* p2,
                                          Hit& h) {
  return hit_tri3(tri3(v, e, elem), p1, p2, h);
}

// Candidate cells of an element: getBoundingBox (max starts at FLT_MIN) / dx,
// widened by one cell, clipped to the grid.  lo/hi inclusive.
template <int DIM>
__device__ __forceinline__ void elem_window(const float* v, const uint32_t* e, int elem, float dx, const int* n, int* lo,
                                            int* hi) {
#pragma unroll
  for (int a = 0; a < DIM; a++) {
    float mn = FLT_MAX, mx = FLT_MIN;
#pragma unroll
    for (int j = 0; j < DIM; j++) {
      const float c = v[DIM * e[DIM * elem + j] + a];
      mn = fminf(mn, c);
      mx = fmaxf(mx, c);
    }
    lo[a] = max((int)(mn / dx) - 1, 0);
    hi[a] = min((int)(mx / dx) + 1, n[a] - 1);
  }
}

// elem_window<2> of a segment given by its end points.
__device__ __forceinline__ void seg_window(f32x2 a, f32x2 b, float dx, const int* n, int* lo, int* hi) {
  const float c[2][2] = {{a.x, b.x}, {a.y, b.y}};
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const float mn = fminf(fminf(FLT_MAX, c[k][0]), c[k][1]);
    const float mx = fmaxf(fmaxf(FLT_MIN, c[k][0]), c[k][1]);
    lo[k] = max((int)(mn / dx) - 1, 0);
    hi[k] = min((int)(mx / dx) + 1, n[k] - 1);
  }
}

}  // namespace ff

#include "ff_internal.h"

namespace ff {

// Lattice vectors of D3Q27 packed two bits per direction (c + 1), for
// direction indices only known at run time.
constexpr unsigned long long d3_pack(int axis) {
  unsigned long long p = 0;
  for (int i = 0; i < 27; i++) {
    const int c = axis == 0 ? D3::cx(i) : (axis == 1 ? D3::cy(i) : D3::cz(i));
    p |= (unsigned long long)(c + 1) << (2 * i);
  }
  return p;
}
__device__ __forceinline__ int d3_c(unsigned long long packed, int i) { return (int)((packed >> (2 * i)) & 3ull) - 1; }

// Lanes that handle one element in the 2D detection and element sums: a DPP
// row.  A segment's candidate window holds 9-20 cells (segments of 0.4-1.5
// cells), so 16 lanes take it in one or two passes and a wave works on four
// elements; with a wave or half a wave per element most lanes had no cell.
constexpr int kRow = 16;

// Lattice vectors of D2Q9 packed two bits per direction (c + 1).
constexpr unsigned d2_pack(int axis) {
  unsigned p = 0;
  for (int i = 0; i < 9; i++) p |= (unsigned)((axis == 0 ? D2::cx(i) : D2::cy(i)) + 1) << (2 * i);
  return p;
}

// 2D link detection (the loops of mrSolver2DComputeOccupancyFlagKernel_v3,
// FsiCoupling2D.cu:44-74): kRow lanes per element, one window cell per lane
// and pass.  A lane tests its cell's eight links against the segment's line
// without a division (seg_link_may_hit), finishes the survivors, enters the
// cell once if any link hit, and offers the hits' depthIndexCompact keys.
// Bound by the chain of dependent loads (element -> vertices -> flags -> table)
// and by instruction issue: with one (cell, direction) task per lane every
// task divided, and every hit walked the table by itself.
// `block` indexes groups of blockDim / kRow elements; the links are entered
// under `tag` for the vertex positions `v`.
__device__ __forceinline__ void build_links_rows2(const LinkArgs& la, long long block, unsigned tag, const float* v) {
  constexpr int K = 8;
  const long long e = block * (long long)(blockDim.x / kRow) + threadIdx.x / kRow;
  if (e >= (long long)la.ne) return;
  const int lane = (int)(threadIdx.x % kRow);
  const u32x2 ends = load2(dev_global(la.e) + 2 * e);
  const f32x2 p3 = load2(dev_global(v) + 2 * (size_t)ends.x), p4 = load2(dev_global(v) + 2 * (size_t)ends.y);
  const int n[2] = {la.nx, la.ny};
  int lo[2], hi[2];
  seg_window(p3, p4, la.cl, n, lo, hi);
  const int wx = hi[0] - lo[0] + 1, wy = hi[1] - lo[1] + 1;
  if (wx <= 0 || wy <= 0) return;
  const int ncell = wx * wy;
  const uint8_t* flags = dev_global(la.flags);
  unsigned long long* cells = table_cells(la, tag);
  unsigned long long* keys = table_keys<2>(la, tag);
  for (int k = lane; k < ncell; k += kRow) {
    const int j0 = k / wx;
    const int i = lo[0] + k - j0 * wx, j = lo[1] + j0;
    const int cell = j * la.nx + i;
    if (!is_updated(flags[cell])) continue;
    const float fi = (float)i, fj = (float)j, x1 = fi * la.cl, y1 = fj * la.cl;
    unsigned may = 0;
#pragma unroll
    for (int l = 1; l <= K; l++)
      if (seg_link_may_hit(x1, y1, (fi - (float)D2::cx(l)) * la.cl, (fj - (float)D2::cy(l)) * la.cl, p3.x, p3.y, p4.x,
                           p4.y))
        may |= 1u << l;
    auto test = [&](int l, Hit& h) {
      const float cx = (float)((int)((d2_pack(0) >> (2 * l)) & 3u) - 1);
      const float cy = (float)((int)((d2_pack(1) >> (2 * l)) & 3u) - 1);
      return hit_seg2(p3.x, p3.y, p4.x, p4.y, x1, y1, (fi - cx) * la.cl, (fj - cy) * la.cl, h);
    };
    unsigned hits = 0;
    for (unsigned m = may; m; m &= m - 1) {
      const int l = __ffs((int)m) - 1;
      Hit h;
      if (test(l, h)) hits |= 1u << l;
    }
    if (!hits) continue;
    const int slot = lt_claim(cells, la.cap, tag, cell, &la.st->overflow);
    if (slot < 0) continue;
    for (unsigned m = hits; m; m &= m - 1) {
      const int l = __ffs((int)m) - 1;
      Hit h;
      test(l, h);
      lt_offer_key(keys, (size_t)slot * K + (l - 1), tag, depth_key(h.depth, (int)e));
    }
  }
}

// 2D link detection of a domain stepped on its own: kRow lanes per (element,
// direction), one window cell per lane.  Eight times the waves of
// build_links_rows2 for the same predicates, hits and keys, and the shorter
// chain (one test and one table walk per lane), which is what a launch of few
// blocks waits for: 5.6 us against 7.4 us for the 600 segments of a 1200x400
// swimmer; with 64 domains (26.9 against 16.9 us) the launch is bound by issue.
// `block` indexes groups of blockDim / kRow pairs.
__device__ __forceinline__ void build_links_pairs2(const LinkArgs& la, long long block, unsigned tag, const float* v) {
  constexpr int K = 8;
  const int lane = (int)(threadIdx.x % kRow);
  const long long pair = block * (long long)(blockDim.x / kRow) + threadIdx.x / kRow;
  if (pair >= (long long)la.ne * K) return;
  const int elem = (int)(pair / K), l = (int)(pair % K) + 1;
  const u32x2 ends = load2(la.e + 2 * (size_t)elem);
  const f32x2 p3 = load2(v + 2 * (size_t)ends.x), p4 = load2(v + 2 * (size_t)ends.y);
  const int n[2] = {la.nx, la.ny};
  int lo[2], hi[2];
  seg_window(p3, p4, la.cl, n, lo, hi);
  const int wx = hi[0] - lo[0] + 1, wy = hi[1] - lo[1] + 1;
  if (wx <= 0 || wy <= 0) return;
  const int ncell = wx * wy;
  const float cx = (float)D2::cx(l), cy = (float)D2::cy(l);
  unsigned long long* cells = table_cells(la, tag);
  unsigned long long* keys = table_keys<2>(la, tag);
  for (int k = lane; k < ncell; k += kRow) {
    const int j0 = k / wx;
    const int i = lo[0] + k - j0 * wx, j = lo[1] + j0;
    const int cell = j * la.nx + i;
    Hit h;
    const bool hit = is_updated(la.flags[cell]) &&
                     hit_seg2(p3.x, p3.y, p4.x, p4.y, (float)i * la.cl, (float)j * la.cl, ((float)i - cx) * la.cl,
                              ((float)j - cy) * la.cl, h);
    const int slot = hit ? lt_claim(cells, la.cap, tag, cell, &la.st->overflow) : -1;
    if (slot >= 0) lt_offer_key(keys, (size_t)slot * K + (l - 1), tag, depth_key(h.depth, elem));
  }
}

// Superset test, without a division, of "num / den rounds into [0, 1] or is
// NaN" (the plane-parameter test of line_triangle_intersect): num = 0 gives
// +-0 or NaN; a zero den otherwise gives +-inf; equal signs need
// |num| <= |den| (1 + 2^-24) for the quotient to round to at most 1, which
// fl(|den| * 1.0001) bounds from above (rounding is monotone); opposite signs
// round to -0 only when the quotient underflows, below 1e-30 by far.
__device__ __forceinline__ bool tri3_t_may_pass(float num, float den) {
  if (num == 0.0f) return true;
  if (den == 0.0f) return false;
  const float an = fabsf(num), ad = fabsf(den);
  return (num > 0.0f) == (den > 0.0f) ? an <= ad * 1.0001f : an < ad * 1e-30f;
}

// Threads that handle one triangle in the 3D detection and element sums: a
// block, or a wave (four elements a block) where the elements fill the chip anyway.
constexpr int kBlock3 = 256;
template <int NT>
__device__ __forceinline__ void group_sync() {
  if constexpr (NT == 64) {  // one wave: its LDS accesses are in order, the compiler's need to be
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
    __syncthreads();
  }
}

// Lists of links of build_links_group3.
template <int NT>
struct Det3Lists {
  static constexpr int CAP = 16 * NT;
  unsigned short may[CAP], hit[CAP];
  int wave[NT / 64], nhit;
};

// 3D link detection with NT threads per element, cell-major: each thread takes
// U cells of the element's window per pass, forms num = n . (v0 - p1), and only
// cells within 2 cl of the triangle's plane go on (no link of length <= sqrt(3)
// cl from a farther cell reaches it; the margin is far above the rounding of
// the link ends for grids up to millions of cells per axis).  Their 26 links
// (unrolled, lattice vectors as constants) whose plane parameter t = num / (n .
// dd) may lie in [0, 1] (tri3_t_may_pass, no division) form a bit mask; a
// prefix sum of the masks' counts lists the survivors in LDS, all threads
// finish them (t itself, parallel test, barycentrics), and the hits, listed
// again, are entered in the table together.  A block per element is bound by
// its chain of loads, barriers and table round trips: one list position per
// direction from an LDS counter, with a barrier every fourth, took 21 us for
// the 320 triangles of a sphere.
template <int NT>
__device__ __forceinline__ void build_links_group3(const LinkArgs& la, int elem, unsigned tag, const float* v,
                                                   Det3Lists<NT>& lds) {
  constexpr int K = 26, NW = NT / 64, U = NT == 64 ? 1 : 2, CAP = Det3Lists<NT>::CAP;
  static_assert(U * NT <= 2048, "a cell of the pass and a direction in 16 bits");
  const int n[3] = {la.nx, la.ny, la.nz};
  const uint32_t* e = dev_global(la.e);
  v = dev_global(v);
  int lo[3], hi[3];
  elem_window<3>(v, e, elem, la.cl, n, lo, hi);
  const int wx = hi[0] - lo[0] + 1, wy = hi[1] - lo[1] + 1, wz = hi[2] - lo[2] + 1;
  if (wx <= 0 || wy <= 0 || wz <= 0) return;  // the same for the whole group, as every branch around a group_sync
  const int ncell = wx * wy * wz;
  const Tri3 T = tri3(v, e, elem);
  const float far = 2.0f * la.cl;
  const uint8_t* flags = dev_global(la.flags);
  unsigned long long* cells = table_cells(la, tag);
  unsigned long long* keys = table_keys<3>(la, tag);
  const int tid = (int)threadIdx.x & (NT - 1), lane = tid & 63, wave = tid >> 6;
  // link q of the pass at c0: bits 5.. the cell's place in the pass, 0-4 the direction
  auto link_test = [&](int c0, unsigned q, int& cell, int& l, Hit& h) {
    const int k = c0 + (int)(q >> 5);
    l = (int)(q & 31u);
    const int i = lo[0] + k % wx, j = lo[1] + (k / wx) % wy, z = lo[2] + k / (wx * wy);
    cell = (z * la.ny + j) * la.nx + i;
    const float p1[3] = {(float)i * la.cl, (float)j * la.cl, (float)z * la.cl};
    const float p2[3] = {((float)i - (float)d3_c(d3_pack(0), l)) * la.cl,
                         ((float)j - (float)d3_c(d3_pack(1), l)) * la.cl,
                         ((float)z - (float)d3_c(d3_pack(2), l)) * la.cl};
    return hit_tri3(T, p1, p2, h);
  };
  for (int c0 = 0; c0 < ncell; c0 += U * NT) {
    unsigned may[U];
    bool upd[U];
#pragma unroll
    for (int w = 0; w < U; w++) {  // the flags in flight together
      const int k = c0 + w * NT + tid;
      upd[w] = false;
      if (k < ncell) {
        const int i = lo[0] + k % wx, j = lo[1] + (k / wx) % wy, z = lo[2] + k / (wx * wy);
        upd[w] = is_updated(flags[(z * la.ny + j) * la.nx + i]);
      }
    }
    int count = 0;
#pragma unroll
    for (int w = 0; w < U; w++) {
      may[w] = 0;
      if (upd[w]) {
        const int k = c0 + w * NT + tid;
        const float fi = (float)(lo[0] + k % wx), fj = (float)(lo[1] + (k / wx) % wy),
                    fz = (float)(lo[2] + k / (wx * wy));
        const float p1[3] = {fi * la.cl, fj * la.cl, fz * la.cl};
        const float num = tri3_num(T, p1);
        if (fabsf(num) <= far) {
#pragma unroll
          for (int l = 1; l <= K; l++) {
            const float p2[3] = {(fi - (float)D3::cx(l)) * la.cl, (fj - (float)D3::cy(l)) * la.cl,
                                 (fz - (float)D3::cz(l)) * la.cl};
            const float dd[3] = {p2[0] - p1[0], p2[1] - p1[1], p2[2] - p1[2]};
            if (tri3_t_may_pass(num, tri3_den(T, dd))) may[w] |= 1u << l;
          }
        }
      }
      count += __popc(may[w]);
    }
    // prefix sum of the counts over the group
    int before = count;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(before, off, 64);
      if (lane >= off) before += o;
    }
    int total = 0;
    if constexpr (NW == 1) {
      total = __shfl(before, 63, 64);
      before -= count;
    } else {
      if (lane == 63) lds.wave[wave] = before;
      group_sync<NT>();
      before -= count;
#pragma unroll
      for (int w = 0; w < NW; w++) {
        before += w < wave ? lds.wave[w] : 0;
        total += lds.wave[w];
      }
    }
    for (int base = 0; base < total; base += CAP) {
      if (tid == 0) lds.nhit = 0;
      int at = before - base;
#pragma unroll
      for (int w = 0; w < U; w++)
        for (unsigned m = may[w]; m; m &= m - 1, at++)
          if (at >= 0 && at < CAP) lds.may[at] = (unsigned short)(((w * NT + tid) << 5) | (__ffs((int)m) - 1));
      group_sync<NT>();
      const int ns = min(total - base, CAP);
      for (int q0 = 0; q0 < ns; q0 += NT) {
        const int q = q0 + tid;
        int cell, l;
        Hit h;
        const bool hit = q < ns && link_test(c0, lds.may[q], cell, l, h);
        const unsigned long long m = __ballot(hit);
        if (m) {
          int pos = 0;
          if (lane == 0) pos = atomicAdd(&lds.nhit, (int)__popcll(m));
          pos = __shfl(pos, 0, 64);
          if (hit) lds.hit[pos + (int)__popcll(m & ((1ull << lane) - 1ull))] = lds.may[q];
        }
      }
      group_sync<NT>();
      const int nh = lds.nhit;
      for (int q = tid; q < nh; q += NT) {
        int cell, l;
        Hit h;
        link_test(c0, lds.hit[q], cell, l, h);
        const int slot = lt_claim(cells, la.cap, tag, cell, &la.st->overflow);
        if (slot >= 0) lt_offer_key(keys, (size_t)slot * K + (l - 1), tag, depth_key(h.depth, elem));
      }
      group_sync<NT>();  // the lists and counters are free again
    }
    if (total == 0) group_sync<NT>();  // lds.wave is read before the next pass writes it
  }
}

// LDS of a detection block.
template <int DIM>
struct DetLds {};
template <>
struct DetLds<3> {
  union {
    Det3Lists<kBlock3> block;
    Det3Lists<64> wave[kBlock3 / 64];
  };
};

// Detection block of 256 threads: 2D takes blockDim / kRow elements (ROWS) or
// (element, direction) pairs, 3D `epb` elements.
template <int DIM, bool ROWS>
__device__ __forceinline__ void detect_block(const LinkArgs& la, long long block, unsigned tag, const float* v,
                                             DetLds<DIM>& lds, int epb) {
  if constexpr (DIM == 3) {
    if (epb == 1) {
      if (block < la.ne) build_links_group3<kBlock3>(la, (int)block, tag, v, lds.block);
    } else {
      const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
      const long long elem = block * (kBlock3 / 64) + wave;
      if (elem < la.ne) build_links_group3<64>(la, (int)elem, tag, v, lds.wave[wave]);
    }
  } else if constexpr (ROWS) {
    build_links_rows2(la, block, tag, v);
  } else {
    build_links_pairs2(la, block, tag, v);
  }
}

}  // namespace ff
