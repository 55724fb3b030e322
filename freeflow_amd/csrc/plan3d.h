// plan3d.h -- how a 3D domain without a tile of its own steps, by its grid:
// the separable form, whole rows, or the shape of its tiles.  Host code only;
// every time below is us a step on one MI355X, periodic boxes, both builds in
// turn.
#pragma once

#include <stddef.h>

#include <algorithm>
#include <vector>

namespace ff {

// Tiles of the whole-row kernels (separable3d.h, rows3d.h).
constexpr int kSepTX = 64, kSepTY = 8;
constexpr int kRowsTX = 64, kRowsTY = 6;

// Cells from which a domain without a body takes columns (default_tile3).
constexpr long long kColumnCells = 580000;

inline long long ceil_div(long long a, long long b) { return (a + b - 1) / b; }

struct Grid3 {
  int nx, ny, nz;
  long long cells() const { return (long long)nx * ny * nz; }
  long long tiles(int tx, int ty) const { return ceil_div(nx, tx) * ceil_div(ny, ty); }
};

// Both moment buffers beyond the 256 MB last-level cache.
inline bool beyond_cache(size_t plane, size_t planes, size_t elem) { return 2.0 * (double)plane * planes * elem > 256e6; }

// FP32 fast step of staged columns of tx x ty x zc cells while the buffers
// stay in the last-level cache: the blocks go round the 256 CUs, and a column
// of n planes takes about n + 1 plane steps.  16x12x8 (0.735 a plane step) and
// 32x12x16 (1.4) within 7 % of 100 measured grids of more than 256 blocks.
inline double columns_us(const Grid3& g, int tx, int ty, int zc, double plane_step) {
  const long long rounds = ceil_div(g.tiles(tx, ty) * ceil_div(g.nz, zc), 256);
  return 8.0 + plane_step * (std::min(g.nz, zc) + 1) * (double)rounds;
}
inline double columns7_us(const Grid3& g) { return columns_us(g, 16, 12, 8, 0.735); }
inline double columns15_us(const Grid3& g) { return columns_us(g, 32, 12, 16, 1.4); }

// The number of z chunks with the fewest plane steps for `cols` columns of
// rows, of which `slots` share the chip: a chunk of n planes takes n + 2.
struct RowChunks {
  int chunks = 0;
  long long steps = 0, rounds = 0;
};
inline RowChunks row_chunks(long long cols, int nz, int slots) {
  RowChunks r;
  for (int c = 1; c <= nz; c++) {
    const long long rounds = ceil_div(cols * c, slots), steps = (ceil_div(nz, c) + 2) * rounds;
    if (!r.chunks || steps < r.steps) r = {c, steps, rounds};
  }
  return r;
}

// Number of z chunks of the separable form for a grid, or 0 where the columns
// or the rows serve.  A pass of blocks over the chip takes about 1.75 a plane
// step and 1.5 at its start, within 6 % while the buffers stay in the
// last-level cache.  Against the best column: 52.7 / 48.1 at 203x101x97, 60 /
// 45 at 17x13x3500, 61.8 / 55.0 at 211x105x125, 61.0 / 36.6 at 1000x1000x1
// (few planes a chunk, each chunk with two more) keep the columns; 31.2 / 32.4
// at 160x96x96, 72.5 / 74.3 at 146x151x150, 53.6 / 51.8 at 130x130x130 and
// 76.8 / 72.3 at 198x175x90 lie at the line.  Beyond the cache the columns lose
// more than this says (145x138x213 112 / 133 at a ratio of 1.03, 2000x1000x4
// 206 / 213 at 1.26, but 1769x1213x2 164 / 137 at 1.41).  Grids whose columns
// take fewer than 57 blocks a plane step were never timed with it.
// Buffers beyond the buffer accesses' 4 GiB take the columns too.
inline int sep3d_chunks(const Grid3& g, size_t plane) {
  if ((10 * plane + (size_t)g.nx * g.ny) * sizeof(float) >= 0xFFFF0000ull) return 0;
  const RowChunks r = row_chunks(g.tiles(kSepTX, kSepTY), g.nz, 256);
  if (57 * r.steps >= g.tiles(16, 12) * ceil_div(g.nz, 8)) return 0;
  const double us = 3.0 + 1.75 * (double)r.steps + 1.5 * (double)r.rounds;
  const double line = beyond_cache(plane, 10, sizeof(float)) ? 1.3 : 1.03;
  return us <= line * std::min(columns7_us(g), columns15_us(g)) ? r.chunks : 0;
}

// Most planes of a chunk for members that take the separable form together
// (chunks do not change a bit): each member's own count would cut a batch that
// fills the chip anyway into chunks of few planes with two more each.  Eight
// 64x128x64 domains: 146 us a step in chunks of 4, 85 of 32 (the columns 117);
// 32 of them 562 and 299, 24 of 179x51x42 380 and 220.
inline int batch_chunk_planes(const std::vector<Grid3>& members) {
  int best = 1, most = 1;
  for (const Grid3& g : members) most = std::max(most, g.nz);
  long long fewest = 0;
  for (int planes = 1; planes <= most; planes++) {
    long long blocks = 0;
    for (const Grid3& g : members) blocks += g.tiles(kSepTX, kSepTY) * ceil_div(g.nz, planes);
    const long long steps = (planes + 2) * ceil_div(blocks, 256);
    if (!fewest || steps < fewest) {
      fewest = steps;
      best = planes;
    }
  }
  return best;
}

// Number of z chunks of the rows for a grid, or 0 where the columns are
// faster.  A step of 512 blocks takes as long as about 100 blocks of the
// 16x12x8 column (2.6 us and 0.027 us a block in FP16 fast, 3.9 and 0.040 in
// FP32 reference order): 51 us against 48 at 203x101x97, 33 against 31 at
// 160x96x96 (padding to 64 cells), 69 against 75 at 256x128x128.  Columns of
// fewer than eight planes take n + 1 of 9 plane steps: FP32 reference order
// 67.9 against 44.7 at 1000x1000x1, 50.8 / 44.4 at 690x429x5,
// 910x352x2 33.2 / 25.7; level up to a ratio of 1.2 (66.0 / 61.6 at 800x700x4,
// but FP16 19.9 / 20.6 at 122x1398x4).  Smaller grids would take boxes (22.0
// against 29.3 at 692x233x3).  Buffers beyond 4 GiB take the columns.
inline int rows3d_chunks(const Grid3& g, size_t plane, size_t planes, size_t elem) {
  if ((plane * planes + (size_t)g.nx * g.ny) * elem >= 0xFFFF0000ull) return 0;
  const RowChunks r = row_chunks(g.tiles(kRowsTX, kRowsTY), g.nz, 512);
  const long long blocks = g.tiles(16, 12) * ceil_div(g.nz, 8);
  if (100 * r.steps >= blocks) return 0;
  if (g.cells() < kColumnCells) return r.chunks;
  return 900.0 * (double)r.steps <= 1.2 * (double)((std::min(g.nz, 8) + 1) * blocks) ? r.chunks : 0;
}

// Tile of a domain whose tile was neither set nor tuned; any tile gives the
// same results.  us a step (FP32 reference order / fast):
//   box 8x8x4: few cells fill the chip only in small boxes.  64^3 16.6 / 13.1
//   against 29.9 / 25.1 of the 16x12x8 column, 80^3 28.4 / 24.8 against
//   33.7 / 28.9, 96x96x64 32.9 / 28.9 against 34.1 / 28.5; at 203x101x97
//   104 / 90 against 66 / 56.  With a body the launch waits for its boundary
//   cells too: 64^3 23.3 / 22.1 against 25.0 / 20.8, 96x64x64 30.4 / 27.8
//   against 30.2 / 24.1, 160x96x96 84.7 / 73.6 against 56.1 / 45.0.
//   Also where the columns are mostly padding: a box takes as long as 3.4
//   plane steps of a column.  8x8x10000 33.4 / 26.9 against 45.5 / 34.8 (5.0
//   steps a box), 8x100x1000 41.9 / 33.8 against 46.0 / 35.8 (3.46), but
//   17x13x3500 65.9 / 51.8 against 59.1 / 46.2 (3.33).
//   column 16x12x8 in between.
//   column 32x12x16 once both moment buffers exceed the last-level cache, so
//   that halo cells are read from memory again, and if its tiles are not
//   padding for more than a fifth: 256x192x160 189 / 177 against 229 / 224
//   (FP16 148 against 153), 384x256x256 650 / 622 against 811 / 807, but
//   100x300x200 (33 % padding) 216 / 198 against 194 / 191, and FP16
//   250x150x150 (225 MB) 126 against 103; 1133x1837x2 147 against 174 (fast,
//   one short column is no padding).  Also where the chunks of eight
//   planes leave a remainder and one of sixteen does not: 196x850x11 51.0 /
//   40.1 against 68.4 / 56.5, 293x378x9 42.8 / 33.5 against 50.2 / 41.9.
inline int default_tile3(const Grid3& g, size_t plane, size_t planes, size_t elem, bool body) {
  const long long n = g.cells();
  if (n < (body ? 350000 : kColumnCells)) return 0;
  const long long boxes = g.tiles(8, 8) * ceil_div(g.nz, 4);
  if ((double)(g.tiles(16, 12) * (g.nz + 2 * ceil_div(g.nz, 8))) > 3.4 * (double)boxes) return 0;
  const long long padded = g.tiles(32, 12) * 32 * 12 * ceil_div(g.nz, 16) * std::min(g.nz, 16);
  if (beyond_cache(plane, planes, elem)) return 5 * padded < 6 * n ? 15 : 7;
  return columns15_us(g) < 0.9 * columns7_us(g) ? 15 : 7;
}

}  // namespace ff
