// tiling.h -- the block-to-tile mapping shared by the tile-marching kernels
// (fused sweep, conduction, gravity force) and the XCD count the batched
// work queues are split by.
#pragma once

#include <hip/hip_runtime.h>

namespace evh {

// Blocks are dispatched round-robin over the 8 XCDs of the chip, each with
// its own L2.  Block b runs on XCD b % 8; giving XCD j the contiguous run of
// tiles [j*T/8, (j+1)*T/8) (x fastest, then y, then z chunk) keeps the halo
// columns a block shares with its x and y neighbours in one L2.  Returns -1
// for the padding blocks of a grid rounded up to a multiple of 8.
constexpr int kXcds = 8;

__device__ __forceinline__ int xcd_tile(int b, int ntiles) {
  const int j = b % kXcds, i = b / kXcds;
  const int base = ntiles / kXcds, rem = ntiles % kXcds;
  const int count = base + (j < rem ? 1 : 0);
  if (i >= count) return -1;
  return j * base + (j < rem ? j : rem) + i;
}

// blocks to launch for ntiles tiles (a multiple of the XCD count)
inline int xcd_blocks(int ntiles) { return kXcds * ((ntiles + kXcds - 1) / kXcds); }

// The column tile of the 3-D march for tile height 12, 192 columns either way:
// 16 x 12, or in FP32 32 x 6 (wide) where that takes at most 5% more tiles to
// cover a plane of the grid (or of all boxes together).  The wide tile's ring
// has half the columns beyond its x sides, each of which costs the L1 a
// request of a whole line for one value, and more columns in all.  FP32 is
// bound by those requests: 512^3 2.64 ms wide against 2.86, 384^3 1.23 against
// 1.31, 256^3 0.429 against 0.440 (7 to 19 steps of a blast, events).  FP64 is
// bound by instruction issue, the ring's included: 512^3 5.65 ms wide against
// 5.49, 384^3 2.45 against 2.39, 256^3 0.838 against 0.805.
inline long long tiles_of(int nx, int ny, int tx, int ty) {
  return (long long)((nx + tx - 1) / tx) * ((ny + ty - 1) / ty);
}
inline bool wide_tile(long long tiles32x6, long long tiles16x12) { return 20 * tiles32x6 <= 21 * tiles16x12; }

// Chunk lengths when the tuning leaves them open.  A block's march is
// serial, so on a small grid long chunks leave most of the GPU idle and a
// pass takes the march's latency; short chunks cost a few planes more of
// loads and primitives per chunk.  The results do not depend on the chunk.

// The time of a march in microseconds, as measured on MI355X: while every
// block is resident (up to `per_cu` on each of the 256 CUs), alone + plane
// times the chunk, both growing with the blocks that share a CU; beyond that
// so many rounds of the resident blocks, where a partly filled second one
// counts two thirds of what it leaves empty; over more rounds the blocks drift
// apart and only the last one's end shows.
struct MarchCost {
  int per_cu;              // resident blocks per CU
  double alone[4];         // with 1, 2, .. blocks per CU: launch and prologue
  double plane[4];         // and each plane (row) of the chunk
  double round, per_plane; // the same for a full round
};
// The constants reproduce the measured times of cubes of 24 to 512, slabs and
// bricks within 15%, and the chunk they lead to is within 8% of the fastest: FP64
// 32^3 13.7 us with 1 plane (21.7 with 4), 64^3 29.8 with 4, 96^3 65 with 12
// (72 with 8), 192^3 338 with 24 (349 with 16); FP32-mixed 64^3 23.5 with 2
// (31.9 with 8), 96^3 35.5 with 6 (42 with 8); 2-D 128^2 11.3 with 1 row (13.4
// with 2), 1024^2 FP32-mixed 31.7 with 8 (38.7 with 4).
constexpr MarchCost kMarch64 = {2, {9.1, 11.5, 0, 0}, {3.15, 4.45, 0, 0}, 7.0, 4.2};
constexpr MarchCost kMarch32 = {4, {10, 10, 13, 13}, {2.5, 3.0, 3.6, 4.3}, 9.0, 3.8};
constexpr MarchCost kMarch2d64 = {3, {8.5, 11, 13, 0}, {2.55, 3.2, 4.4, 0}, 8.0, 4.9};
constexpr MarchCost kMarch2d32 = {4, {7.6, 9, 14, 14}, {2.0, 2.3, 2.7, 3.1}, 6.0, 3.2};

// the chunk of n planes (rows), `most` at most, that the march of `columns`
// tiles per plane takes the least time with
inline int march_chunk(const MarchCost &m, long long columns, int n, int most) {
  constexpr int kCus = 256;
  constexpr int tries[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64, 96, 128};
  int best = 1;
  double least = 0;
  for (int c : tries) {
    if (c > most || (c > 1 && c / 2 >= n)) break;
    const long long blocks = columns * ((n + c - 1) / c);
    const int share = (int)((blocks + kCus - 1) / kCus < m.per_cu ? (blocks + kCus - 1) / kCus : m.per_cu);
    double t;
    if (blocks <= (long long)kCus * m.per_cu) {
      t = m.alone[share - 1] + m.plane[share - 1] * c;
    } else {
      const double r = (double)blocks / (kCus * m.per_cu);
      const double up = (double)(long long)r + ((double)(long long)r < r ? 1 : 0);
      t = m.alone[0] / 2 + (r < 2 ? r + 0.65 * (up - r) : 0.93 * r + 0.3) * (m.round + m.per_plane * c);
    }
    if (c == 1 || t < least) {
      least = t;
      best = c;
    }
  }
  return best;
}

// z_chunk: planes per block of the conduction and gravity passes with
// `columns` column tiles per plane: `start`, halved while the grid would give
// fewer than 2048 blocks, but not below nz/8 (a power of two, 4 at least): the
// conduction pass of a 128^3 hot blob 0.082 ms at 16 planes against 0.207 ms
// at 4 (1024 blocks of 4 planes).
inline int z_chunk(long long columns, int nz, int start) {
  int lo = 4;
  while (lo < start && 2 * lo * 8 <= nz) lo *= 2;
  int c = start;
  while (c > lo && columns * ((nz + c - 1) / c) < 2048) c /= 2;
  return c;
}

}  // namespace evh
