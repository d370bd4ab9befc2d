// Projections of 65 to some hundred rows: whether, and into how many pieces, K is shared between workgroups
// (host code, no device types: also compiled by the CPU tests).
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace ellm {
namespace proj {

// Tiles of 128 token_blocks tokens x one head, k_split workgroups a tile (1: K stays whole), with 128 tokens of four waves
// of a head each or eight of half a head.
struct ProjectSplit {
  uint32_t token_blocks, k_split;
  bool half_heads;
};

inline size_t split_floats(const ProjectSplit& s, uint32_t rows, uint32_t heads) {
  return s.k_split > 1 ? (size_t)s.k_split * rows * heads * 128 : 0;
}

// Estimated time (us, 256 units).  A chunk of 64 of K takes 0.5 us a workgroup of 128 tokens and 0.65 of 256 (weights
// from memory); the operands of all tiles come out of the L2s at 14 TB/s and the weights from memory at 4.6; the second
// launch and the partial sums, written and read, are 4 us and their bytes at 6 TB/s.
inline double project_tiles_us(const ProjectSplit& s, uint32_t rows, uint32_t heads, uint32_t K) {
  const double chunks = (K / 64 + s.k_split - 1) / s.k_split, tokens = 128.0 * s.token_blocks;
  const double tiles = (rows + 128 * s.token_blocks - 1) / (128 * s.token_blocks) * (double)heads;
  const double chain = chunks * (s.token_blocks == 1 ? 0.5 : 0.65);
  if (s.k_split == 1) return 5.0 + chain;
  const double operands = tiles * (tokens + 128) * K * 2 / 14e6, weights = (double)heads * 128 * K * 2 / 4.6e6;
  const double walk = chain > operands ? chain : operands;
  return 9.0 + (walk > weights ? walk : weights) + 2.0 * split_floats(s, rows, heads) * 4 / 6e6;
}

// Three to eight workgroups a tile, all of them at once, one per unit, pieces of at least four chunks; where that is
// estimated 5 % below one round of whole tiles.  Follows from the sizes alone.  Two a tile gained nothing that lasts
// (2048 <- 4096, 700 rows 32.9 / 33.0), nor did three of 256 tokens below 96 chunks (a layer of 800 rows, 2048 wide, 73.7 /
// 75.0; 4096 <- 4096, 400 rows 31.7 / 30.9), nor any of 256 tokens on all units at once (those 800 rows, four, 73.1 / 78.0).  Whole / shared, weights from memory, f16 (us; tokens a tile / pieces):
//   2048 <- 4096   79 rows 32.4 / 14.6 (128 / 8)   128 37.2 / 16.0 (128 / 8)   234 35.2 / 18.6 (128 / 8)   400 30.0 / 22.6 (128 / 4)
//                  700 32.9 / 28.1 (256 / 4)
//   5120 <- 2048   79 21.0 / 15.5 (128 / 6)   128 23.4 / 17.8 (128 / 6)   400 stays whole: 20.3 / 26.2 and more
//   4096 <- 4096   79 34.7 / 17.8 (128 / 8)   128 39.6 / 20.3   234 37.2 / 23.7 (128 / 4)   400 stays whole
//   10240 <- 8192  79 67.6 / 45.1 (128 / 3)   128 77.2 / 49.7   234 73.3 / 63.3 (256 / 3)
//   8192 <- 8192   79 64.8 / 42.9 (128 / 4)   128 74.5 / 46.9   234 70.5 / 56.9 (256 / 4)
// These with four waves a workgroup of 128 tokens.  One wave a SIMD waits for every operand; eight waves of half a head read
// a fifth more from LDS, but take turns (layer of a chunk, four / eight waves: 2048 wide, 65 rows 32.5 / 28.1, 128 37.3 /
// 33.0, 300 46.5 / 42.4; 4096 wide, 128 55.4 / 51.8; 8192 wide, 65 82.2 / 75.2, 128 93.7 / 90.7), except where all units are
// at work: 500 rows 2048 wide, 256 workgroups, 52.5 / 55.5; 256 rows 4096 wide 62.7 / 64.2.
inline ProjectSplit project_split(uint32_t rows, uint32_t heads, uint32_t K, uint32_t n_cu) {
  const ProjectSplit whole = {1, 1, false};
  if (rows <= 64 || ((size_t)rows + 127) / 128 * heads > n_cu) return whole;
  ProjectSplit best = whole;
  double best_us = 0.95 * project_tiles_us(whole, rows, heads, K);
  for (uint32_t blocks = 1; blocks <= 2; ++blocks) {
    const uint32_t tiles = (rows + 128 * blocks - 1) / (128 * blocks) * heads;
    for (uint32_t n = blocks == 2 && K / 64 < 96 ? 4 : 3; n <= 8 && n * tiles <= n_cu && 4 * n <= K / 64; ++n) {
      const bool spare = 16 * n * tiles <= 15 * n_cu;
      const ProjectSplit s = {blocks, n, blocks == 1 && spare};
      if (blocks == 2 && !spare) break;
      const double us = project_tiles_us(s, rows, heads, K);
      if (us < best_us) {
        best_us = us;
        best = s;
      }
    }
  }
  return best;
}

// Room for the sums of every call of up to max_rows rows of a matrix (at most 256 tokens x 128 columns a unit).  The
// rows of a 128-token tile have the same tiles, and with them a plan's estimate is a straight line, the steeper the more
// pieces: from row to row pieces only get fewer, and the rows that have as many end where a bisection finds it.
inline size_t project_split_room(uint32_t heads, uint32_t K, uint32_t n_cu, size_t max_rows) {
  size_t most = 0;
  for (size_t first = 65; first <= max_rows && (first + 127) / 128 * heads <= n_cu;) {
    const size_t tile_end = (first + 127) / 128 * 128;
    const uint32_t pieces = project_split((uint32_t)first, heads, K, n_cu).k_split;
    size_t last = tile_end < max_rows ? tile_end : max_rows;
    if (project_split((uint32_t)last, heads, K, n_cu).k_split != pieces) {
      size_t same = first;   // and `last` has fewer
      while (last - same > 1) {
        const size_t mid = (same + last) / 2;
        (project_split((uint32_t)mid, heads, K, n_cu).k_split == pieces ? same : last) = mid;
      }
      last = same;
    }
    const size_t f = split_floats({1, pieces, false}, (uint32_t)last, heads);
    if (f > most) most = f;
    first = last + 1;
  }
  return most;
}

// A handle's one block of device memory: the few-rows kernel's workspace and, behind it, room for shared sums.
// `alloc(bytes)` returns 0 and takes the block; where it does not, whatever the reason, the workspace alone is asked for, and K
// stays whole: *part_floats becomes 0.  Returns alloc's last answer.
template <typename Alloc>
inline int project_block(size_t ws_floats, size_t* part_floats, Alloc alloc) {
  if (*part_floats) {
    if (alloc((ws_floats + *part_floats) * sizeof(float)) == 0) return 0;
    *part_floats = 0;
  }
  return alloc(ws_floats * sizeof(float));
}

}  // namespace proj
}  // namespace ellm
