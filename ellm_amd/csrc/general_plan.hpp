// Which kernel a call with heads other than 128 wide, or in binary32, runs, and how it cuts the work
// (host code, no device types: also compiled by the CPU tests).
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "chunk_plan.hpp"
#include "decode_plan.hpp"

namespace ellm {
namespace gen {

constexpr uint32_t kGeneralStepRows = 16;   // query rows of a workgroup of the step kernel
constexpr uint32_t kRowTurn = 16;           // keys a workgroup of the row kernel takes together

// Blocks of 32 elements the matrix kernels pad a head to: 1, 2, 3, 4, 6 or 8 (2, 4 or 8 for rows that are
// not made of whole aligned 16-byte pieces).
inline int head_blocks(uint32_t head_size, bool vec) {
  const int n = (int)((head_size + 31) / 32);
  if (!vec) return n <= 2 ? 2 : n <= 4 ? 4 : 8;
  return n <= 4 ? n : n <= 6 ? 6 : 8;
}

// Key groups of a chunk kernel's workgroup of `row_blocks` x 32 query rows: as many as its registers (a
// wave's queries, accumulators and scores) and LDS (two steps of K and V a group) allow.
constexpr int chunk_key_groups(bool f32, int nb, int row_blocks) {
  if (f32) return 1;
  if (row_blocks == 4) return nb <= 6 ? 2 : 1;
  return nb <= 4 ? 4 : 1;
}

// Workspace of an operator: partial rows (pitch floats each, then 2 of maximum and sum) and arrival counters.
struct GeneralWorkspace {
  size_t rows, counters;
  uint32_t pitch;
};
inline GeneralWorkspace general_workspace(uint32_t max_interval, uint32_t batch_capacity, uint32_t n_q_heads,
                                          uint32_t n_kv_heads, uint32_t head_size, uint32_t n_cu) {
  GeneralWorkspace w;
  const uint32_t group = n_q_heads / n_kv_heads;
  w.pitch = 32 * (uint32_t)head_blocks(head_size, false);   // (never below the pitch of the vector form)
  size_t rows = decode_workspace(batch_capacity, n_q_heads, n_kv_heads, n_cu).rows;
  const size_t chunk = prefill_workspace_rows(max_interval, batch_capacity, n_q_heads, n_cu);
  if (chunk > rows) rows = chunk;
  const size_t cap = (size_t)512 * n_cu * 128 / w.pitch;         // 68 MB on 256 units
  w.rows = rows < cap ? rows : cap;
  const uint32_t tiles = (group + kGeneralStepRows - 1) / kGeneralStepRows;
  w.counters = (size_t)batch_capacity * n_kv_heads * (tiles > 2 ? tiles : 2);
  return w;
}

struct GeneralCall {
  uint32_t planes;      // K/V planes: sequences x key-value heads
  uint32_t group;       // query heads of a plane
  uint32_t interval;    // query positions
  uint32_t max_len;     // keys of the last of them
  uint32_t n_cu;
  uint32_t head_size;
  bool f32, vec;        // binary32 storage; rows of whole aligned 16-byte pieces
  size_t room;          // partial rows the workspace holds, per query row of the call
  size_t rows() const { return (size_t)interval * group; }   // query rows of a plane
};

enum GeneralKernel { kGeneralRows, kGeneralStep, kGeneralChunk };

struct GeneralPlan {
  GeneralKernel kernel;
  int nb;                                                  // matrix kernels: padded head blocks
  uint32_t row_tiles, n_split, split_len;
  uint32_t tile_rows, key_groups, turn_at;                 // chunk kernel
  bool max_first;                                          // ... its form that looks for the row maximum every step
};

// Estimated times (us, 256 units) of a call, fitted to graph replays of calls of 4 to 32 heads; measured ones in
// brackets are row / matrix kernel.
//
// Row kernel: one workgroup per query row, a chain of turns of 16 keys.  Binary32, heads of 64: 1 turn 3.9, 2 5.3,
// 4 8.0, 25 40; heads of 256 4.3, 5.7, 8.6, 45; binary16, heads of 64 / 256: 1 turn 4.2 / 6.0, 25 45 / 84.
// Beyond about a thousand rows it is the turns of all rows that count (9600 rows x 10 turns 106 us).
inline double general_rows_us(const GeneralCall& c) {
  const double quarter = (c.head_size + 63) / 64;          // elements a lane holds
  const double turn = c.f32 ? 1.27 + 0.09 * quarter : 1.25 + 0.47 * quarter;
  const double row_turn = (c.f32 ? 1.1e-3 + 1e-4 * quarter : 1.05e-3 + 2.7e-4 * quarter) * 256 / c.n_cu;
  const double longest = whole_up(c.max_len / (double)kRowTurn);
  const double mean = (c.max_len - 0.5 * (c.interval - 1)) / kRowTurn + 0.5;
  const double chain = turn * longest, all = row_turn * c.planes * c.rows() * mean;
  // (many sequences: the rows of one workgroup after another share nothing in the caches)
  const double apart = c.interval == 1 ? 0.9e-3 * quarter * c.planes * c.group * 256 / c.n_cu : 0.0;
  return 2.6 + (chain > all ? chain : all) + apart;
}

// Step kernel: a launch, a request's way through the registers, and requests after the first.
inline double general_step_us(const GeneralCall& c, const GeneralPlan& p) {
  double first = c.f32 ? (p.nb <= 4 ? 4.75 + 0.22 * p.nb : 4.6 + 0.5 * p.nb) : 4.3 + 0.08 * p.nb;
  if (!c.vec) first += c.f32 ? (p.nb <= 4 ? 1.4 : 4.6) : 0.9 + 0.12 * p.nb;
  if (c.interval > 1) first += 0.9;
  const double kb = p.nb * (c.f32 ? 128 : 64) / 16384.0 * (c.max_len < p.split_len ? c.max_len : p.split_len);   // requests of 16 KB,
  const double rounds = whole_up(c.planes * (double)p.row_tiles * p.n_split / ((c.f32 && p.nb > 4 ? 1.0 : 2.0) * c.n_cu));   // four at a time
  return first + (p.n_split > 1 ? 2.0 : 0.0) + (rounds - 1) * (first - 1.0) + rounds * 0.6 * (kb > 4 ? kb / 4 - 1 : 0.0);
}

// Chunk kernel: steps of 32 keys, the longest walk or all of them over the units.
inline double general_chunk_us(const GeneralCall& c, const GeneralPlan& p) {
  const double step = c.f32 ? (p.nb <= 4 ? 1.45 : 1.65) * p.nb * (c.vec ? 1.0 : 1.15) : (c.vec ? 0.25 : 0.4) * p.nb / p.key_groups;
  const double walk = whole_up((c.max_len < p.split_len ? c.max_len : p.split_len) / 32.0);
  const double rounds = whole_up(c.planes * (double)p.row_tiles * p.n_split / c.n_cu);
  const double mean = (c.max_len - 0.5 * (c.interval - 1)) / c.max_len;
  const double work = rounds > 1 ? (1 + (rounds - 1) * mean) * walk : walk;
  return (c.f32 ? 3.8 : 4.5 + 0.2 * p.nb + (c.vec ? 0.0 : 0.4 * p.nb)) + step * work + (p.n_split > 1 ? 6.0 : 0.0);
}

// Whether the chunk kernel looks for a row's maximum every step (16-bit heads; see its compute()): with heads above 128
// always; with one key group and heads up to 64, whose walks are two steps, too (128 tokens x 40, 32 / 32 heads of 32: 16.5
// us, else 17.7, for the registers it takes); with heads of 65 to 96 and one key group, whose other form has registers for two workgroups a unit
// instead of three, where the third is worth more than the maxima.  That is from three workgroups a unit on
// (us, every step / only where it may have to move, heads of 80 and 96: 700 tokens x 4, 32 / 32 heads 32.0 / 36.4, 300 x 12
// 31.8 / 37.8, 2048 x 4 174 / 180), and from two on unless what the first two leave are short walks: those of
// the shortest rows, at most a third of the longest walk or, with few row tiles a plane, a fifth (1400 x 2, 32 / 8 heads
// 50.3 / 45.5, 1500 x 2, 32 / 4 56.9 / 51.2, 700 x 3, 32 / 32 28.9 / 27.8; but 300 x 7, 32 / 32 20.0 / 24.3, 500 x 5 on 300
// 42.0 / 51.3).  Up to two a unit: 1600 tokens, 32 / 8 51.2 / 47.5.
inline bool chunk_max_first(const GeneralCall& c, const GeneralPlan& p) {
  if (c.f32 || p.nb > 4 || (p.nb <= 2 && p.key_groups == 1)) return true;
  const size_t workgroups = (size_t)c.planes * p.row_tiles * p.n_split, pair = 2 * (size_t)c.n_cu;
  if (p.nb != 3 || p.key_groups != 1 || workgroups <= pair) return false;
  if (workgroups >= 3 * (size_t)c.n_cu) return true;
  const size_t left = p.row_tiles - pair / c.planes;          // row tiles of a plane behind the first two a unit
  const double longest = c.max_len, tail = c.max_len - c.interval + (double)left * p.tile_rows / c.group;
  return tail * (p.row_tiles >= 16 ? 3 : 5) > longest;
}

// The matrix kernel of a call and its cut.
inline GeneralPlan general_matrix_plan(const GeneralCall& c) {
  GeneralPlan p = {};
  const size_t rows = c.rows();
  p.nb = head_blocks(c.head_size, c.vec);
  p.tile_rows = p.key_groups = p.turn_at = 0;
  // Few query rows per plane: the call is a stream of K and V.  Two workgroups of sixteen rows read a
  // plane twice (the second time from a cache); from 33 rows on the chunk kernel reads it once.
  if (c.interval == 1 || rows <= 2 * kGeneralStepRows) {
    p.kernel = kGeneralStep;
    p.row_tiles = (uint32_t)((rows + kGeneralStepRows - 1) / kGeneralStepRows);
    DecodePlan plan = decode_plan(c.max_len, c.planes * p.row_tiles, 1, c.n_cu);
    if (plan.n_split > c.room) {
      const uint32_t n = c.room > 1 ? (uint32_t)c.room : 1;
      plan.split_len = ((c.max_len + n - 1) / n + 63) / 64 * 64;
      plan.n_split = (c.max_len + plan.split_len - 1) / plan.split_len;
    }
    p.split_len = plan.split_len;
    p.n_split = plan.n_split;
    return p;
  }
  p.kernel = kGeneralChunk;
  auto tiles_of = [&](size_t n) { return (rows + n - 1) / n; };
  // Key groups put more waves on a row's keys: 64 rows and four groups while all workgroups find a
  // unit of their own (131 tokens on 378, 32 / 8 heads of 64: 15.2 -> 9.7 us), else 128 rows.  With
  // more workgroups than units, heads of 65 to 128 elements keep two small workgroups a unit, whose
  // starts and ends overlap (408 tokens x 4 on 152, 32 / 32 heads of 96: 26 us, 32 with two groups);
  // heads up to 64 leave room for two workgroups of two groups, and wider ones have one wave per SIMD
  // without them.  Up to 128 keys there is nothing to share (21 tokens: 5.8 against 6.2 us).
  p.tile_rows = 128;
  p.key_groups = 1;
  if (c.max_len > 128) {
    if (chunk_key_groups(c.f32, p.nb, 2) > 1 && c.planes * tiles_of(64) <= c.n_cu) p.tile_rows = 64;
    const bool one_each = c.planes * tiles_of(p.tile_rows) <= c.n_cu;
    if (one_each || p.nb <= 2 || p.nb > 4) p.key_groups = (uint32_t)chunk_key_groups(c.f32, p.nb, p.tile_rows / 32);
  }
  p.row_tiles = (uint32_t)tiles_of(p.tile_rows);
  const uint32_t items = c.planes * p.row_tiles;
  const uint32_t tiles = (c.max_len + 63) / 64;
  p.n_split = 1;
  p.split_len = tiles * 64;
  p.turn_at = items <= 2 * c.n_cu && c.planes <= c.n_cu ? c.n_cu / c.planes : p.row_tiles;
  // too few workgroups to fill the part: split the key range, in pieces of at least 512 keys or, four
  // waves a workgroup, 256
  const uint32_t slots = (!c.f32 && p.nb <= 4 && p.key_groups == 1 ? 2 : 1) * c.n_cu;
  if (2 * (size_t)items <= slots && tiles >= 8 && c.room > 1) {
    const double tile_us = (c.f32 ? 1.7 : 0.5) * p.nb;
    const double split_us = (double)c.planes * rows * (32 * p.nb + 2) * 8 / 4e6;
    const KeySplit ks = plan_key_split(tiles, items, slots, p.key_groups > 1 ? 8 : 4,
                                       (uint32_t)(c.room < 4096 ? c.room : 4096), split_us / tile_us);
    if (ks.n_split > 1) {
      p.n_split = ks.n_split;
      p.split_len = ks.split_tiles * 64;
    }
  }
  p.max_first = chunk_max_first(c, p);
  return p;
}

// The row kernel where its estimate is below the matrix kernel's: up to 16 keys (4.2 against 4.5 us and
// more, heads of 64), short binary32 prompts (64 tokens, 32 / 32 heads of 128: 11 against 17 us, 128 tokens 27
// against 31), and wide heads in binary32 or of no whole pieces on few rows (300 tokens on 100, 4 / 4 heads of
// 256 in binary32: 45 against 180 us).
inline GeneralPlan general_plan(const GeneralCall& c) {
  GeneralPlan p = general_matrix_plan(c);
  const double matrix = p.kernel == kGeneralStep ? general_step_us(c, p) : general_chunk_us(c, p);
  if (c.planes * c.rows() <= 0x7fffffffu && general_rows_us(c) < matrix) {
    p.kernel = kGeneralRows;
    p.n_split = 1;
  }
  return p;
}

}  // namespace gen
}  // namespace ellm
