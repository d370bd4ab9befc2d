// How the chunk kernels split the key range of a call with too few query rows to fill the
// device (host code, no device types: also compiled by the CPU tests).
//
// A call has `items` independent pieces of work (row blocks of one K/V plane), each a walk
// over `tiles` key tiles.  Splitting every walk into pieces of `split_tiles` tiles (the last
// piece of a walk takes what is left) gives items x n_split workgroups, dispatched in the
// order of their linear id: every item's first piece, then every item's second piece, ...,
// so the short last pieces start last and fill the slots that the long pieces leave free.
// A piece costs its tile count; every split of a walk also costs the write and the read of
// one partial row (128 + 2 floats) per query row, `split_cost` tiles in all.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace ellm {

// Partial rows (128 + 2 floats each) a handle keeps for calls whose key range is split: 256
// splits of every row it can be asked for, at most 512 per compute unit (68 MB on 256 units).
inline size_t prefill_workspace_rows(uint32_t max_interval, uint32_t batch_capacity, uint32_t n_q_heads, uint32_t n_cu) {
  if (max_interval < 2) return 0;  // single-token calls take the other kernel
  const size_t rows = (size_t)max_interval * batch_capacity * n_q_heads;
  const size_t cap = (size_t)512 * n_cu;
  return rows * 256 < cap ? rows * 256 : cap;
}

struct KeySplit {
  uint32_t split_tiles;  // tiles per piece (the last piece of a walk may be shorter)
  uint32_t n_split;      // pieces per walk
};

// Time, in tiles, until the last workgroup ends when items x n_split workgroups of
// split_tiles tiles (the last of each walk `rest` tiles) are dealt in id order to `slots`
// workgroup slots.  The long pieces run in whole rounds; the short ones share what the last,
// part-filled round of long pieces leaves free and whatever becomes free when it ends.
inline uint64_t key_split_makespan(uint32_t items, uint32_t slots, uint32_t split_tiles,
                                   uint32_t n_split, uint32_t rest) {
  const uint64_t longs = (uint64_t)items * (n_split - 1);
  const uint64_t full_rounds = longs / slots;
  const uint32_t in_last = (uint32_t)(longs % slots);  // long pieces of the part-filled round
  const uint64_t t0 = full_rounds * split_tiles;       // that round starts here
  if (in_last == 0) return t0 + (uint64_t)((items + slots - 1) / slots) * rest;
  // shorts first fill the slots - in_last free slots, round after round, until the long
  // pieces of this round end at t0 + split_tiles; what is left then has all slots
  const uint32_t free_slots = slots - in_last;
  const uint64_t rounds_before = rest ? split_tiles / rest : 0;  // whole short rounds that fit
  const uint64_t done_before = rounds_before * free_slots;
  if (done_before >= items) {
    const uint64_t rounds = ((uint64_t)items + free_slots - 1) / free_slots;
    const uint64_t shorts_end = t0 + rounds * rest;
    const uint64_t longs_end = t0 + split_tiles;
    return shorts_end > longs_end ? shorts_end : longs_end;
  }
  const uint64_t left = items - done_before;
  return t0 + split_tiles + (left + slots - 1) / slots * rest;
}

// The split with the lowest estimated time among pieces of at least min_tiles tiles and at
// most max_split pieces a walk.  split_cost: tiles' worth of time that one more piece per
// walk adds for the whole call (partial rows written and read).  Candidates per piece count
// n: equal pieces, and n - 1 long pieces L with a short rest such that r rounds of rests
// take as long as one long piece (L = tiles r / (r (n - 1) + 1), r = 1..4).
inline KeySplit plan_key_split(uint32_t tiles, uint32_t items, uint32_t slots, uint32_t min_tiles,
                               uint32_t max_split, double split_cost) {
  // (the last answer is kept: a serving loop asks the same question launch after launch)
  struct Memo {
    uint32_t tiles, items, slots, min_tiles, max_split;
    double split_cost;
    KeySplit answer;
  };
  static thread_local Memo memo = {0, 0, 0, 0, 0, 0.0, {0, 0}};
  if (memo.tiles == tiles && memo.items == items && memo.slots == slots && memo.min_tiles == min_tiles &&
      memo.max_split == max_split && memo.split_cost == split_cost && memo.answer.n_split)
    return memo.answer;
  KeySplit best = {tiles, 1};
  if (items == 0 || slots == 0 || tiles == 0) return best;
  double best_cost = (double)((items + slots - 1) / slots) * tiles;
  if (min_tiles < 1) min_tiles = 1;
  auto consider = [&](uint32_t len) {
    if (len < min_tiles || len >= tiles) return;
    const uint32_t n = (tiles + len - 1) / len;
    if (n > max_split) return;
    const uint32_t rest = tiles - (n - 1) * len;
    const double cost = (double)key_split_makespan(items, slots, len, n, rest) + n * split_cost;
    if (cost < best_cost) {
      best_cost = cost;
      best = {len, n};
    }
  };
  // more pieces than fill the slots twice over cannot pay
  const uint32_t useful = 2 * ((slots + items - 1) / items) + 2;
  const uint32_t n_max = max_split < useful ? max_split : useful;
  for (uint32_t n = 2; n <= n_max; ++n) {
    consider((tiles + n - 1) / n);
    for (uint32_t r = 1; r <= 4; ++r) {
      const uint32_t den = r * (n - 1) + 1;
      consider((uint32_t)(((uint64_t)tiles * r + den - 1) / den));
    }
  }
  memo = {tiles, items, slots, min_tiles, max_split, split_cost, best};
  return best;
}

// ---- short prompts -------------------------------------------------------------------------
// Estimated time of a chunk call (us, launch included, 256 compute units) through the kernels that
// can take it.  `planes` K/V planes of interval x group query rows each, the first at position p0.
// The constants are fits to back-to-back calls (binary16; 32 / 4, 32 / 32 and 64 / 8 heads).
struct ChunkShape {
  uint32_t p0, interval, group, planes, n_cu;
  double rows() const { return (double)interval * group; }
  double keys() const { return (double)p0 + interval; }
  double stream_us(double tb_s) const { return planes * keys() * 512 / (tb_s * 1e6); }   // every K/V row once
};
inline double whole_up(double x) { return (double)(uint64_t)(x + 0.999999); }

// short_prompt_kernel with wr = 1 (four waves of keys) or 2 (two): workgroup starts and merges plus
// steps of 32 rows x 32 keys, or the longest walk, or the K/V rows from memory.  Estimated (measured):
// one row block wide: 512 tokens x 32 heads 11.0 (10.9) us, 1000 x 1 23.3 (23.3), 300 x 4 16 (18),
// 40 x 8 on 1250 18 (21), 3 x 24 on 300, 32 / 32 heads 29 (23); two wide: 512 tokens, 64 / 8 heads 14.7
// (14.1), 1000 x 1 20.7 (21.5), 600 x 4 31 (29), 40 x 21 on 1250 33 (33).
inline double short_prompt_us(const ChunkShape& c, uint32_t wr) {
  const double wgs = c.planes * whole_up(c.rows() / (32 * wr));
  const double steps = c.planes * whole_up(c.rows() / 32) * ((c.p0 + 0.5 * c.interval) / 32 + 1);
  const double work = (wr == 1 ? 0.0052 * wgs + 0.00078 * steps : 0.0065 * wgs + 0.00075 * steps) * 256 / c.n_cu;
  const double chain = 1.5 + (wr == 1 ? 0.80 : 0.95) * wr * whole_up(c.keys() / 32) / 4;
  const double t = work > chain ? work : chain, stream = c.stream_us(5.0);
  return 5.0 + (t > stream ? t : stream);
}

// The merge launch of a split call and its partial rows, written and read once.
inline double merge_us(const ChunkShape& c, uint32_t n_split) {
  return n_split > 1 ? 4.0 + c.planes * c.rows() * n_split * (128 + 2) * 8 / 5e6 : 0.0;
}

// chunk_stream_kernel: 16 x 24 on 1024 28 (29.5), 40 x 8 on 1250 32 (33.5), 40 x 21 on 1250 44 (42),
// 46 x 11 on 1713, 32 / 32 heads 58 (58), 24 x 7 on 8724, 64 / 8 heads 80 (86).
inline double chunk_stream_us(const ChunkShape& c, uint32_t waves, const KeySplit& ks) {
  const double tile = waves == 4 ? 1.9 : waves == 8 ? 2.0 : 2.5, slots = (waves == 4 ? 2.0 : 1.0) * c.n_cu;
  double tiles = ks.split_tiles * whole_up(c.planes * (double)ks.n_split / slots);   // equal pieces, whole rounds
  if (waves != 4) {                                                                  // pieces dealt over the units
    const double mean = 1.08 * c.planes * whole_up(c.keys() / 64) / slots;
    tiles = mean > ks.split_tiles ? mean : ks.split_tiles;
  }
  const double walk = tiles * tile, stream = c.stream_us(7.0);
  return 5.0 + (walk > stream ? walk : stream) + merge_us(c, ks.n_split);
}

// prefill_pingpong_kernel, `wgs` workgroups of one compute unit each: 128 tokens 11.6 (11.7), 512 19.4 (20),
// 1000 30 (29), 1000 x 4 43 (48); split: 128 on 4096 31 (30).
inline double pingpong_us(const ChunkShape& c, double wgs, const KeySplit& ks) {
  if (ks.n_split > 1) return 7.0 + 1.6 * ks.split_tiles + merge_us(c, ks.n_split);
  const double longest = whole_up(c.keys() / 64), mean = wgs / c.n_cu * ((c.p0 + 0.5 * c.interval) / 64 + 1);
  return 4.5 + 4.5 * whole_up(wgs / c.n_cu) + 1.3 * (longest > mean ? longest : mean);
}

// The row blocks per workgroup (1 or 2) short_prompt_kernel should take a call with, or 0: it does not take
// less than `margin` of another kernel's estimated time (the estimates are no better).  Up to 1920 keys and
// 115 MB of K and V: there the XCDs' L2s hold the planes that are being walked, which the estimate takes for
// granted (261 tokens on 4868 keys: 60 us where it says 42; 150 tokens x 6 on 1750, 32 / 32 heads, 187 MB: 71 us
// where it says 51, and the other kernel takes 67).
constexpr uint32_t kShortPromptKeys = 1920;
constexpr double kShortPromptMb = 115.0;
inline uint32_t short_prompt_wr(const ChunkShape& c, double other_us, double margin = 0.87) {
  if (c.p0 + c.interval > kShortPromptKeys || c.planes * c.keys() * 512e-6 > kShortPromptMb) return 0;
  const double one = short_prompt_us(c, 1), two = short_prompt_us(c, 2);
  if ((one < two ? one : two) > margin * other_us) return 0;
  return one < two ? 1 : 2;
}

// ---- the choice ------------------------------------------------------------------------------
// A chunk call of 128-wide 16-bit heads, the kernel it runs and how the work is cut.
constexpr uint32_t kChunkTile = 64;         // keys per tile of the ping-pong and streaming kernels
constexpr uint32_t kPingpongRowBlocks = 8;  // 32-row blocks of a ping-pong workgroup
// Unsplit ping-pong walks of this many keys and more fetch their tiles straight into LDS, three ahead (through
// registers / straight, us): 8192 tokens on 120000 26230 / 25810, 8000 tokens 444 / 437, 1624 on 10535 291 / 287,
// layer of 64 x 24 on 4096 189 / 181-187, 3140 x 3, 32 / 32 heads 284 / 282; but 412 x 19, 32 / 32 heads, 103 / 108,
// 519 x 3 36 / 38, 120 x 8 on 1400 57 / 59-65; 255 on 11150 in splits 55.3 / 55.3.
constexpr uint32_t kDirectKeys = 64 * kChunkTile;
// Other walks of the ping-pong kernel run on 32x32x16 instructions while the units are busy for at most this share of
// the longest walk or piece (then the board's power does not set the time) and the XCDs' L2s serve K and V.  16x16x32
// / 32x32x16, us:
//   bf16  busy 0.53 (1030 tokens on 1400, 32 / 4 heads) 59.9 / 54.8   0.57 (1536 on 1400) 72.5 / 71.3   0.58 (2048 on 300)
//         61.3 / 60.3   0.64 (2048 on 700) 73.2 / 73.2   0.67 (2048 on 1400) 92.2 / 93.2
//   f16   0.48 (900 tokens, 64 / 8 heads) 29.2 / 27.8   0.53 (600 on 2000) 63.6 / 62.3   0.55 (700 on 1000) 46.2 / 46.1   0.60
//         (768 on 1400) 57.5 / 58.5   0.67 (900 on 2000) 82.4 / 85.4
//   split: 2000 / 3000 / 4000 tokens, 8 / 1 heads, f16 32.5 / 31.3, 45.0 / 42.3, 61.0 / 57.1; 0.59 (300 on 2000,
//         32 / 4) 31.0 / 30.0   0.86 (300 on 3000) 32.6 / 33.1
//   K and V of 70 MB (250 x 5 on 600, 32 / 32 heads, f16) 34.2 / 37.0; of 49 MB (64 x 19 on 1200, bf16) 37.6 / 36.0; of 41 MB
//         (64 x 19 on 1000, f16) 33.9 / 34.5
constexpr double kWideBusy = 0.6, kWideBusyF16 = 0.55;   // (bfloat16 and splits; unsplit binary16)
constexpr double kWideMbBf16 = 56.0, kWideMbF16 = 32.0;

struct ChunkCall {
  uint32_t p0, interval;                    // positions p0 .. p0 + interval - 1
  uint32_t batch, batch_capacity, n_q_heads, n_kv_heads, n_cu;
  size_t part_rows;                         // partial rows the workspace holds (0: none)
  bool bf16;                                // storage: bfloat16, else binary16
};

enum ChunkKernel { kChunkStream, kChunkPingpong, kChunkShort };
// Forms of the ping-pong kernel: 16x16x32 instructions with tiles through registers or straight into LDS;
// 32x32x16 instructions
enum PingpongForm { kPingpongRegisters, kPingpongDirect, kPingpongWide };

struct ChunkPlan {
  ChunkKernel kernel;
  uint32_t waves;                           // streaming kernel: 4, 8 or 12
  uint32_t row_blocks;                      // short-prompt kernel: 32-row blocks a workgroup, 1 or 2
  PingpongForm form;                        // ping-pong kernel
  uint32_t n_split, split_tiles;            // key range of a plane, in tiles (one split: split_tiles may be 0)
  // ping-pong workgroup: heads_per_wg heads of a group x tblocks_per_wg blocks of 32 tokens
  uint32_t heads_per_wg, tblocks_per_wg, head_groups;
  uint32_t combos, n_wg_tokens;             // independent walks x workgroups along their rows
  uint32_t xcd_mode;                        // how workgroup ids map to those (see the kernels)
  uint32_t n_wg;                            // workgroups of the launch, per split
};

inline uint32_t gcd_u32(uint32_t a, uint32_t b) {
  while (b) {
    const uint32_t t = a % b;
    a = b;
    b = t;
  }
  return a;
}

// Row tiles and workgroup ids of short_prompt_kernel.
inline void plan_short_prompt(const ChunkShape& shape, uint32_t wr, ChunkPlan* p) {
  const uint32_t planes = shape.planes, wg_rows = 32 * wr;
  p->kernel = kChunkShort;
  p->row_blocks = wr;
  p->n_split = 1;
  p->combos = planes;
  p->n_wg_tokens = (uint32_t)(((size_t)shape.interval * shape.group + wg_rows - 1) / wg_rows);
  // Planes that are no multiple of the XCDs, or that together overflow their L2s, go to one XCD each
  // (40 tokens x 21 sequences on 1250, 84 planes: 55.7 -> 39.9 us); else all planes advance together,
  // longest rows first over the whole call (512 tokens x 32 heads: 10.8 against 12.8 us).
  const double xcd_mb = planes / 8.0 * shape.keys() * 512e-6;
  p->xcd_mode = planes <= 8 && 8 % planes == 0 ? 1 : planes >= 32 && (planes % 8 || xcd_mb > 8.0) ? 2 : 0;
  p->n_wg = planes * p->n_wg_tokens;
  if (p->xcd_mode == 1) p->n_wg = 8 * ((p->n_wg_tokens + 8 / planes - 1) / (8 / planes));
  if (p->xcd_mode == 2) p->n_wg = (planes + 7) / 8 * 8 * p->n_wg_tokens;
}

inline ChunkPlan plan_chunk(const ChunkCall& c) {
  ChunkPlan p = {};
  const uint32_t group = c.n_q_heads / c.n_kv_heads, planes = c.batch * c.n_kv_heads;
  const ChunkShape shape = {c.p0, c.interval, group, planes, c.n_cu};
  p.heads_per_wg = gcd_u32(group, kPingpongRowBlocks);
  p.tblocks_per_wg = kPingpongRowBlocks / p.heads_per_wg;
  p.head_groups = group / p.heads_per_wg;
  const uint32_t wg_tokens = 32 * p.tblocks_per_wg;
  p.n_wg_tokens = (c.interval + wg_tokens - 1) / wg_tokens;
  p.combos = planes * p.head_groups;
  p.xcd_mode = (p.combos <= 8 && 8 % p.combos == 0) ? 1 : 0;

  // Few query rows per plane on a cache long enough to be worth streaming: one workgroup
  // covers all rows of a GQA group, the key range is split until there are two
  // workgroups per compute unit (splits of at least 256 keys), as far as the workspace holds
  // the partial rows.
  const uint32_t all_tiles = (c.p0 + c.interval - 1) / kChunkTile + 1;
  const size_t all_rows = (size_t)c.interval * c.batch_capacity * c.n_q_heads;
  const size_t plane_rows = (size_t)c.interval * group;
  const size_t room = c.part_rows ? c.part_rows / all_rows : 1;
  const uint32_t max_split = (uint32_t)(room < 4096 ? room : 4096);
  // what one more partial row per query row costs: written and read once, at about 4 TB/s
  const double split_us = (double)c.interval * c.batch * c.n_q_heads * (128 + 2) * 8 / 4e6;
  if (plane_rows <= 384 && all_tiles >= 8) {
    // workgroups of four waves: two per compute unit (with one chunk in flight three were
    // better); of eight or twelve waves: one.  Pieces of at least four tiles.
    p.waves = plane_rows <= 128 ? 4 : plane_rows <= 256 ? 8 : 12;
    const uint32_t slots = (p.waves == 4 ? 2 : 1) * c.n_cu;
    // a workgroup's time per tile (us, measured on 24 sequences x 8192 keys)
    const double tile_us = p.waves == 8 ? 2.0 : 2.5;
    if (p.waves == 4) {
      // Two workgroups share a compute unit's throughput, so a slot that opens early is not
      // spare capacity: equal pieces, never more workgroups than slots (24 sequences on 8192
      // keys, 2 / 8 tokens: 67.6 / 73.1 us; as 5 pieces of 25 tiles and one of 4: 70.1 / 78.9)
      uint32_t want = slots / planes;
      if (want > max_split) want = max_split;
      if (want > all_tiles / 4) want = all_tiles / 4;
      if (want < 1) want = 1;
      p.split_tiles = (all_tiles + want - 1) / want;
      p.n_split = (all_tiles + p.split_tiles - 1) / p.split_tiles;
    } else {
      const KeySplit ks = plan_key_split(all_tiles, planes, slots, 4, max_split, split_us / tile_us);
      p.split_tiles = ks.split_tiles;
      p.n_split = ks.n_split;
    }
    // enough workgroups to be worth it (a lone sequence with one split would leave the part idle)
    if ((size_t)planes * p.n_split * 2 >= c.n_cu || planes * p.n_split >= p.combos * p.n_wg_tokens) {
      if (const uint32_t wr = short_prompt_wr(shape, chunk_stream_us(shape, p.waves, {p.split_tiles, p.n_split}))) {
        plan_short_prompt(shape, wr, &p);
        return p;
      }
      p.kernel = kChunkStream;
      p.tblocks_per_wg = (c.interval + 31) / 32;  // (the merge derives every row's live splits from the chunk's last token)
      p.n_wg = planes;
      return p;
    }
  }

  p.kernel = kChunkPingpong;
  if (p.xcd_mode) {
    const uint32_t per = 8 / p.combos;
    p.n_wg = 8 * ((p.n_wg_tokens + per - 1) / per);
  } else {
    p.n_wg = p.combos * p.n_wg_tokens;
  }
  // Few row blocks on a long cache: split the key range over more workgroups, as far as the
  // workspace holds the partial rows (plan_key_split weighs the longest chain of pieces a
  // compute unit runs against the partial rows every piece adds).
  p.n_split = 1;
  p.split_tiles = 0;
  const uint32_t base = p.combos * p.n_wg_tokens;
  // This search only while the unsplit launch leaves at least half of the compute units idle: the more of them are
  // busy, the less the board's power leaves for the others, and the partial rows are added (64 tokens x 24 sequences
  // on 8192 keys, 192 workgroups: 229 us unsplit, 235 us as pieces of 97 + 32 tiles on all 256 units).
  if (c.part_rows && 2 * base <= c.n_cu && all_tiles >= 16) {
    // pieces of at least eight tiles (each pays the pipeline's first and last step); 1.9 us a
    // tile and workgroup (measured, 64 tokens x 24 sequences on 8192 keys)
    const KeySplit ks = plan_key_split(all_tiles, base, c.n_cu, 8, max_split, split_us / 1.9);
    if (ks.n_split > 1) {
      p.split_tiles = ks.split_tiles;
      p.n_split = ks.n_split;
    }
  }
  // More than half of the units, but not most of them: two pieces a walk, sized for how the hardware deals them.  A
  // launch fills its shader engines (groups of eight units) in turn, so with m long first pieces on each the
  // second ones run on the other 8 - m units, in r = m / (8 - m) rounds, and should take 1 / r of a first one.
  // (168 workgroups, m = 6, cut for r = 2 as the count of all free units has it: 281 us against 278 unsplit.)
  // A tile takes 1.35 us, 1.56 with all units at work; K and V, which unsplit workgroups read in step, cost a split
  // call their bytes at 12 TB/s.  Unsplit / split (us): 32 / 4 heads, bf16, 1030 tokens on 4100 113.6 / 99.9, on 12000 270
  // / 226, 1167 on 12000 273 / 243, 1344 on 4100 119.7 / 113.3, 1536 on 4100 128.9 / 124.6, on 12000 312 / 300; 600 on
  // 12000, 64 / 8 heads 262 / 237; 1089 on 4100, 32 / 32 heads 114.3 / 104.7; 64 x 18 on 8192, f16 190 / 184; 5000 tokens,
  // 8 / 1 heads 108 / 88.  Left whole: 64 x 18 on 4096 95.6 / 99.0, 660 on 4100, 64 / 8 heads 109 / 111.
  if (c.part_rows && 2 * base > c.n_cu && 4 * base <= 3 * c.n_cu && max_split >= 2) {
    const uint32_t m = (8 * base + c.n_cu - 1) / c.n_cu, r = (m + (8 - m) - 1) / (8 - m);   // m: 5 or 6
    const uint32_t len = (all_tiles * r + r) / (r + 1);
    const double mean = (c.p0 + 0.5 * c.interval) / kChunkTile + 1;
    const double chain = 1.35 * len, work = 1.56 * base * mean / c.n_cu;
    const double split = (chain > work ? chain : work) + merge_us(shape, 2) + shape.stream_us(12.0);
    if (split < 0.98 * 1.35 * all_tiles) {
      p.split_tiles = len;
      p.n_split = 2;
    }
  }
  // (beyond 1536 keys pieces of a split walk take less than the estimate: 300 tokens x 2 on 1500, 32 / 4 heads, 34 us
  // against 38 in the short-prompt kernel)
  const double margin = all_tiles > 24 ? 0.82 : 0.87;
  if (const uint32_t wr = short_prompt_wr(shape, pingpong_us(shape, base, {p.split_tiles, p.n_split}), margin))
    plan_short_prompt(shape, wr, &p);
  if (p.kernel == kChunkPingpong) {
    const uint32_t longest = p.n_split > 1 ? p.split_tiles : all_tiles;
    const double busy = base * ((c.p0 + 0.5 * c.interval) / kChunkTile + 0.5) / ((double)c.n_cu * longest);
    if (p.n_split == 1 && c.p0 + c.interval >= kDirectKeys)
      p.form = kPingpongDirect;
    else if (base <= c.n_cu && busy <= (c.bf16 || p.n_split > 1 ? kWideBusy : kWideBusyF16) &&
             planes * shape.keys() * 512e-6 <= (c.bf16 ? kWideMbBf16 : kWideMbF16))
      p.form = kPingpongWide;
  }
  return p;
}

}  // namespace ellm
