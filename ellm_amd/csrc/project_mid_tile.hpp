// The tile of the projections: tokens x one or two heads, the body of project_mid_kernel and of
// project_kernel.  C^T = W . X^T on v_mfma_f32_16x16x32, a lane owns tokens; a wave owns one head (eight
// blocks of 16 columns) x 32 MB tokens.  K runs in chunks of 64 (one 128-byte line of every operand row)
// that go from memory straight into LDS, through two to four stages.
// Every shape adds up K in the same order, so an output's bits do not depend on the shape that made it (pieces of K are
// added to each other afterwards, in order: those bits depend on the plan, that is on the sizes, and on whether the handle
// has the room a plan's sums take: one made when memory was out has none and keeps K whole).
//
// What bounds it: on ordinary operands the board's power, and with it the time the matrix pipe idles.
// A 256 x 256 x 64 loop on N(0,1) operands, probe kernels, TFLOP/s: 32x32x16 instructions 1494-1543 without
// staging, 1262 with; 16x16x32 1620-1708 and 1360 (zeros: 2438 / 1961 and 2111 / 1761: fewer joules a product,
// but half the clocks an instruction covers, so a lone wave that waits for LDS starves the pipe and two waves a
// SIMD are needed).
#pragma once

#include "project_epilogue.hpp"

namespace ellm {
namespace proj {

constexpr int kMidKc = 64;                        // K elements per chunk: one 128-byte line per row
constexpr int kMidRowPitch = kMidKc * 2;          // unpadded; pieces permuted
// Forms in use, all with 32 MB tokens a wave: 4 waves x (MB 1) x one head = 128 x 128; 8 x (MB 1) x one head =
// 256 x 128; 8 x (MB 2) x two heads = 256 x 256.  CH 2: a wave owns half of a head's columns (kModePart, whose
// epilogue needs no whole rows): 8 waves x (MB 1) x half a head = 128 x 128, two waves a SIMD.
template <int MB, int WAVES, int HEADS, int CH = 1>
struct MidShape {
  static constexpr int kThreads = 64 * WAVES;
  static constexpr int kTokens = 32 * MB * WAVES / (HEADS * CH);
  static constexpr int kStageBytes = (kTokens + HEADS * kHeadDim) * kMidRowPitch;  // X rows then W rows: 32, 48 or 64 KB
  // Small chunks: three or four stages, chunk c in stage c % kStages, chunk c + kStages - 1 requested early in
  // iteration c.  64 KB chunks (kHalves): five slots of half a chunk, weight rows of chunk c in slot 2 c % 5, token
  // rows in slot (2 c + 1) % 5; when chunk c is read its slots take the token rows of chunk c + 2 and the weight
  // rows of chunk c + 3: the weights come from further away (with two whole stages 1161 rows 8192 -> 8192 took
  // 182 us).
  static constexpr bool kHalves = kStageBytes > 48 * 1024;
  static constexpr int kStages = kStageBytes > 32 * 1024 ? 3 : 4;
  static constexpr int kSlotBytes = kTokens * kMidRowPitch;
  static_assert(!kHalves || kTokens == HEADS * kHeadDim, "slots of equal size");
  static constexpr int kRingBytes = kHalves ? 5 * kSlotBytes : kStages * kStageBytes;
  static constexpr int kLdsBytes = kRingBytes > WAVES * kEpWaveBytes ? kRingBytes : WAVES * kEpWaveBytes;   // (the epilogue reuses it)
  static constexpr int kRowsPerLoad = 8 * WAVES;    // rows one load of every wave moves (1 KB = 8 rows a wave)
  static constexpr int kXLoads = kTokens / kRowsPerLoad, kWLoads = HEADS * kHeadDim / kRowsPerLoad;
  static constexpr int kLoads = kXLoads + kWLoads;  // 1 KB wave loads per chunk and wave
  static constexpr int kXAhead = kHalves ? 2 : kStages - 1;   // chunks requested before the loop
  static constexpr int kWAhead = kHalves ? 3 : kStages - 1;
  // loads a wave may still have outstanding where it waits for its pieces of the next chunk, and before the
  // loop for those of the first one (the literals of mid_tile's s_waitcnt)
  static constexpr int kMayBePending = kHalves ? kWLoads : (kStages - 2) * kLoads;
  static_assert(kMayBePending == (kHalves ? 4 : CH == 2 ? 8 : (WAVES == 8 ? 6 : 16)), "s_waitcnt vmcnt literals in mid_tile");
  static_assert((kXAhead - 1) * kXLoads + (kWAhead - 1) * kWLoads == (kHalves ? 12 : CH == 2 ? 8 : (WAVES == 8 ? 6 : 16)), "s_waitcnt vmcnt literals in mid_tile");
  static_assert(kLdsBytes <= 160 * 1024, "LDS of a compute unit");
};

// The tile of token rows row0.. x heads head0.., by a workgroup of WAVES waves.
template <typename S, int MODE, int MB, int WAVES, int HEADS, int CH = 1>
__device__ __forceinline__ void mid_tile(const ProjectKernelArgs& p, uint32_t row0, uint32_t head0, uint8_t* mid_smem) {
  using M = Mfma<S>;
  using Shape = MidShape<MB, WAVES, HEADS, CH>;
  static_assert(CH == 1 || (MODE == kModePart && HEADS == 1), "half heads");
  constexpr int kLoads = Shape::kLoads;
  constexpr bool kHalves = Shape::kHalves;
  constexpr int kXLoads = Shape::kXLoads, kHeadLoads = Shape::kWLoads / HEADS, TB = 2 * MB;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c16 = lane & 15, g = lane >> 4;
  const int wn = wave % HEADS, wm = wave / (HEADS * CH), half = CH == 2 ? wave % 2 : 0;
  const uint32_t K = p.K;
  // kModePart: piece blockIdx.y of K, as many chunks as the others or one more
  const uint32_t all_chunks = K / kMidKc, first_chunk = MODE == kModePart ? blockIdx.y * all_chunks / p.k_split : 0u;
  const uint32_t n_chunks = MODE == kModePart ? (blockIdx.y + 1) * all_chunks / p.k_split - first_chunk : all_chunks;
  const uint32_t rows_here = min(p.rows - row0, (uint32_t)Shape::kTokens);
  // (descriptors as four plain words: base, base >> 32, bytes, flags; they go into inline asm)
  auto make_rsrc = [](uint64_t base, uint32_t bytes) {
    return u32x4{(uint32_t)base, (uint32_t)(base >> 32) & 0xffffu, bytes, (uint32_t)kBufFlags};
  };
  u32x4 x_rsrc = make_rsrc(uniform64(p.x) + (uint64_t)row0 * K * 2, rows_here * K * 2);
  auto head_rsrc = [&](uint32_t hh) {   // a head past the last one (odd head count) reads zeros
    const uint16_t* base = p.w[0];
    uint32_t hs = hh, bytes = kHeadDim * K * 2;
    if (hh >= p.heads0 + p.heads_kv) {
      base = p.w[2];
      hs = hh - p.heads0 - p.heads_kv;
    } else if (hh >= p.heads0) {
      base = p.w[1];
      hs = hh - p.heads0;
    }
    if (hh >= p.heads0 + 2 * p.heads_kv) {
      base = p.w[0];
      hs = 0;
      bytes = 0;
    }
    return make_rsrc(uniform64(base) + (uint64_t)hs * kHeadDim * K * 2, bytes);
  };
  u32x4 w_rsrc[HEADS];
#pragma unroll
  for (int h = 0; h < HEADS; ++h) w_rsrc[h] = head_rsrc(head0 + h);

  // staging: lane l of a wave instruction delivers its 16 bytes to M0 + 16 l, so a wave fills
  // 1 KB = eight whole rows of a stage per instruction; thread -> row tid / 8 (+ 8 WAVES i: the
  // X rows for i < kXLoads, then the W rows), LDS piece tid % 8.  The permutation of the pieces
  // within a row (piece p of row r sits at p ^ ((r >> 1) & 7): the sixteen lanes that a 128-bit read serves
  // at once meet no bank twice) is applied on the memory side:
  // which piece of the line a lane asks for.  Eight lanes still fetch one whole 128-byte line.
  // Rows past the end of the activations read zeros.
  const uint32_t st_row = tid >> 3, st_piece = (tid & 7) ^ ((tid >> 4) & 7);
  constexpr int kOffsets = kXLoads > kHeadLoads ? kXLoads : kHeadLoads;
  uint32_t src_off[kOffsets];
#pragma unroll
  for (int i = 0; i < kOffsets; ++i) src_off[i] = (st_row + Shape::kRowsPerLoad * i) * K * 2 + st_piece * 16;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)mid_smem;
  const uint32_t st_wave = lds0 + (uint32_t)__builtin_amdgcn_readfirstlane(wave) * 1024;
  // Written as asm: the compiler's own form of this load makes it wait for every outstanding
  // one before each later LDS read (it cannot see that the two touch different stages).  M0
  // carries the LDS address of the wave's 1 KB; one wait state between its write and the load.
  // (M0 is a register the compiler reserves and, in the kernels that call this, never uses itself.)
  auto load_lds = [](const u32x4& rsrc, uint32_t voff, uint32_t soff, uint32_t lds_at) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(lds_at), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
  };
  // A chunk past the last one is requested through descriptors whose size has become zero: no memory
  // access, zeros into a stage nobody reads, and every iteration issues the same loads.
  uint32_t x_to = 0, w_to = 0, x_off = 0, w_off = 0;
  auto aim_x = [&](uint32_t chunk, uint32_t at) __attribute__((always_inline)) {   // what load_piece() takes, and where to
    x_to = st_wave + at;
    x_off = (first_chunk + chunk) * (kMidKc * 2);
    if (chunk >= n_chunks) x_rsrc[2] = 0;
  };
  auto aim_w = [&](uint32_t chunk, uint32_t at) __attribute__((always_inline)) {
    w_to = st_wave + at;
    w_off = (first_chunk + chunk) * (kMidKc * 2);
    if (chunk >= n_chunks) {
#pragma unroll
      for (int h = 0; h < HEADS; ++h) w_rsrc[h][2] = 0;
    }
  };
  auto load_piece = [&](int i) __attribute__((always_inline)) {
    const int w = i - kXLoads;
    if (i < kXLoads)
      load_lds(x_rsrc, src_off[i], x_off, x_to + 1024 * WAVES * i);
    else
      load_lds(w_rsrc[w / kHeadLoads], src_off[w % kHeadLoads], w_off, w_to + 1024 * WAVES * w);
  };
  // where the token and the weight rows of the next chunk lie, given those of one
  constexpr uint32_t kStep = kHalves ? 2 * Shape::kSlotBytes : Shape::kStageBytes;
  constexpr uint32_t kX0 = kHalves ? Shape::kSlotBytes : 0, kW0 = kHalves ? 0 : Shape::kTokens * kMidRowPitch;
  auto next_at = [](uint32_t at) { return at + kStep >= (uint32_t)Shape::kRingBytes ? at + kStep - Shape::kRingBytes : at + kStep; };

  constexpr int kNb = 8 / CH, kOps = 2 * kNb;   // blocks of 16 columns; weight operands a chunk
  f32x4 acc[kNb][TB];  // [16 columns][16 tokens]
#pragma unroll
  for (int nb = 0; nb < kNb; ++nb)
#pragma unroll
    for (int t = 0; t < TB; ++t) acc[nb][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // operand reads: lane (c16, g) takes row c16 of a 16-row block, piece 4 step + g, permuted.  One base
  // register a stage and step for the token rows and one for the weight rows, formed where the stage is
  // entered (opaque, so that every read is an immediate offset on top of it).
  const uint32_t swz = (c16 >> 1) & 7;
  const uint32_t x_row = lds0 + (wm * 32 * MB + c16) * kMidRowPitch;
  const uint32_t w_row = lds0 + (wn * kHeadDim + half * 64 + c16) * kMidRowPitch;
  auto base = [&](uint32_t row, int st, uint32_t stage) __attribute__((always_inline)) {
    uint32_t at = row + ((4 * st + g) ^ swz) * 16 + stage;
    asm volatile("" : "+v"(at));
    return at;
  };
  auto read_block = [](uint32_t at, int block) { return (u32x4) * (const LdsVec4*)(at + 16 * block * kMidRowPitch); };

  // prologue: the first kAhead chunks on their way; chunk 0 has landed in every wave's rows
  // (in the order the loop requests them: weight rows, then token rows of the chunk before in kHalves)
  {
    uint32_t xa = kX0, wa = kW0;
#pragma unroll
    for (int k = 0; k < Shape::kWAhead; ++k) {
      aim_w(k, wa);
      aim_x(k, xa);
      if constexpr (kHalves) {
#pragma unroll
        for (int i = kXLoads; i < kLoads; ++i) load_piece(i);
      }
      if (k < Shape::kXAhead) {
#pragma unroll
        for (int i = 0; i < (kHalves ? kXLoads : kLoads); ++i) load_piece(i);
      }
      xa = next_at(xa);
      wa = next_at(wa);
    }
  }
  // (requested behind the first chunks where registers are left for it, used after the loop: destinations,
  // positions and the first rows of the rotary table or the residual)
  HeadRows<MB> head;
  if constexpr (MB == 1 && MODE != kModePart) head = prepare_head<S, MODE, MB>(p, head0 + wn, row0 + 32 * MB * wm, lane);
  if constexpr (kHalves)
    asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
  else if constexpr (CH == 2)
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  else if constexpr (WAVES == 8)
    asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
  else
    asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
  __syncthreads();

  // One iteration = one chunk = two 32-wide steps = 16 weight operands, each followed by its TB MFMAs.
  // Weight operands are read kRing ahead of their use, token operands during the step before.  The last
  // read of a chunk's stage is that of operand 15, after operand 15 - kRing; two (three) operands later
  // it has returned, the wave waits for its own pieces of the next chunk and meets the others at the
  // iteration's one barrier, and the reads that would have touched the next stage in between are made up.
  // The barrier orders both hazards: the next chunk is complete, and the stage behind it is read.
  constexpr int kRing = CH == 2 ? 4 : TB == 4 ? 6 : 8;
  constexpr int kBarrier = CH == 2 ? 5 : TB == 4 ? 11 : 10;
  static_assert(kBarrier > kOps - 1 - kRing && kBarrier < kOps - 1 && kRing <= kNb && (kHalves || kLoads <= kBarrier), "the barrier stands behind the last read of a stage");
  u32x4 xop[2][TB], wop[kRing];
#pragma unroll
  for (int t = 0; t < TB; ++t) xop[0][t] = read_block(base(x_row, 0, kX0), t);
  uint32_t w_at = base(w_row, 0, kW0);   // step 0 of the present chunk
#pragma unroll
  for (int o = 0; o < kRing; ++o) wop[o] = read_block(w_at, o);
  uint32_t cur_x = kX0, cur_w = kW0;
  uint32_t prev = Shape::kRingBytes - kStep;   // stage of the chunk before (not kHalves)
  // (kRing may not divide 16: the ring index runs on over a period of chunks)
  constexpr int kPeriod = kOps % kRing == 0 ? 1 : 3;
  static_assert(kOps * kPeriod % kRing == 0, "ring position at the start of a period");
  auto chunk_step = [&](auto phase_, uint32_t c) __attribute__((always_inline)) {
    constexpr int at = kOps * decltype(phase_)::value;   // operands before this chunk in its period
    const uint32_t nxt_x = next_at(cur_x), nxt_w = next_at(cur_w);
    if constexpr (kHalves) {
      aim_x(c + 2, cur_w);   // (slot 2 (c + 2) + 1 = 2 c modulo 5)
      aim_w(c + 3, cur_x);
    } else {
      aim_x(c + Shape::kXAhead, prev + kX0);
      aim_w(c + Shape::kWAhead, prev + kW0);
    }
    const uint32_t x1 = base(x_row, 1, cur_x), w1 = base(w_row, 1, cur_w), x0 = base(x_row, 0, nxt_x), w0 = base(w_row, 0, nxt_w);
    __builtin_amdgcn_sched_barrier(0);
    static_for<kOps>([&](auto o_) {
      constexpr int o = decltype(o_)::value;
      constexpr int st = o / kNb, nb = o % kNb;
#pragma unroll
      for (int t = 0; t < TB; ++t) {
        const int tt = (nb & 1) ? TB - 1 - t : t;
        acc[nb][tt] = M::m16x16x32(wop[(at + o) % kRing], xop[st][tt], acc[nb][tt]);
      }
      if constexpr (o + kRing < kOps) wop[(at + o) % kRing] = o + kRing < kNb ? read_block(w_at, o + kRing) : read_block(w1, o + kRing - kNb);
      if constexpr (o < TB) xop[1][o] = read_block(x1, o);
      if constexpr (o == kBarrier) {
        if constexpr (kHalves)
          asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
        else if constexpr (CH == 2)
          asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
        else if constexpr (WAVES == 8)
          asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)" ::: "memory");
        else
          asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
#pragma unroll
        for (int t = 0; t < TB; ++t) xop[0][t] = read_block(x0, t);
#pragma unroll
        for (int k = kOps; k <= o + kRing; ++k) wop[(at + k) % kRing] = read_block(w0, k - kOps);
      }
      if constexpr (o > kBarrier) wop[(at + o) % kRing] = read_block(w0, o + kRing - kOps);
      if constexpr (kHalves) {
        constexpr int kSlots = kOps - 1 - kBarrier, kEach = (kLoads + kSlots - 1) / kSlots;
        if constexpr (o > kBarrier) {
#pragma unroll
          for (int i = 0; i < kEach; ++i)
            if ((o - kBarrier - 1) * kEach + i < kLoads) load_piece((o - kBarrier - 1) * kEach + i);
        }
      } else {
        if constexpr (o < kLoads) load_piece(o);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    prev = cur_x;
    cur_x = nxt_x;
    cur_w = nxt_w;
    w_at = w0;
  };
  if constexpr (kPeriod == 1) {
    for (uint32_t c = 0; c < n_chunks; ++c) chunk_step(std::integral_constant<int, 0>{}, c);
  } else {
    uint32_t c = 0;
    for (; c + 3 <= n_chunks; c += 3) {
      chunk_step(std::integral_constant<int, 0>{}, c);
      chunk_step(std::integral_constant<int, 1>{}, c + 1);
      chunk_step(std::integral_constant<int, 2>{}, c + 2);
    }
    if (c < n_chunks) chunk_step(std::integral_constant<int, 0>{}, c);
    if (c + 1 < n_chunks) chunk_step(std::integral_constant<int, 1>{}, c + 1);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the last (empty) requests still write LDS
  if constexpr (MODE == kModePart) {   // a lane's four columns of its tokens, plain stores: the next launch reads them
    const uint32_t n_cols = (p.heads0 + 2 * p.heads_kv) * kHeadDim;
#pragma unroll
    for (int t = 0; t < TB; ++t) {
      const uint32_t row = row0 + 32 * MB * wm + 16 * t + c16;
      if (row >= p.rows) continue;
      float* to = p.part + ((size_t)blockIdx.y * p.rows + row) * n_cols + (head0 + wn) * kHeadDim + 64 * half + 4 * g;
#pragma unroll
      for (int nb = 0; nb < kNb; ++nb) *(f32x4*)(to + 16 * nb) = acc[nb][t];
    }
    return;
  }
  __syncthreads();
  if constexpr (MB != 1) head = prepare_head<S, MODE, MB>(p, head0 + wn, row0 + 32 * MB * wm, lane);
  if constexpr (MODE != kModePart) finish_head<S, MODE, MB>(p, acc, head, lds0 + wave * kEpWaveBytes, lane);
}

}  // namespace proj
}  // namespace ellm
