// Causal GQA attention for a chunk of new tokens (position_interval > 1) on
// gfx950 MFMA, FlashAttention-style: K/V tiles staged in LDS, binary32 online
// soft-max in registers, causal tile skipping.
//
// Replaces the (token, sequence, query head) task loop of Attention::run
// (reference: src/compiler/mul/attention.rs:83-153) and its leaf
// flash_attention (src/kernel/x86_64/f16_512/flash_attention.rs:30-92), which
// walks keys 0..=position once per query row.  Same result per row:
// softmax(scale * q.K[0..=position]^T) . V[0..=position].
//
// Formulation (everything transposed so that one lane owns whole query rows):
//   S^T[key][row] = K . Q^T     A = K tile from LDS, B = Q in registers
//   O^T[d][row]  += V^T . P^T   A = V^T from LDS (transposing read), B = P^T in registers
// The C layout of S^T (lane = row, registers = keys) is, up to a fixed
// permutation of keys, the B layout the second MFMA wants; the V^T operand is read with the
// same permutation, so P never leaves the lane that produced it and row max / row sum need one
// or two cross-lane exchanges.
// The tile kernel and the one for few rows run on 16x16x32 instructions, the one for short prompts and the tile
// kernel's form for calls that leave units idle on 32x32x16: on N(0,1) operands a 256 x 256 x 64 loop of the former sustains 1620-1708 TFLOP/s and of the
// latter 1494-1543 (operands from LDS, nothing else in the loop; on zeros 2111 and 2438: fewer joules a
// product, more instructions to issue).  What holds long calls back is the board's power; a short prompt is a
// chain of latencies, 1 to 6 % longer on 16x16x32 (512 tokens, 32 / 32 heads 10.9 -> 11.0 us, 700 tokens, 64 / 8
// heads 23.4 -> 25.0).
//
// A workgroup (8 waves) owns 8 blocks of 32 query rows that all read the same
// K/V plane: up to 8 query heads of one GQA group x consecutive token blocks.
// Stacking the group's heads makes each LDS tile feed 8 times more MFMA work
// and keeps the token span (and so the masked part of the diagonal tile) short.
#include <type_traits>

#include "chunk_plan.hpp"
#include "common.hpp"
#include "kernels.hpp"

namespace ellm {
namespace {

constexpr int kBK = 64;                     // keys per tile
constexpr int kKsPitch = kHeadDim + 8;      // halves per K row (272 B)
constexpr float kRescaleStep = 8.0f;        // log2 units

struct PrefillKernelArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* out;
  float* lse;
  size_t q_token_stride;  // elements between consecutive tokens of Q/O
  size_t kv_stride_seq, kv_stride_head, kv_stride_pos;
  const size_t* seq_offsets;  // per-sequence plane offsets (null: sequence x kv_stride_seq)
  uint32_t batch_pitch;
  uint32_t n_q_heads, n_kv_heads, group;
  uint32_t heads_per_wg;     // query heads stacked in one workgroup
  uint32_t tblocks_per_wg;   // 32-token blocks per workgroup
  uint32_t head_groups;      // group / heads_per_wg
  uint32_t n_wg_tokens;      // workgroups along the token axis
  uint32_t combos;           // batch * kv_heads * head_groups
  uint32_t xcd_mode;         // 1: workgroup id % 8 selects the K/V plane
  uint32_t position_index, interval;
  uint32_t negate_q;         // scale < 0: fold the sign into Q (exact) so that c > 0
  float c;                   // |scale| * log2(e), > 0
  // Key range split over gridDim.y workgroups (few row blocks on a long cache): split s
  // walks tiles [s * split_tiles, (s + 1) * split_tiles) and leaves, per query row, its
  // unnormalised output row, running maximum (log2 units) and denominator in
  // part_o [row][n_split][128] / part_ml [row][n_split][2] for prefill_merge_kernel.
  uint32_t n_split, split_tiles;
  float* part_o;
  float* part_ml;
};

// ---------------------------------------------------------------------------
// Ping-pong kernel: 8 waves, two per SIMD.  Waves 0-3 and waves 4-7 run the
// same per-tile sequence  S^T = K.Q^T -> soft-max -> O^T += V^T.P^T  half a
// step apart: while one group is in its matrix phase (P.V of the previous tile
// and Q.K of the next one, plus moving the following K or V tile into LDS) the
// other group is in its vector phase (mask, exponentials, packing), and
// a workgroup barrier flips the roles.  Two waves that share a SIMD are thus
// never both in the same phase, which is what lets the MFMA pipe and the vector
// ALU work at the same time; left to themselves, two identical workgroups on a
// compute unit run in lockstep and the two pipes take turns instead.
// Rows: wave w owns row block w (32 rows) of 8; all 256 rows read the same K/V
// tiles.  Waves 0-3 stage the K tiles, waves 4-7 the V tiles.
// What bounds it: the board's power on long calls of ordinary operands (1.25-1.30 PFLOP/s at the clock the
// board allows; 1.68 PFLOP/s on K = V = 0), and a phase of ~1500 clocks for 1024 of matrix work: an
// instruction of the vector phase takes 8.2 clocks beside 16x16x32 instructions of the other wave (an
// exponential 15.8; 5.6 and 10.9 beside 32x32x16), staging and operand reads cost the matrix phase 190 clocks each.
// Measured, 32x32x16 instructions with a row maximum every tile -> this form
// (us, in turn on one board): 8192 tokens on 120000, 64 / 8 heads, bf16 27390 -> 26230; 32768 tokens, 32 / 4, f16 7820
// -> 7370; 8000 tokens 469 -> 444; 1624 on 10535 306 -> 291; 255 on 11150 (split) 57.6 -> 55.3; 64 tokens x 24 on 4096
// 120.8 -> 118.1; 412 x 19, 32 / 32 heads 108.4 -> 103.1.  Of that: 16x16x32 alone -1 to +0.5 %, the maximum only where
// it may have to move 3 to 5 %, going first in the vector phase 1 %, the mask from one register 4 % of short
// calls.  Tried and dropped: Q.K on 32x32x16 and P.V on 16x16x32 (eight
// v_permlane16_swap a tile hand P over: 150 clocks of the vector phase), 6 % slower than this; all on 32x32x16
// with the other changes 5 % slower; the barrier ahead of a matrix phase's last operands, so that the other
// group's begins early, 5 %; the tile's stores earlier in the phase 2 %; six or seven operands ahead instead of eight 1 to 3 %.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t uniform64(const void* p) {  // the compiler cannot see that p is wave-uniform
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uint64_t)p);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)p >> 32));
  return ((uint64_t)hi << 32) | (uint64_t)lo;
}
// Bytes a buffer descriptor may cover from byte `off` of a plane whose last visible byte ends at
// `valid`: what is left, capped at the 32 bits the descriptor's size field has (a tile or chunk
// reaches at most 64 rows beyond `off`, far less than that).  Both offsets are 64-bit: a plane
// of the reference's own [position][sequence][kv_head][128] state spans more than 2^32 bytes at
// 33 sequences x 131072 positions.  Scalar arithmetic (the arguments are wave-uniform).
__device__ __forceinline__ uint32_t bytes_left(uint64_t valid, uint64_t off) {
  // (both below 2^63; told apart by the high word, because the scalar unit has no ordered 64-bit compare)
  const uint64_t left = valid - off;
  const int32_t hi = (int32_t)(left >> 32);
  const uint32_t capped = hi < 0 ? 0u : (hi > 0 ? 0xffffffffu : (uint32_t)left);
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)capped);
}
__device__ __forceinline__ uint64_t uniform_u64(uint64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | (uint64_t)lo;
}
typedef __attribute__((address_space(3))) uint16_t LdsHalf;
typedef __attribute__((address_space(3))) u32x4 LdsU32x4;
typedef __attribute__((address_space(3))) u32x2 LdsU32x2;
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 LdsI16x4;
// V rows in LDS: 288 B apart, so that the four rows a 16-lane block of a
// transposing read touches (32 B of each) fall into disjoint banks
constexpr int kVsPitch = kHeadDim + 16;
constexpr int kVsHalves = kBK * kVsPitch;
constexpr int kKsHalves = kBK * kKsPitch;
constexpr int kPpWaves = 8;
constexpr int kPpThreads = kPpWaves * kWave;
constexpr int kLdsAhead = 8;   // LDS operand reads in flight ahead of their MFMA
constexpr int kTileHalves = kBK * kHeadDim;
constexpr int kPpBuffers = 4;                // DIRECT: tiles of K, and of V, in LDS: 128 KB
constexpr int kPpAhead = kPpBuffers - 1;     // DIRECT: tiles requested ahead of the one being multiplied
static_assert(kPpAhead == 3, "s_waitcnt vmcnt literals in prefill_pingpong_kernel");
constexpr int kBufferFlags = 0x00020000;  // raw buffer of 32-bit data, no swizzle (word 3 of the descriptor)

// 16 bytes a lane from memory straight to LDS address lds_at + 16 x lane.  Written as asm: the compiler's
// own form of this load makes it wait for every outstanding one before each later LDS read (it cannot see
// that the two touch different buffers).  M0 carries the address; one wait state between its write and the
// load.  (M0 is a register the compiler reserves and, in the kernel that calls this, never uses itself.)
__device__ __forceinline__ void load_to_lds(const u32x4& rsrc, uint32_t voff, uint32_t lds_at) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :: "s"(lds_at), "v"(voff), "s"(rsrc) : "memory");
}

template <typename T, bool SPLIT, bool DIRECT>
__global__ __launch_bounds__(kPpThreads, 2) void prefill_pingpong_kernel(PrefillKernelArgs p) {
  // Through registers: K tiles [2][64][kVsPitch] then V tiles [3][64][kVsPitch]; V is staged one step
  // earlier than it is read, so that every operand of a matrix step is in LDS a whole
  // phase before the step starts and can be requested ahead of the barrier.  (288-byte rows: the sixteen lanes that
  // a 128-bit read serves at once, rows 0-3 and 12-15 of one piece and 4-11 of its neighbour, meet no bank twice.)
  // DIRECT: K tiles [4][64][128] then V tiles [4][64][128], rows unpadded (a wave instruction delivers four
  // whole rows), their sixteen 16-byte pieces permuted to the same end: piece x of K row r sits at x ^ (r & 15),
  // of V row r at x ^ 2 (r & 7).
  __shared__ __attribute__((aligned(256))) uint16_t smem[DIRECT ? 2 * kPpBuffers * kTileHalves : 5 * kVsHalves];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = tid >> 6;
  const int c16 = lane & 15, g = lane >> 4;
  const int grp = wave >> 2;  // 0: waves 0-3, 1: waves 4-7

  uint32_t combo, order;
  if (p.xcd_mode) {
    const uint32_t xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const uint32_t per = 8 / p.combos;
    combo = xcd % p.combos;
    order = slot * per + xcd / p.combos;
  } else {
    combo = blockIdx.x % p.combos;
    order = blockIdx.x / p.combos;
  }
  if (order >= p.n_wg_tokens) return;
  const uint32_t wg_tok = p.n_wg_tokens - 1 - order;
  const uint32_t seq = combo / (p.n_kv_heads * p.head_groups);
  const uint32_t kvh = (combo / p.head_groups) % p.n_kv_heads;
  const uint32_t hgrp = combo % p.head_groups;
  const uint32_t t_base = wg_tok * 32 * p.tblocks_per_wg;
  const uint32_t S = p.interval, P0 = p.position_index;
  const uint32_t wg_last_tok = min(S, t_base + 32 * p.tblocks_per_wg) - 1;
  const uint32_t kmax = P0 + wg_last_tok;
  const uint32_t all_tiles = kmax / kBK + 1;
  // the tiles of this workgroup: all of them, or its share of the key range
  const uint32_t kt0 = SPLIT ? blockIdx.y * p.split_tiles : 0u;
  if (SPLIT && kt0 >= all_tiles) return;  // (prefill_merge_kernel derives the live splits the same way)
  const uint32_t n_tiles = SPLIT ? min(all_tiles - kt0, p.split_tiles) : all_tiles;

  const uint32_t hg = wave % p.heads_per_wg, tb = wave / p.heads_per_wg;
  const uint32_t head = kvh * p.group + hgrp * p.heads_per_wg + hg;
  const uint32_t tok0 = t_base + 32 * tb;
  // this lane's rows: 16 rb + c16 of the wave's 32 (those past the last token repeat its row and are not stored)
  auto token_of = [&](int rb) { return min(tok0 + 16 * rb + c16, S - 1); };
  const uint32_t first_pos = P0 + min(tok0, S - 1);  // lowest position in this row block

  u32x4 qreg[2][4];   // [row block][32 dims]
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    const uint16_t* qrow =
        p.q + (size_t)token_of(rb) * p.q_token_stride + ((size_t)seq * p.n_q_heads + head) * kHeadDim;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      qreg[rb][s] = load16(qrow + 32 * s + 8 * g);
      if (p.negate_q) qreg[rb][s] ^= 0x80008000u;
    }
  }
  const float c = p.c;

  const size_t plane_at = seq_plane_offset(p.seq_offsets, p.kv_stride_seq, seq) + kvh * p.kv_stride_head;
  const uint16_t* kplane = p.k + plane_at;
  const uint16_t* vplane = p.v + plane_at;

  // staging: the 256 threads of a group move one 64 x 128 tile, four 16-byte pieces
  // each (rows ld_r + 16 i, columns 8 ld_c ..), K and V alike: V sits in LDS row by
  // row as it does in memory and is transposed by the LDS read (ds_read_b64_tr_b16).
  const int st_tid = tid & 255;
  const int ld_r = st_tid >> 4;
  const int ld_c = DIRECT ? (st_tid & 15) ^ (grp ? 2 * (ld_r & 7) : ld_r) : st_tid & 15;
  const uint16_t* plane = grp ? vplane : kplane;                  // wave-uniform
  const uint32_t stride_pos = (uint32_t)p.kv_stride_pos;
  // Tiles are fetched with buffer loads: the descriptor (base of tile kt, bytes
  // left up to the last key this workgroup may see) is scalar arithmetic, the
  // per-lane byte offsets of the four pieces never change, and rows past the
  // last key read as zero instead of needing a clamp: no vector instruction
  // per load.  The plane base goes through readfirstlane because the compiler
  // cannot see that it is wave-uniform.
  // (readfirstlane returns a signed int: the casts keep the low word from sign-extending)
  const uint32_t plane_lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uint64_t)plane);
  const uint32_t plane_hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)plane >> 32));
  const uint64_t plane_u = ((uint64_t)plane_hi << 32) | (uint64_t)plane_lo;
  const uint32_t tile_bytes = kBK * stride_pos * 2;   // (API bound: 64 rows span < 2^32 bytes)
  const uint64_t valid_bytes = uniform_u64(((uint64_t)kmax * stride_pos + kHeadDim) * 2);
  uint32_t piece_off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) piece_off[i] = ((ld_r + 16 * i) * stride_pos + 8 * ld_c) * 2;
  // LDS addresses are kept as byte offsets: the buffers span more than the 64 KB an
  // instruction's immediate offset reaches, so each step forms one base register
  // per tile (step_base) and everything else is an immediate on top of it.
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LdsHalf*)smem;
  auto step_base = [](uint32_t addr) {
    asm volatile("" : "+v"(addr));  // opaque: keeps the compiler from folding the sum another way
    return addr;
  };
  const uint32_t ks_store = lds0 + 2 * (ld_r * kVsPitch + 8 * ld_c);
  const uint32_t vs_store = ks_store + 2 * 2 * kVsHalves;
  u32x4 stg[4];
  auto load_piece = [&](uint32_t kt, int i) {  // kt (relative to kt0) must be wave-uniform to the compiler
    const uint64_t off = (uint64_t)(kt0 + kt) * tile_bytes;
    const uint32_t left = bytes_left(valid_bytes, off);
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc((void*)(plane_u + off), 0, left, kBufferFlags);
    stg[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, piece_off[i], 0, 0);
  };
  // (the group comes as a compile-time constant where the caller runs behind the scalar
  // branch on the group, as the run-time value in the prologue)
  // base: step_base of this lane's place in the destination buffer
  auto store_piece = [&](uint32_t base, int i) {
    *(LdsU32x4*)(base + 2 * 16 * i * kVsPitch) = stg[i];
  };
  auto load_tile = [&](uint32_t kt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) load_piece(kt, i);
  };
  auto store_base = [&](auto group, int buf) {
    return step_base((group ? vs_store : ks_store) + 2 * buf * kVsHalves);
  };
  auto store_tile = [&](int buf) {
    const uint32_t base = store_base(grp, buf);
#pragma unroll
    for (int i = 0; i < 4; ++i) store_piece(base, i);
  };

  const uint32_t wave_lds = lds0 + 4 * 2 * kHeadDim * ((uint32_t)__builtin_amdgcn_readfirstlane(wave) & 3);
  auto load_direct = [&](auto group, uint32_t kt) __attribute__((always_inline)) {   // tile kt into its buffer
    const uint64_t off = (uint64_t)(kt0 + kt) * tile_bytes, at = plane_u + off;
    const u32x4 rsrc = {(uint32_t)at, (uint32_t)(at >> 32) & 0xffffu, bytes_left(valid_bytes, off), (uint32_t)kBufferFlags};
    const uint32_t to = wave_lds + (uint32_t)__builtin_amdgcn_readfirstlane(
                                       (int)(((group ? kPpBuffers : 0) + (kt & (kPpBuffers - 1))) * 2 * kTileHalves));
#pragma unroll
    for (int i = 0; i < 4; ++i) load_to_lds(rsrc, piece_off[i], to + 16 * i * 2 * kHeadDim);
  };

  // per row: minus its reference maximum (log2 units; +inf: no key seen yet), this lane's share of
  // the denominator
  float neg_m[2] = {INFINITY, INFINITY}, l_run[2] = {0.0f, 0.0f};
  f32x4 oacc[8][2];   // [16 dims][row block]
#pragma unroll
  for (int db = 0; db < 8; ++db)
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) oacc[db][rb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 st[4][2];     // [16 keys][row block]
  u32x4 pk[2][2];     // [32 keys][row block]
#pragma unroll
  for (int kc = 0; kc < 2; ++kc)
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) pk[kc][rb] = u32x4{0u, 0u, 0u, 0u};  // P(-1) = 0

  // Every matrix step runs the same straight-line code, the first and the last
  // included: step 0 multiplies P(-1) = 0 by a zeroed "V(-1)" buffer, step n_tiles
  // multiplies Q by whatever finite K tile its buffer still holds and nobody reads
  // the result; tiles past the last one are fetched as zeros (the buffer
  // descriptor has no bytes left) and stored where nothing reads them.
  // prologue: K(0) and V(0) into LDS, K(1) and V(1) on their way into the staging
  // registers, zeros into the V^T buffer that step 0 reads.
  // (DIRECT: V(-1) is buffer 3, and the first kPpAhead tiles are on their way)
  if constexpr (DIRECT) {
    if (grp) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *(LdsU32x4*)(lds0 + 2 * (2 * kPpBuffers - 1) * kTileHalves + st_tid * 16 + i * 4096) = u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int kt = 0; kt < kPpAhead; ++kt) load_direct(grp, kt);
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");   // 4 (kPpAhead - 1): tile 0 is there
  } else {
    if (grp) {
#pragma unroll
      for (int i = 0; i < 4; ++i) stg[i] = u32x4{0u, 0u, 0u, 0u};
      store_tile(2);
    }
    load_tile(0);
    store_tile(0);
    load_tile(1);
  }
  __syncthreads();

  // Matrix step kt = P.V of tile kt-1 and Q.K of tile kt, their MFMAs interleaved
  // (no MFMA waits on the one before it); then the group stores its tile kt+1 (group 0: K, group 1: V)
  // and fetches tile kt+2.  K(kt) sits in buffer kt % 2, V(kt) in buffer kt % 3: V is
  // staged one step before the first step that reads it, so that all operands of
  // a matrix step are in LDS a whole phase before it starts.  Operands come from
  // LDS kLdsAhead reads ahead of the MFMA that consumes them: issued just in
  // time, every operand's MFMAs (32 cycles) would wait out a full LDS round trip
  // (100+ cycles).  The first kLdsAhead are requested before the barrier that
  // opens the step (prefetch_ring), so the round trip overlaps the barrier wait.
  // DIRECT: tile kt of K and of V sits in buffer kt % 4 of its own.  A vector step kt requests tile kt + 3
  // into the buffer of tile kt - 1, whose last reader, matrix step kt (V) or kt - 1 (K) of either group, has
  // ended; matrix step kt + 1 waits for tile kt + 2 at its end, where the barrier shows it to all.
  // A operand of P.V (rows = 16 dims, 32 keys): lane (dim c16, key quarter g) holds keys
  // {4g..4g+3, 16+4g..16+4g+3} of the 32, the order in which the soft-max leaves P in
  // registers.  ds_read_b64_tr_b16 hands lane t of a 16-lane block element
  // (t & 3) of what lanes 4e + (t >> 2), e = 0..3, of that block address: with lane
  // s pointing at key s >> 2, dims 4 (s & 3).. of the 16 dims, lane t ends
  // up with dim t of 4 consecutive keys.  Two such reads (keys +0 and +16) make one operand.
  const uint32_t k_read = lds0 + (DIRECT ? 2 * kHeadDim * c16 + 16 * (g ^ c16) : 2 * (c16 * kVsPitch + 8 * g));
  const int v_row = 4 * g + (c16 >> 2);
  const uint32_t v_read = lds0 + (DIRECT ? 2 * (kPpBuffers * kTileHalves + v_row * kHeadDim) + 32 * (v_row & 7) + 8 * (c16 & 3)
                                         : 2 * (2 * kVsHalves + v_row * kVsPitch + 4 * (c16 & 3)));
  auto mod3 = [](uint32_t x) { return x % 3u; };
  constexpr int kPitch = DIRECT ? kHeadDim : kVsPitch;
  auto k_base = [&](uint32_t kt) __attribute__((always_inline)) {
    return step_base(k_read + (DIRECT ? 2 * (kt & (kPpBuffers - 1)) * kTileHalves : 2 * (kt & 1) * kVsHalves));
  };
  auto v_base = [&](uint32_t kt) __attribute__((always_inline)) {   // V(kt - 1)
    return step_base(v_read + (DIRECT ? 2 * ((kt - 1) & (kPpBuffers - 1)) * kTileHalves : 2 * mod3(kt + 2) * kVsHalves));
  };
  // operand n of the stream of matrix step kt: P.V 0, Q.K 0, P.V 1, Q.K 1, ...
  // (lane part of the address once per step, operand part as a compile-time offset)
  auto stream_operand = [&](uint32_t ks, uint32_t vs, int n) {
    const int i = n >> 1;
    if (n & 1) {  // K: i = 4 s + kb, keys 16 kb.., dims 32 s..
      const int s = i >> 2, kb = i & 3;
      return (u32x4) * (const LdsU32x4*)((DIRECT ? ks ^ (64 * s) : ks + 64 * s) + 2 * 16 * kb * kPitch);
    }
    // V: i = 8 kc + db, keys 32 kc.., dims 16 db..
    const int kc = i >> 3, db = i & 7;
    const uint32_t at = (DIRECT ? vs ^ (32 * db) : vs + 32 * db) + 2 * 32 * kc * kPitch;
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4*)at);
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4*)(at + 2 * 16 * kPitch));
    const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
    return u32x4{l2[0], l2[1], h2[0], h2[1]};
  };
  u32x4 ring[kLdsAhead];
  auto prefetch_ring = [&](uint32_t kt) __attribute__((always_inline)) {
    const uint32_t ks = k_base(kt), vs = v_base(kt);
#pragma unroll
    for (int n = 0; n < kLdsAhead; ++n) ring[n] = stream_operand(ks, vs, n);
  };
  auto matrix_step = [&](auto group, uint32_t kt) __attribute__((always_inline)) {
    __builtin_amdgcn_s_setprio(0);
    const uint32_t ks = k_base(kt), vs = v_base(kt);
    uint32_t store_at = 0;
    if constexpr (!DIRECT) store_at = store_base(group, group ? (int)mod3(kt + 1) : (int)((kt + 1) & 1));
    // staging work is dealt out between the MFMAs, and a full scheduling barrier
    // after every MFMA keeps the compiler from regrouping any of it
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < 32; ++n) {
      const int i = n >> 1;
      const u32x4 a = ring[n % kLdsAhead];
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        if (n & 1)
          st[i & 3][rb] = Mfma<T>::m16x16x32(a, qreg[rb][i >> 2], i < 4 ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : st[i & 3][rb]);
        else
          oacc[i & 7][rb] = Mfma<T>::m16x16x32(a, pk[i >> 3][rb], oacc[i & 7][rb]);
      }
      if (n + kLdsAhead < 32) ring[n % kLdsAhead] = stream_operand(ks, vs, n + kLdsAhead);
      // staging last: the loads issued at the end of the previous matrix step have had
      // almost a whole iteration (~2 us) to arrive before their registers are stored
      if (!DIRECT && n >= 24 && n < 28) store_piece(store_at, n - 24);
      if (!DIRECT && n >= 28 && n < 32) load_piece(kt + 2, n - 28);
      __builtin_amdgcn_sched_barrier(0);
    }
    // the barrier that follows carries no wait of its own: wait here for the LDS stores
    // (DIRECT: for tile kt + 1, behind which one younger one is on its way, and for the operand reads)
    if constexpr (DIRECT)
      asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
    else
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  };

  const int last_key = (int)(P0 + tok0 + c16) - 4 * g;   // relative to the lane's first key of a tile
  // P = exp2(c s + neg) of the tile's scores, packed, and this lane's sums of it
  auto exponentials = [&](const float (&neg)[2], float (&psum)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      psum[rb] = 0.0f;
#pragma unroll
      for (int kc = 0; kc < 2; ++kc)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const f32x4& s4 = st[2 * kc + (w >> 1)][rb];
          const float p0 = fast_exp2(__builtin_fmaf(s4[2 * (w & 1)], c, neg[rb]));
          const float p1 = fast_exp2(__builtin_fmaf(s4[2 * (w & 1) + 1], c, neg[rb]));
          pk[kc][rb][w] = Mfma<T>::pack2(p0, p1);
          psum[rb] += p0 + p1;
        }
    }
  };

  // Vector step kt = soft-max of tile kt: mask on the diagonal, exponentials, packing, row sum; row maximum
  // and rescaling of O^T where they are due.  (Its wave goes first where both waves of a SIMD have something
  // to issue: 0.5 to 1 % on long calls.)
  auto vector_step = [&](auto group, uint32_t kt) __attribute__((always_inline)) {
    if constexpr (DIRECT) load_direct(group, kt + kPpAhead);
    __builtin_amdgcn_s_setprio(2);
    const uint32_t kb = (kt0 + kt) * kBK;
    if (kb + kBK - 1 > first_pos) {  // tile crosses this row block's diagonal
      const int past = last_key - (int)kb;   // row block 0 sees keys 0 .. past of this lane's, row block 1 sixteen more
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int rb = 0; rb < 2; ++rb) st[b][rb][r] = 16 * (b - rb) + r <= past ? st[b][rb][r] : -INFINITY;
    }
    // Exponentials against the reference maximum each row already has: while no lane's sum of them
    // passes kMaxSum, the true maximum is not looked for.  A row without a reference (neg_m = +inf)
    // makes its sums infinite or NaN and so asks for one; so does a score that is not finite.
    float psum[2];
    exponentials(neg_m, psum);
    const uint64_t over[2] = {__ballot(!(psum[0] <= Mfma<T>::kMaxSum)), __ballot(!(psum[1] <= Mfma<T>::kMaxSum))};
    if (over[0] | over[1]) {
      float rmax[2], safe[2];
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        rmax[rb] = st[0][rb][0];
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) rmax[rb] = fmaxf(rmax[rb], st[b][rb][r]);
      }
      max_over_quarters(rmax[0], rmax[1]);
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        // (a row moves by what its own four lanes saw: its bits do not depend on its neighbours)
        const uint64_t any = over[rb] >> c16;
        const bool moves = ((any | any >> 16 | any >> 32 | any >> 48) & 1) != 0;
        const float neg_new = moves ? fminf(neg_m[rb], -(rmax[rb] * c)) : neg_m[rb];   // (+inf while no key of the row is visible)
        safe[rb] = neg_new == INFINITY ? 0.0f : neg_new;
        const float alpha = fast_exp2(safe[rb] - neg_m[rb]);       // (a row's first reference: exp2(-inf) = 0)
        neg_m[rb] = neg_new;
        l_run[rb] *= alpha;
#pragma unroll
        for (int db = 0; db < 8; ++db) oacc[db][rb] *= alpha;
      }
      exponentials(safe, psum);
    }
    l_run[0] += psum[0];
    l_run[1] += psum[1];
  };

  // Phases, one workgroup barrier apart: group 0 runs matrix(0) | vector(0) |
  // matrix(1) | vector(1) ... matrix(n_tiles); group 1 runs the same sequence one
  // phase later.  One loop per group behind a scalar branch (the wave number goes
  // through readfirstlane so that the compiler knows a wave runs one of them
  // only; in a shared loop body it keeps the two groups' values apart and
  // runs out of registers).  A vector step has no LDS traffic, so it leaves the
  // operand requests for the next matrix step in flight across the barrier.
  constexpr std::integral_constant<int, 0> kGroup0;
  constexpr std::integral_constant<int, 1> kGroup1;
  if (__builtin_amdgcn_readfirstlane(grp) == 0) {
    prefetch_ring(0);
    matrix_step(kGroup0, 0);
    __builtin_amdgcn_s_barrier();
    for (uint32_t kt = 0; kt < n_tiles; ++kt) {
      vector_step(kGroup0, kt);
      prefetch_ring(kt + 1);
      __builtin_amdgcn_s_barrier();
      matrix_step(kGroup0, kt + 1);
      __builtin_amdgcn_s_barrier();
    }
  } else {
    prefetch_ring(0);
    __builtin_amdgcn_s_barrier();
    for (uint32_t kt = 0; kt < n_tiles; ++kt) {
      matrix_step(kGroup1, kt);
      __builtin_amdgcn_s_barrier();
      vector_step(kGroup1, kt);
      prefetch_ring(kt + 1);
      __builtin_amdgcn_s_barrier();
    }
    matrix_step(kGroup1, n_tiles);
  }
  if constexpr (DIRECT) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the last requests still write LDS

#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    const float l = sum_over_quarters(l_run[rb]);
    const float m = -neg_m[rb];
    const uint32_t tok = tok0 + 16 * rb + c16;
    if (tok >= S) continue;
    if constexpr (SPLIT) {
      const size_t part = (((size_t)tok * p.batch_pitch + seq) * p.n_q_heads + head) * p.n_split + blockIdx.y;
      float* orow = p.part_o + part * kHeadDim;
#pragma unroll
      for (int db = 0; db < 8; ++db) *(f32x4*)(orow + 16 * db + 4 * g) = oacc[db][rb];
      if (g == 0) *(float2*)(p.part_ml + part * 2) = float2{m, l};
    } else {
      const float inv = 1.0f / l;
      uint16_t* orow =
          p.out + (size_t)tok * p.q_token_stride + ((size_t)seq * p.n_q_heads + head) * kHeadDim;
#pragma unroll
      for (int db = 0; db < 8; ++db) {
        u32x2 w;
        w[0] = Mfma<T>::pack2(oacc[db][rb][0] * inv, oacc[db][rb][1] * inv);
        w[1] = Mfma<T>::pack2(oacc[db][rb][2] * inv, oacc[db][rb][3] * inv);
        *(u32x2*)(orow + 16 * db + 4 * g) = w;
      }
      if (p.lse && g == 0)
        p.lse[((size_t)tok * p.batch_pitch + seq) * p.n_q_heads + head] =
            (m + fast_log2(l)) * kLn2;
    }
  }
}

// ---------------------------------------------------------------------------
// The same kernel on 32x32x16 instructions, tiles through registers and a row maximum every tile: a wave owns its 32
// rows as one block, lane (j, g) row j and half g of the keys.  For walks, whole or in splits, that leave units idle
// (kWideBusy): there the board's power holds nothing back, and a phase is shorter where the matrix instructions leave the
// vector phase of the other wave more of the issue (5.6 clocks an instruction against 8.2).  Phases, buffers, prefetch
// ring and scheduling barriers are those of the kernel above.
// 16x16x32 form / this one (us, in turn on one board): 1030 tokens on 1000, 32 / 4 heads, bf16 52.0 / 48.0, 1200 on 1400
// 64.0 / 58.8, 1480 tokens 41.0 / 37.9; 520 on 2000, 64 / 8, f16 62.2 / 56.8; 120 x 9 on 1200, 32 / 4, bf16 38.4 / 36.0.
// ---------------------------------------------------------------------------
template <typename T, bool SPLIT>
__global__ __launch_bounds__(kPpThreads, 2) void prefill_pingpong32_kernel(PrefillKernelArgs p) {
  // K tiles [2][64][kKsPitch] then V tiles [3][64][kVsPitch]
  __shared__ __attribute__((aligned(16))) uint16_t smem[2 * kKsHalves + 3 * kVsHalves];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = tid >> 6;
  const int j = lane & 31, g = lane >> 5;
  const int grp = wave >> 2;  // 0: waves 0-3, 1: waves 4-7

  uint32_t combo, order;
  if (p.xcd_mode) {
    const uint32_t xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const uint32_t per = 8 / p.combos;
    combo = xcd % p.combos;
    order = slot * per + xcd / p.combos;
  } else {
    combo = blockIdx.x % p.combos;
    order = blockIdx.x / p.combos;
  }
  if (order >= p.n_wg_tokens) return;
  const uint32_t wg_tok = p.n_wg_tokens - 1 - order;
  const uint32_t seq = combo / (p.n_kv_heads * p.head_groups);
  const uint32_t kvh = (combo / p.head_groups) % p.n_kv_heads;
  const uint32_t hgrp = combo % p.head_groups;
  const uint32_t t_base = wg_tok * 32 * p.tblocks_per_wg;
  const uint32_t S = p.interval, P0 = p.position_index;
  const uint32_t wg_last_tok = min(S, t_base + 32 * p.tblocks_per_wg) - 1;
  const uint32_t kmax = P0 + wg_last_tok;
  const uint32_t all_tiles = kmax / kBK + 1;
  const uint32_t kt0 = SPLIT ? blockIdx.y * p.split_tiles : 0u;
  if (SPLIT && kt0 >= all_tiles) return;  // (prefill_merge_kernel derives the live splits the same way)
  const uint32_t n_tiles = SPLIT ? min(all_tiles - kt0, p.split_tiles) : all_tiles;

  const uint32_t hg = wave % p.heads_per_wg, tb = wave / p.heads_per_wg;
  const uint32_t head = kvh * p.group + hgrp * p.heads_per_wg + hg;
  const uint32_t tok0 = t_base + 32 * tb;
  const uint32_t tok = min(tok0 + j, S - 1);
  const bool row_valid = tok0 + j < S;
  const uint32_t rowpos = P0 + tok;
  const uint32_t first_pos = P0 + min(tok0, S - 1);  // lowest position in this row block

  u32x4 qreg[8];
  {
    const uint16_t* qrow =
        p.q + (size_t)tok * p.q_token_stride + ((size_t)seq * p.n_q_heads + head) * kHeadDim;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      qreg[s] = load16(qrow + 16 * s + 8 * g);
      if (p.negate_q) qreg[s] ^= 0x80008000u;
    }
  }
  const float c = p.c;

  const size_t plane_at = seq_plane_offset(p.seq_offsets, p.kv_stride_seq, seq) + kvh * p.kv_stride_head;
  const uint16_t* kplane = p.k + plane_at;
  const uint16_t* vplane = p.v + plane_at;

  const int st_tid = tid & 255;
  const int ld_c = st_tid & 15, ld_r = st_tid >> 4;
  const uint16_t* plane = grp ? vplane : kplane;                  // wave-uniform
  const uint32_t stride_pos = (uint32_t)p.kv_stride_pos;
  const uint64_t plane_u = uniform64(plane);
  const uint32_t tile_bytes = kBK * stride_pos * 2;   // (API bound: 64 rows span < 2^32 bytes)
  const uint64_t valid_bytes = uniform_u64(((uint64_t)kmax * stride_pos + kHeadDim) * 2);
  uint32_t piece_off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) piece_off[i] = ((ld_r + 16 * i) * stride_pos + 8 * ld_c) * 2;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LdsHalf*)smem;
  auto step_base = [](uint32_t addr) {
    asm volatile("" : "+v"(addr));  // opaque: keeps the compiler from folding the sum another way
    return addr;
  };
  const uint32_t ks_store = lds0 + 2 * (ld_r * kKsPitch + 8 * ld_c);
  const uint32_t vs_store = lds0 + 2 * (2 * kKsHalves + ld_r * kVsPitch + 8 * ld_c);
  u32x4 stg[4];
  auto load_piece = [&](uint32_t kt, int i) {  // kt (relative to kt0) must be wave-uniform to the compiler
    const uint64_t off = (uint64_t)(kt0 + kt) * tile_bytes;
    const uint32_t left = bytes_left(valid_bytes, off);
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc((void*)(plane_u + off), 0, left, kBufferFlags);
    stg[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, piece_off[i], 0, 0);
  };
  auto store_piece = [&](auto group, uint32_t base, int i) {
    *(LdsU32x4*)(base + 2 * 16 * i * (group ? kVsPitch : kKsPitch)) = stg[i];
  };
  auto load_tile = [&](uint32_t kt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) load_piece(kt, i);
  };
  auto store_base = [&](auto group, int buf) {
    return step_base(group ? vs_store + 2 * buf * kVsHalves : ks_store + 2 * buf * kKsHalves);
  };
  auto store_tile = [&](int buf) {
    const uint32_t base = store_base(grp, buf);
#pragma unroll
    for (int i = 0; i < 4; ++i) store_piece(grp, base, i);
  };

  float m_run = -INFINITY, l_run = 0.0f;
  f32x16 oacc[4];
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[db][r] = 0.0f;
  f32x16 st[2];
  u32x4 pk[4];
#pragma unroll
  for (int cc = 0; cc < 4; ++cc) pk[cc] = u32x4{0u, 0u, 0u, 0u};  // P(-1) = 0

  if (grp) {
#pragma unroll
    for (int i = 0; i < 4; ++i) stg[i] = u32x4{0u, 0u, 0u, 0u};
    store_tile(2);
  }
  load_tile(0);
  store_tile(0);
  load_tile(1);
  __syncthreads();

  // A operand of P.V (rows = 32 dims, 16 keys): lane (dim j, key half g) holds keys {4g..4g+3, 8+4g..8+4g+3} of the
  // 16, in two transposing reads (keys +0 and +8).
  const uint32_t k_read = lds0 + 2 * (j * kKsPitch + 8 * g);
  const uint32_t v_read = lds0 + 2 * (2 * kKsHalves + (4 * g + ((lane & 15) >> 2)) * kVsPitch +
                                      16 * ((lane >> 4) & 1) + 4 * (lane & 3));
  auto mod3 = [](uint32_t x) { return x % 3u; };
  auto stream_operand = [&](uint32_t ks, uint32_t vs, int n) {
    const int i = n >> 1;
    if (n & 1) {  // K rows: i = 2 s + mb
      const int s = i >> 1, mb = i & 1;
      return (u32x4) * (const LdsU32x4*)(ks + 2 * (32 * mb * kKsPitch + 16 * s));
    }
    // V: i = 4 cc + db, keys 16 cc.., dims 32 db..
    const int cc = i >> 2, db = i & 3;
    const uint32_t at = vs + 2 * (16 * cc * kVsPitch + 32 * db);
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4*)at);
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4*)(at + 2 * 8 * kVsPitch));
    const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
    return u32x4{l2[0], l2[1], h2[0], h2[1]};
  };
  u32x4 ring[kLdsAhead];
  auto prefetch_ring = [&](uint32_t kt) __attribute__((always_inline)) {
    const uint32_t ks = step_base(k_read + 2 * (kt & 1) * kKsHalves);
    const uint32_t vs = step_base(v_read + 2 * mod3(kt + 2) * kVsHalves);  // V(kt-1)
#pragma unroll
    for (int n = 0; n < kLdsAhead; ++n) ring[n] = stream_operand(ks, vs, n);
  };
  auto matrix_step = [&](auto group, uint32_t kt) __attribute__((always_inline)) {
    const uint32_t ks = step_base(k_read + 2 * (kt & 1) * kKsHalves);
    const uint32_t vs = step_base(v_read + 2 * mod3(kt + 2) * kVsHalves);
    const uint32_t store_at = store_base(group, group ? (int)mod3(kt + 1) : (int)((kt + 1) & 1));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < 32; ++n) {
      const int i = n >> 1;
      if (n & 1) {
        const int s = i >> 1, mb = i & 1;
        if (s == 0) {
          f32x16 z;
#pragma unroll
          for (int r = 0; r < 16; ++r) z[r] = 0.0f;
          st[mb] = Mfma<T>::m32x32x16(ring[n % kLdsAhead], qreg[s], z);
        } else {
          st[mb] = Mfma<T>::m32x32x16(ring[n % kLdsAhead], qreg[s], st[mb]);
        }
      } else {
        oacc[i & 3] = Mfma<T>::m32x32x16(ring[n % kLdsAhead], pk[i >> 2], oacc[i & 3]);
      }
      if (n + kLdsAhead < 32) ring[n % kLdsAhead] = stream_operand(ks, vs, n + kLdsAhead);
      if (n >= 24 && n < 28) store_piece(group, store_at, n - 24);
      if (n >= 28 && n < 32) load_piece(kt + 2, n - 28);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  };

  // mask on the diagonal, row maximum, rescaling of O^T where it passed the step, exponentials, packing, row sum
  auto vector_step = [&](uint32_t kt) __attribute__((always_inline)) {
    const uint32_t kb = (kt0 + kt) * kBK;
    if (kb + kBK - 1 > first_pos) {  // tile crosses this row block's diagonal
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const uint32_t key = kb + 32 * mb + 8 * (r >> 2) + 4 * g + (r & 3);
          st[mb][r] = (key <= rowpos) ? st[mb][r] : -INFINITY;
        }
    }
    float rmax = st[0][0];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) rmax = fmaxf(rmax, st[mb][r]);
    rmax = max_with_partner_half(rmax);
    const float tmax = rmax * c;
    const bool grow = tmax > m_run + kRescaleStep;
    if (__any(grow)) {
      const float m_new = grow ? tmax : m_run;
      const float alpha = grow ? fast_exp2(m_run - m_new) : 1.0f;
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < 4; ++db) oacc[db] *= alpha;
    }
    const float neg_m = (m_run == -INFINITY) ? 0.0f : -m_run;
    float psum = 0.0f;
#pragma unroll
    for (int cc = 0; cc < 4; ++cc) {
      const int mb = cc >> 1, r0 = 8 * (cc & 1);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float p0 = fast_exp2(__builtin_fmaf(st[mb][r0 + 2 * w], c, neg_m));
        const float p1 = fast_exp2(__builtin_fmaf(st[mb][r0 + 2 * w + 1], c, neg_m));
        pk[cc][w] = Mfma<T>::pack2(p0, p1);
        psum += p0 + p1;
      }
    }
    l_run += psum;
  };

  constexpr std::integral_constant<int, 0> kGroup0;
  constexpr std::integral_constant<int, 1> kGroup1;
  if (__builtin_amdgcn_readfirstlane(grp) == 0) {
    prefetch_ring(0);
    matrix_step(kGroup0, 0);
    __builtin_amdgcn_s_barrier();
    for (uint32_t kt = 0; kt < n_tiles; ++kt) {
      vector_step(kt);
      prefetch_ring(kt + 1);
      __builtin_amdgcn_s_barrier();
      matrix_step(kGroup0, kt + 1);
      __builtin_amdgcn_s_barrier();
    }
  } else {
    prefetch_ring(0);
    __builtin_amdgcn_s_barrier();
    for (uint32_t kt = 0; kt < n_tiles; ++kt) {
      matrix_step(kGroup1, kt);
      __builtin_amdgcn_s_barrier();
      vector_step(kt);
      prefetch_ring(kt + 1);
      __builtin_amdgcn_s_barrier();
    }
    matrix_step(kGroup1, n_tiles);
  }

  const float l = sum_with_partner_half(l_run);
  if (!row_valid) return;
  if constexpr (SPLIT) {
    const size_t part = (((size_t)tok * p.batch_pitch + seq) * p.n_q_heads + head) * p.n_split + blockIdx.y;
    float* orow = p.part_o + part * kHeadDim;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        *(f32x4*)(orow + 32 * db + 8 * q4 + 4 * g) =
            f32x4{oacc[db][4 * q4], oacc[db][4 * q4 + 1], oacc[db][4 * q4 + 2], oacc[db][4 * q4 + 3]};
    if (g == 0) *(float2*)(p.part_ml + part * 2) = float2{m_run, l};
  } else {
    const float inv = 1.0f / l;
    uint16_t* orow = p.out + (size_t)tok * p.q_token_stride + ((size_t)seq * p.n_q_heads + head) * kHeadDim;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        u32x2 w;
        w[0] = Mfma<T>::pack2(oacc[db][4 * q4] * inv, oacc[db][4 * q4 + 1] * inv);
        w[1] = Mfma<T>::pack2(oacc[db][4 * q4 + 2] * inv, oacc[db][4 * q4 + 3] * inv);
        *(u32x2*)(orow + 32 * db + 8 * q4 + 4 * g) = w;
      }
    if (p.lse && g == 0)
      p.lse[((size_t)tok * p.batch_pitch + seq) * p.n_q_heads + head] = (m_run + fast_log2(l)) * kLn2;
  }
}

// ---------------------------------------------------------------------------
// Few query rows per K/V plane: the short last chunk of a prompt (1 - 63 tokens x 24
// sequences on caches of thousands of tokens in the reference's serving loop,
// src/serving/start copy.rs:71-101).  The ping-pong kernel above is built for tiles that
// are re-used by thousands of rows and sit in L2; here every K/V byte is used once by at
// most 384 rows and the call is a stream from HBM, like the single-token kernel: with few
// rows what matters is bytes in flight, not MFMA issue.  One workgroup = 4, 8 or 12 waves x
// 32 query rows = all (token, head) pairs of one GQA group (row r of the plane = token
// r / group, head r % group), so a plane is read once; the key range is split over gridDim.y
// workgroups (36 KB of LDS each), which leave partial rows for prefill_merge_kernel as the
// split form of the kernel above does.  Chunks of 32 keys go memory -> registers -> LDS
// (double-buffered, one barrier a chunk, the next chunks' loads in flight during the MFMAs of
// this one); operands and soft-max as above.  What bounds it: the stream up to 8 tokens, from 16 on the
// board's power; 32x32x16 instructions with a row maximum every chunk -> 16x16x32 and none (24 sequences on 8191
// keys, 32 / 4 heads, us): 2 tokens 67.3 -> 67.2, 8 72.9 -> 72.3, 13 88.6 -> 84.1, 24 129.4 -> 114.8, 33 161 ->
// 146, 48 195 -> 175; 17 x 5 on 6487 34.3 -> 32.3.  Rows and tokens are worked out again behind the loop: kept
// across it they cost 14 registers, and the form with twelve waves (168) spilled.
// ---------------------------------------------------------------------------
constexpr int kSK = 32;                        // keys per compute step
constexpr int kStStagersMax = 8 * kWave;       // one 16-byte piece of K and of V each moves a whole chunk

// kStDepth = chunks of loads a workgroup keeps in flight, each in its own set of staging
// registers (16 KB a chunk).  The call is bound by bytes in flight: with one chunk a workgroup
// moves 16 KB per memory round trip, whatever else it does.  Two chunks and two workgroups
// per compute unit measured 4-12 % faster than one chunk and three workgroups (24 sequences
// on 8192 keys: 2 tokens 70.1 -> 67.1 us, 8 tokens 80.2 -> 73.0, 16 tokens 94.9 -> 91.2; 16
// tokens x 16 sequences 78.4 -> 68.6); three chunks no better than two.
constexpr int kStDepth = 2;
// WAVES = 4, 8 or 12 waves of 32 query rows each: up to 128, 256 or 384 rows of a plane (16, 32
// or 48 tokens of a sequence with eight heads a group).  Four waves leave room for two
// workgroups a compute unit; eight and twelve fill a unit with one.
template <typename T, int WAVES>
__global__ __launch_bounds__(WAVES * kWave, WAVES == 4 ? 2 : 1) void chunk_stream_kernel(PrefillKernelArgs p) {
  constexpr int DEPTH = kStDepth;
  constexpr int kThreads = WAVES * kWave;
  constexpr int kStagers = kThreads < kStStagersMax ? kThreads : kStStagersMax;  // threads that move K/V
  constexpr int kCK = kSK;                       // keys per staged chunk
  constexpr int kStHalves = kCK * kVsPitch;      // K and V rows alike 288 B apart: operand reads meet no bank twice
  constexpr int kPieces = kCK * 16 / kStagers;   // 16-byte pieces of K (and of V) a staging thread moves per chunk
  constexpr int kPieceRows = kStagers / 16;      // rows between a thread's pieces
  static_assert(kPieces * kStagers == kCK * 16, "the staging threads must tile a chunk");
  __shared__ __attribute__((aligned(16))) uint16_t smem[4 * kStHalves];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c16 = lane & 15, g = lane >> 4;
  const uint32_t seq = blockIdx.x / p.n_kv_heads, kvh = blockIdx.x % p.n_kv_heads;
  const uint32_t S = p.interval, P0 = p.position_index;
  const uint32_t kmax = P0 + S - 1;
  const uint32_t all_tiles = kmax / kBK + 1;
  const uint32_t kt0 = blockIdx.y * p.split_tiles;
  if (kt0 >= all_tiles) return;  // (prefill_merge_kernel derives the live splits the same way)
  const uint32_t n_tiles = min(all_tiles - kt0, p.split_tiles);
  const uint32_t k0 = kt0 * kBK;                                   // first key of this split
  const uint32_t n_chunks = (min(kmax + 1, k0 + n_tiles * kBK) - k0 + kCK - 1) / kCK;

  const uint32_t rows = S * p.group;                                // query rows of the plane, <= 32 WAVES
  // this lane's rows: 16 rb + c16 of the wave's 32 (those past the last one repeat it and are not stored)
  uint32_t first_row = 32 * wave + c16;
  auto row_of = [&](int rb) { return first_row + 16 * rb; };
  auto token_of = [&](int rb) { return min(row_of(rb), rows - 1) / p.group; };
  auto head_of = [&](int rb) { return kvh * p.group + min(row_of(rb), rows - 1) % p.group; };
  uint32_t rowpos[2];
  // positions of the wave's first and last row: chunks past the last are skipped, chunks up to
  // the first need no mask
  const uint32_t wave_first_pos = P0 + min(32u * wave, rows - 1) / p.group;
  const uint32_t wave_last_pos = P0 + min(32u * wave + 31u, rows - 1) / p.group;
  const bool wave_has_rows = 32u * wave < rows;

  u32x4 qreg[2][4];   // [row block][32 dims]
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    const uint32_t tok = token_of(rb);
    rowpos[rb] = P0 + tok;
    const uint16_t* qrow =
        p.q + (size_t)tok * p.q_token_stride + ((size_t)seq * p.n_q_heads + head_of(rb)) * kHeadDim;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      qreg[rb][s] = load16(qrow + 32 * s + 8 * g);
      if (p.negate_q) qreg[rb][s] ^= 0x80008000u;
    }
  }
  const float c = p.c;

  const size_t plane_at = seq_plane_offset(p.seq_offsets, p.kv_stride_seq, seq) + kvh * p.kv_stride_head;
  const uint16_t* kplane = p.k + plane_at;
  const uint16_t* vplane = p.v + plane_at;
  const uint32_t stride_pos = (uint32_t)p.kv_stride_pos;
  // staging: the first 256 or 512 threads move one 32 x 128 chunk of K and one of V, two or one
  // 16-byte pieces of each (rows ld_r + 16 i or row ld_r, columns 8 ld_c ..), through buffer loads
  // whose descriptor ends at the last visible key: rows beyond it read as zeros.
  const bool stager = kThreads == kStagers || __builtin_amdgcn_readfirstlane(wave) < kStagers / kWave;
  const int ld_c = tid & 15, ld_r = (tid >> 4) & (kPieceRows - 1);
  const uint64_t kplane_u = uniform64(kplane), vplane_u = uniform64(vplane);
  const uint32_t chunk_bytes = kCK * stride_pos * 2;
  const uint64_t valid_bytes = uniform_u64(((uint64_t)kmax * stride_pos + kHeadDim) * 2);
  const uint32_t piece_off0 = (ld_r * stride_pos + 8 * ld_c) * 2;
  const uint32_t piece_step = kPieceRows * stride_pos * 2;
  u32x4 stg[DEPTH][2 * kPieces];
  auto load_chunk = [&](uint32_t ck, u32x4 (&st)[2 * kPieces]) {  // ck relative to this split's first chunk; wave-uniform
    if (!stager) return;
    const uint64_t off = (uint64_t)k0 * stride_pos * 2 + (uint64_t)ck * chunk_bytes;
    const uint32_t left = bytes_left(valid_bytes, off);
    const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc((void*)(kplane_u + off), 0, left, kBufferFlags);
    const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc((void*)(vplane_u + off), 0, left, kBufferFlags);
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      st[i] = __builtin_amdgcn_raw_buffer_load_b128(kr, piece_off0 + i * piece_step, 0, 2);   // 2: non-temporal, read once
      st[kPieces + i] = __builtin_amdgcn_raw_buffer_load_b128(vr, piece_off0 + i * piece_step, 0, 2);
    }
  };
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LdsHalf*)smem;
  const uint32_t ks_store = lds0 + 2 * (ld_r * kVsPitch + 8 * ld_c), vs_store = ks_store + 2 * 2 * kStHalves;
  auto store_chunk = [&](uint32_t buf, const u32x4 (&st)[2 * kPieces]) {
    if (!stager) return;
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      *(LdsU32x4*)(ks_store + 2 * (buf * kStHalves + kPieceRows * i * kVsPitch)) = st[i];
      *(LdsU32x4*)(vs_store + 2 * (buf * kStHalves + kPieceRows * i * kVsPitch)) = st[kPieces + i];
    }
  };
  // operand addresses: as in the kernel above (K rows as the A operand of S^T = K.Q^T, V through
  // the transposing read as the A operand of O^T += V^T.P^T, keys in the order P is left in)
  const uint32_t k_read = lds0 + 2 * (c16 * kVsPitch + 8 * g);
  const uint32_t v_read = lds0 + 2 * (2 * kStHalves + (4 * g + (c16 >> 2)) * kVsPitch + 4 * (c16 & 3));

  // per row: minus its reference maximum (+inf: no key seen yet), this lane's share of the denominator
  float neg_m[2] = {INFINITY, INFINITY}, l_run[2] = {0.0f, 0.0f};
  f32x4 oacc[8][2];   // [16 dims][row block]
#pragma unroll
  for (int db = 0; db < 8; ++db)
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) oacc[db][rb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  auto compute = [&](uint32_t ck) __attribute__((always_inline)) {
    const uint32_t kb = k0 + ck * kCK;
    const uint32_t buf = ck & 1;
    if (wave_has_rows && kb <= wave_last_pos) {
      const uint32_t ks = k_read + 2 * buf * kStHalves;
      const uint32_t vs = v_read + 2 * buf * kStHalves;
      f32x4 st[2][2];   // [16 keys][row block]
#pragma unroll
      for (int s = 0; s < 4; ++s) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const u32x4 a = *(const LdsU32x4*)(ks + 2 * (16 * b * kVsPitch + 32 * s));
#pragma unroll
          for (int rb = 0; rb < 2; ++rb)
            st[b][rb] = Mfma<T>::m16x16x32(a, qreg[rb][s], s ? st[b][rb] : f32x4{0.0f, 0.0f, 0.0f, 0.0f});
        }
      }
      if (kb + kSK - 1 > wave_first_pos) {  // chunk crosses the diagonal of some row of this wave
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int rb = 0; rb < 2; ++rb)
              st[b][rb][r] = (kb + 16 * b + 4 * g + r <= rowpos[rb]) ? st[b][rb][r] : -INFINITY;
      }
      u32x4 pk[2];   // [row block]
      float psum[2];
      auto exponentials = [&](const float (&neg)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
          psum[rb] = 0.0f;
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const f32x4& s4 = st[w >> 1][rb];
            const float p0 = fast_exp2(__builtin_fmaf(s4[2 * (w & 1)], c, neg[rb]));
            const float p1 = fast_exp2(__builtin_fmaf(s4[2 * (w & 1) + 1], c, neg[rb]));
            pk[rb][w] = Mfma<T>::pack2(p0, p1);
            psum[rb] += p0 + p1;
          }
        }
      };
      // (the reference maximum moves where a lane's sum passes kMaxSum: as in the kernel above)
      exponentials(neg_m);
      const uint64_t over[2] = {__ballot(!(psum[0] <= Mfma<T>::kMaxSum)), __ballot(!(psum[1] <= Mfma<T>::kMaxSum))};
      if (over[0] | over[1]) {
        float rmax[2], safe[2];
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
          rmax[rb] = st[0][rb][0];
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) rmax[rb] = fmaxf(rmax[rb], st[b][rb][r]);
        }
        max_over_quarters(rmax[0], rmax[1]);
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
          const uint64_t any = over[rb] >> c16;
          const bool moves = ((any | any >> 16 | any >> 32 | any >> 48) & 1) != 0;
          const float neg_new = moves ? fminf(neg_m[rb], -(rmax[rb] * c)) : neg_m[rb];
          safe[rb] = neg_new == INFINITY ? 0.0f : neg_new;
          const float alpha = fast_exp2(safe[rb] - neg_m[rb]);
          neg_m[rb] = neg_new;
          l_run[rb] *= alpha;
#pragma unroll
          for (int db = 0; db < 8; ++db) oacc[db][rb] *= alpha;
        }
        exponentials(safe);
      }
      l_run[0] += psum[0];
      l_run[1] += psum[1];
#pragma unroll
      for (int db = 0; db < 8; ++db) {
        const uint32_t at = vs + 2 * 16 * db;
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4*)at);
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4*)(at + 2 * 16 * kVsPitch));
        const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
          oacc[db][rb] = Mfma<T>::m16x16x32(u32x4{l2[0], l2[1], h2[0], h2[1]}, pk[rb], oacc[db][rb]);
      }
    }
  };
  // chunk n travels through register set n % DEPTH; LDS is double-buffered by chunk parity
#pragma unroll
  for (int d = 0; d < DEPTH; ++d)
    if ((uint32_t)d < n_chunks) load_chunk(d, stg[d]);
  store_chunk(0, stg[0]);
  if ((uint32_t)DEPTH < n_chunks) load_chunk(DEPTH, stg[0]);
  __syncthreads();
  for (uint32_t ck0 = 0; ck0 < n_chunks; ck0 += DEPTH) {
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) {
      const uint32_t ck = ck0 + u;
      if (ck < n_chunks) {  // (uniform over the workgroup: the barrier below is reached by all or none)
        compute(ck);
        if (ck + 1 < n_chunks) {
          const int set = (u + 1) % DEPTH;
          store_chunk((ck & 1) ^ 1, stg[set]);
          if (ck + 1 + DEPTH < n_chunks) load_chunk(ck + 1 + DEPTH, stg[set]);
        }
        __syncthreads();
      }
    }
  }

  asm volatile("" : "+v"(first_row));   // (tokens and heads are worked out again instead of being kept)
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    const float l = sum_over_quarters(l_run[rb]), m = -neg_m[rb];
    if (row_of(rb) >= rows) continue;
    const uint32_t tok = token_of(rb), head = head_of(rb);
    if (p.n_split > 1) {
      const size_t part = (((size_t)tok * p.batch_pitch + seq) * p.n_q_heads + head) * p.n_split + blockIdx.y;
      float* orow = p.part_o + part * kHeadDim;
#pragma unroll
      for (int db = 0; db < 8; ++db) *(f32x4*)(orow + 16 * db + 4 * g) = oacc[db][rb];
      if (g == 0) *(float2*)(p.part_ml + part * 2) = float2{m, l};
    } else {
      const float inv = 1.0f / l;
      uint16_t* orow =
          p.out + (size_t)tok * p.q_token_stride + ((size_t)seq * p.n_q_heads + head) * kHeadDim;
#pragma unroll
      for (int db = 0; db < 8; ++db) {
        u32x2 w;
        w[0] = Mfma<T>::pack2(oacc[db][rb][0] * inv, oacc[db][rb][1] * inv);
        w[1] = Mfma<T>::pack2(oacc[db][rb][2] * inv, oacc[db][rb][3] * inv);
        *(u32x2*)(orow + 16 * db + 4 * g) = w;
      }
      if (p.lse && g == 0) p.lse[((size_t)tok * p.batch_pitch + seq) * p.n_q_heads + head] = (m + fast_log2(l)) * kLn2;
    }
  }
}

// ---------------------------------------------------------------------------
// Short prompts: a call whose whole causal triangle is a few thousand key tiles, where the kernels
// above leave most of the part idle or pay a merge launch.  A workgroup owns 32 WR query rows (row r of
// a plane = token r / group, head r % group); its WK groups of WR waves take the keys in turns of 32,
// each group with tiles of its own in LDS, and meet once at the end: many short workgroups whose
// longest walk is 1 / WK of the row's keys.  What a wider WR buys is K/V traffic: every 32-key tile is
// fetched once per workgroup, and a compute unit takes in 55-60 GB/s, which is what bounds the form
// with one row block (16 KB a step: 15 TB/s over the part).  Two workgroups of four waves a unit.
// Eight waves of keys (1 x 8) only paid on long walks (128 tokens on 4096 keys 28.7 us, split ping-pong
// launch 30), four row blocks (4 x 2) nowhere.  Measured against the kernels above, back to back: 512
// tokens, 32 = 32 heads 20.0 -> 11.3 us; 256 tokens, 32 / 4 heads 14.3 -> 7.3; 1000 tokens 28.9 -> 21.5;
// 16 x 24 on 1024 30 -> 21; 40 x 21 on 1250 42 -> 33; 128 on 1000 24 -> 13; 50 x 4 on 1620 25 -> 17.
// ---------------------------------------------------------------------------
constexpr int kShKsHalves = kSK * kKsPitch, kShVsHalves = kSK * kVsPitch;
constexpr int kShTileHalves = kShKsHalves + kShVsHalves;
constexpr int kShRedPitch = kHeadDim + 4;   // floats per row of the merge

template <typename T, int WR, int WK>
__global__ __launch_bounds__(WR* WK* kWave, 2) void short_prompt_kernel(PrefillKernelArgs p) {
  constexpr int kThreads = WR * WK * kWave;
  constexpr int kBufs = WR == 1 ? 1 : 2;        // one wave: its LDS accesses are in order, no second buffer
  constexpr int kPieces = 8 / WR;               // 16-byte pieces of K (and of V) a thread moves per tile
  constexpr int kRows = 32 * WR;
  __shared__ __attribute__((aligned(16))) uint16_t smem[WK * kBufs * kShTileHalves];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rw = wave % WR, kg = wave / WR;
  const int j = lane & 31, g = lane >> 5;
  // One XCD (workgroup id % 8) takes a plane's row tiles one after the other, longest first, so that
  // they find its K/V rows in that XCD's L2; with fewer planes than XCDs several share one, with
  // counts in between the planes are dealt round.
  const uint32_t planes = p.combos, tiles = p.n_wg_tokens;   // batch * kv_heads
  uint32_t plane, order;
  if (p.xcd_mode == 2) {
    plane = (blockIdx.x & 7) + 8 * ((blockIdx.x >> 3) / tiles);
    order = (blockIdx.x >> 3) % tiles;
  } else if (p.xcd_mode == 1) {
    plane = (blockIdx.x & 7) % planes;
    order = (blockIdx.x >> 3) * (8 / planes) + (blockIdx.x & 7) / planes;
  } else {
    plane = blockIdx.x % planes;
    order = blockIdx.x / planes;
  }
  if (plane >= planes || order >= tiles) return;
  const uint32_t rows = p.interval * p.group;
  const uint32_t row0 = kRows * (tiles - 1 - order);
  const uint32_t seq = plane / p.n_kv_heads, kvh = plane % p.n_kv_heads;
  const uint32_t P0 = p.position_index;
  const uint32_t last_row = min(rows, row0 + kRows) - 1;
  const uint32_t kmax = P0 + last_row / p.group;
  const uint32_t n_chunks = kmax / kSK + 1;
  const uint32_t rc = min(row0 + 32 * rw + j, last_row);
  const uint32_t tok = rc / p.group, head = kvh * p.group + rc % p.group;
  const uint32_t rowpos = P0 + tok;
  const uint32_t wave_row0 = min(row0 + 32u * rw, last_row), wave_row1 = min(wave_row0 + 31u, last_row);
  const uint32_t wave_first_pos = P0 + wave_row0 / p.group, wave_last_pos = P0 + wave_row1 / p.group;

  const size_t plane_at = seq_plane_offset(p.seq_offsets, p.kv_stride_seq, seq) + kvh * p.kv_stride_head;
  const uint64_t kplane_u = uniform64(p.k + plane_at), vplane_u = uniform64(p.v + plane_at);
  const uint32_t stride_pos = (uint32_t)p.kv_stride_pos;
  const uint32_t chunk_bytes = kSK * stride_pos * 2;
  const uint64_t valid_bytes = uniform_u64(((uint64_t)kmax * stride_pos + kHeadDim) * 2);
  const int ld_c = lane & 15, ld_r = 4 * rw + (lane >> 4);   // rows ld_r + 4 WR i of a tile
  const uint32_t piece_off0 = (ld_r * stride_pos + 8 * ld_c) * 2, piece_step = 4 * WR * stride_pos * 2;
  u32x4 kst[kPieces], vst[kPieces];
  auto load_chunk = [&](uint32_t ck) {
    const uint64_t off = (uint64_t)ck * chunk_bytes;
    const uint32_t left = bytes_left(valid_bytes, off);
    const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc((void*)(kplane_u + off), 0, left, kBufferFlags);
    const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc((void*)(vplane_u + off), 0, left, kBufferFlags);
#pragma unroll
    for (int i = 0; i < kPieces; ++i) kst[i] = __builtin_amdgcn_raw_buffer_load_b128(kr, piece_off0 + i * piece_step, 0, 0);
#pragma unroll
    for (int i = 0; i < kPieces; ++i) vst[i] = __builtin_amdgcn_raw_buffer_load_b128(vr, piece_off0 + i * piece_step, 0, 0);
  };
  if ((uint32_t)kg < n_chunks) load_chunk(kg);
  u32x4 qreg[8];
  {
    const uint16_t* qrow = p.q + (size_t)tok * p.q_token_stride + ((size_t)seq * p.n_q_heads + head) * kHeadDim;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      qreg[s] = load16(qrow + 16 * s + 8 * g);
      if (p.negate_q) qreg[s] ^= 0x80008000u;
    }
  }
  const float c = p.c;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LdsHalf*)smem + 2 * kg * kBufs * kShTileHalves;
  const uint32_t ks_store = lds0 + 2 * (ld_r * kKsPitch + 8 * ld_c);
  const uint32_t vs_store = lds0 + 2 * (kShKsHalves + ld_r * kVsPitch + 8 * ld_c);
  auto store_chunk = [&](uint32_t buf) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      *(LdsU32x4*)(ks_store + 2 * (buf * kShTileHalves + 4 * WR * i * kKsPitch)) = kst[i];
      *(LdsU32x4*)(vs_store + 2 * (buf * kShTileHalves + 4 * WR * i * kVsPitch)) = vst[i];
    }
  };
  // operand addresses as in the kernels above
  const uint32_t k_read0 = lds0 + 2 * (j * kKsPitch + 8 * g);
  const uint32_t v_read0 = lds0 + 2 * (kShKsHalves + (4 * g + ((lane & 15) >> 2)) * kVsPitch + 16 * ((lane >> 4) & 1) + 4 * (lane & 3));
  float m_run = -INFINITY, l_run = 0.0f;
  f32x16 oacc[4];
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) oacc[db][e] = 0.0f;

  auto compute = [&](uint32_t ck, uint32_t buf) __attribute__((always_inline)) {
    const uint32_t kb = ck * kSK;
    if (kb > wave_last_pos) return;
    const uint32_t k_read = k_read0 + 2 * buf * kShTileHalves, v_read = v_read0 + 2 * buf * kShTileHalves;
    f32x16 st;
#pragma unroll
    for (int e = 0; e < 16; ++e) st[e] = 0.0f;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const u32x4 a = *(const LdsU32x4*)(k_read + 2 * 16 * s);
      st = Mfma<T>::m32x32x16(a, qreg[s], st);
    }
    if (kb + kSK - 1 > wave_first_pos) {   // chunk crosses the diagonal of some row
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const uint32_t key = kb + 8 * (e >> 2) + 4 * g + (e & 3);
        st[e] = (key <= rowpos) ? st[e] : -INFINITY;
      }
    }
    float rmax = st[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) rmax = fmaxf(rmax, st[e]);
    rmax = max_with_partner_half(rmax);
    const float tmax = rmax * c;
    const bool grow = tmax > m_run + kRescaleStep;
    if (__any(grow)) {
      const float m_new = grow ? tmax : m_run;
      const float alpha = grow ? fast_exp2(m_run - m_new) : 1.0f;
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < 4; ++db) oacc[db] *= alpha;
    }
    const float neg_m = (m_run == -INFINITY) ? 0.0f : -m_run;
    float psum = 0.0f;
    u32x4 pk[2];
#pragma unroll
    for (int cc = 0; cc < 2; ++cc)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float p0 = fast_exp2(__builtin_fmaf(st[8 * cc + 2 * w], c, neg_m));
        const float p1 = fast_exp2(__builtin_fmaf(st[8 * cc + 2 * w + 1], c, neg_m));
        pk[cc][w] = Mfma<T>::pack2(p0, p1);
        psum += p0 + p1;
      }
    l_run += psum;
#pragma unroll
    for (int cc = 0; cc < 2; ++cc)
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const uint32_t at = v_read + 2 * (16 * cc * kVsPitch + 32 * db);
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4*)at);
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4*)(at + 2 * 8 * kVsPitch));
        const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
        oacc[db] = Mfma<T>::m32x32x16(u32x4{l2[0], l2[1], h2[0], h2[1]}, pk[cc], oacc[db]);
      }
  };
  if constexpr (WR == 1) {
    for (uint32_t ck = kg; ck < n_chunks; ck += WK) {
      store_chunk(0);
      if (ck + WK < n_chunks) load_chunk(ck + WK);
      __builtin_amdgcn_wave_barrier();
      compute(ck, 0);
      __builtin_amdgcn_wave_barrier();
    }
  } else {   // every group makes the same number of steps, so that all meet at the barriers
    const uint32_t n_steps = (n_chunks + WK - 1) / WK;
    if ((uint32_t)kg < n_chunks) store_chunk(0);
    if ((uint32_t)kg + WK < n_chunks) load_chunk(kg + WK);
    __syncthreads();
    for (uint32_t step = 0; step < n_steps; ++step) {
      const uint32_t ck = kg + WK * step;
      if (ck < n_chunks) compute(ck, step & 1);
      if (ck + WK < n_chunks) {
        store_chunk((step & 1) ^ 1);
        if (ck + 2 * WK < n_chunks) load_chunk(ck + 2 * WK);
      }
      __syncthreads();
    }
  }
  const float l_wave = sum_with_partner_half(l_run);
  auto store_lse = [&](uint32_t t, uint32_t h, float v) { p.lse[((size_t)t * p.batch_pitch + seq) * p.n_q_heads + h] = v * kLn2; };
  float* red = (float*)smem;
  // the groups' rows meet in LDS: red[group][row][128 sums, maximum, denominator]
  static_assert(WK * kRows * kShRedPitch * 4 <= WK * kBufs * kShTileHalves * 2, "the merge must fit in the staging buffers");
  __syncthreads();
  float* mine = red + (kg * kRows + 32 * rw + j) * kShRedPitch;
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4)
      *(f32x4*)(mine + 32 * db + 8 * q4 + 4 * g) =
          f32x4{oacc[db][4 * q4], oacc[db][4 * q4 + 1], oacc[db][4 * q4 + 2], oacc[db][4 * q4 + 3]};
  if (g == 0) *(f32x2*)(mine + kHeadDim) = f32x2{m_run, l_wave};
  __syncthreads();
  // a thread finishes eight columns of a row, a wave four whole rows at a time
#pragma unroll
  for (int n = 0; n < kRows * 16 / kThreads; ++n) {
    const uint32_t rr = kThreads / 16 * n + (tid >> 4), d8 = tid & 15;
    if (row0 + rr > last_row) continue;
    f32x2 ml[WK];
    float m = -INFINITY;
#pragma unroll
    for (int w = 0; w < WK; ++w) {
      ml[w] = *(const f32x2*)(red + (w * kRows + rr) * kShRedPitch + kHeadDim);
      m = fmaxf(m, ml[w][0]);
    }
    float l = 0.0f;
    f32x4 o[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
    for (int w = 0; w < WK; ++w) {
      const float wgt = fast_exp2(ml[w][0] - m);   // (a group without keys left -inf: weight 0; m is finite, key 0 counts)
      const float* src = red + (w * kRows + rr) * kShRedPitch + 8 * d8;
      l += wgt * ml[w][1];
      o[0] += wgt * *(const f32x4*)src;
      o[1] += wgt * *(const f32x4*)(src + 4);
    }
    const float inv = 1.0f / l;
    const uint32_t t = (row0 + rr) / p.group, h = kvh * p.group + (row0 + rr) % p.group;
    u32x4 w4;
#pragma unroll
    for (int e = 0; e < 4; ++e) w4[e] = Mfma<T>::pack2(o[e >> 1][2 * (e & 1)] * inv, o[e >> 1][2 * (e & 1) + 1] * inv);
    store16(p.out + (size_t)t * p.q_token_stride + ((size_t)seq * p.n_q_heads + h) * kHeadDim + 8 * d8, w4);
    if (p.lse && d8 == 0) store_lse(t, h, m + fast_log2(l));
  }
}

// Folds the partial results of a split launch: G lanes per (query row, four columns) take
// the row's splits in turn and combine through lane exchanges (with hundreds of splits and
// few rows a thread walking them alone would be one long chain of memory round trips).
// A row's live splits are those whose first tile is at or before the last key any row of
// its workgroup sees, as in the kernel above; a split whose keys are all masked for this row
// left (max = -inf, sum = 0) and weighs nothing.  Split 0 always holds key 0, so the maximum
// is finite.
template <typename T, int G, int TURN>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillKernelArgs p, uint32_t batch) {
  const uint32_t quads = kHeadDim / 4;
  const size_t items = (size_t)p.interval * batch * p.n_q_heads * quads;
  const size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t sub = gid % G;
  const bool valid = gid / G < items;
  const size_t item = valid ? gid / G : 0;  // idle groups keep their lanes in the exchanges
  const uint32_t dq = item % quads;
  size_t r = item / quads;
  const uint32_t head = r % p.n_q_heads;
  r /= p.n_q_heads;
  const uint32_t seq = r % batch;
  const uint32_t tok = r / batch;
  const uint32_t wg_tokens = 32 * p.tblocks_per_wg;
  const uint32_t wg_last_tok = min(p.interval, (tok / wg_tokens + 1) * wg_tokens) - 1;
  const uint32_t all_tiles = (p.position_index + wg_last_tok) / kBK + 1;
  const uint32_t live = (all_tiles + p.split_tiles - 1) / p.split_tiles;
  const size_t row = ((size_t)tok * p.batch_pitch + seq) * p.n_q_heads + head;
  float l;
  f32x4 o;
  const float m = fold_splits<G, TURN>(p.part_ml + row * p.n_split * 2, p.part_o + row * p.n_split * kHeadDim + 4 * dq, kHeadDim,
                                 sub, live, p.n_split, l, o);
  if (!valid || sub != 0) return;
  const float inv = 1.0f / l;
  u32x2 w;
  w[0] = Mfma<T>::pack2(o[0] * inv, o[1] * inv);
  w[1] = Mfma<T>::pack2(o[2] * inv, o[3] * inv);
  *(u32x2*)(p.out + (size_t)tok * p.q_token_stride + ((size_t)seq * p.n_q_heads + head) * kHeadDim + 4 * dq) = w;
  if (p.lse && dq == 0) p.lse[row] = (m + fast_log2(l)) * kLn2;
}

template <typename T>
hipError_t launch_chunk(const AttnArgs& a, hipStream_t stream) {
  static_assert(kPingpongRowBlocks == kPpWaves && kChunkTile == kBK, "what the plan is made for");
  ChunkCall call;
  call.p0 = a.position_index;
  call.interval = a.position_interval;
  call.batch = a.batch;
  call.batch_capacity = a.batch_pitch;
  call.n_q_heads = a.n_q_heads;
  call.n_kv_heads = a.n_kv_heads;
  call.n_cu = a.n_cu;
  call.bf16 = a.dtype != 0;
  call.part_rows = a.prefill_part_o ? a.prefill_part_rows : 0;
  const ChunkPlan plan = plan_chunk(call);

  PrefillKernelArgs p;
  p.q = (const uint16_t*)a.q;
  p.k = (const uint16_t*)a.k;
  p.v = (const uint16_t*)a.v;
  p.out = (uint16_t*)a.out;
  p.lse = a.lse;
  p.q_token_stride = (size_t)a.batch_pitch * a.n_q_heads * kHeadDim;
  p.kv_stride_seq = a.kv_stride_seq;
  p.kv_stride_head = a.kv_stride_head;
  p.kv_stride_pos = a.kv_stride_pos;
  p.seq_offsets = a.seq_offsets;
  p.batch_pitch = a.batch_pitch;
  p.n_q_heads = a.n_q_heads;
  p.n_kv_heads = a.n_kv_heads;
  p.group = a.group;
  p.heads_per_wg = plan.heads_per_wg;
  p.tblocks_per_wg = plan.tblocks_per_wg;
  p.head_groups = plan.head_groups;
  p.n_wg_tokens = plan.n_wg_tokens;
  p.combos = plan.combos;
  p.xcd_mode = plan.xcd_mode;
  p.n_split = plan.n_split;
  p.split_tiles = plan.split_tiles;
  p.position_index = a.position_index;
  p.interval = a.position_interval;
  float c = a.scale * kLog2e;
  p.negate_q = c < 0.0f ? 1u : 0u;
  c = c < 0.0f ? -c : c;
  // scale == 0 (uniform attention): a tiny positive c keeps -inf * c == -inf for masked keys
  p.c = c > 0.0f ? c : 1e-37f;
  p.part_o = a.prefill_part_o;
  p.part_ml = a.prefill_part_ml;

  const dim3 grid(plan.n_wg, plan.n_split);
  auto go = [&](auto kernel, uint32_t threads) { hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, stream, p); };
  if (plan.kernel == kChunkShort) {
    if (plan.row_blocks == 2)
      go(short_prompt_kernel<T, 2, 2>, 4 * kWave);
    else
      go(short_prompt_kernel<T, 1, 4>, 4 * kWave);
  } else if (plan.kernel == kChunkStream) {
    if (plan.waves == 4)
      go(chunk_stream_kernel<T, 4>, 4 * kWave);
    else if (plan.waves == 8)
      go(chunk_stream_kernel<T, 8>, 8 * kWave);
    else
      go(chunk_stream_kernel<T, 12>, 12 * kWave);
  } else if (plan.n_split == 1) {
    if (plan.form == kPingpongDirect)
      go(prefill_pingpong_kernel<T, false, true>, kPpThreads);
    else if (plan.form == kPingpongWide)
      go(prefill_pingpong32_kernel<T, false>, kPpThreads);
    else
      go(prefill_pingpong_kernel<T, false, false>, kPpThreads);
  } else if (plan.form == kPingpongWide) {
    go(prefill_pingpong32_kernel<T, true>, kPpThreads);
  } else {
    go(prefill_pingpong_kernel<T, true, false>, kPpThreads);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || plan.n_split == 1) return e;

  const size_t items = (size_t)a.position_interval * a.batch * a.n_q_heads * (kHeadDim / 4);
  auto merge = [&](auto kernel, size_t lanes) {
    hipLaunchKernelGGL(kernel, dim3((uint32_t)((items * lanes + 255) / 256)), dim3(256), 0, stream, p, a.batch);
    return hipGetLastError();
  };
  // Lanes a row's partials are shared by and partials a lane takes at once: eight lanes where there are more than eight
  // and the grid stays small, 64 from 33 on; else one.  One partial a trip to memory / this (us, the call): 189 tokens on 4704,
  // 32 / 4 heads, 10 pieces 37.6 / 30.6 (eight lanes there 36.0); 16 x 4 on 8000, 26 pieces 33.7 / 31.8; 34 x 5 on 28920, 13
  // 129.1 / 125.1; 110 x 2 on 3656, 8 29.5 / 28.6 (eight at once 28.7); 24 x 24 on 8191, 3 115.3 / 115.0.
  if (p.n_split > 8 && items * 8 <= kMergeLanes) {
    if (p.n_split > 32) return merge(prefill_merge_kernel<T, 64, 4>, 64);
    return p.n_split > 16 ? merge(prefill_merge_kernel<T, 8, 4>, 8) : merge(prefill_merge_kernel<T, 8, 2>, 8);
  }
  return p.n_split > 2 ? merge(prefill_merge_kernel<T, 1, 4>, 1) : merge(prefill_merge_kernel<T, 1, 2>, 1);
}

}  // namespace

hipError_t launch_prefill(const AttnArgs& a, hipStream_t stream) {
  if (a.dtype == 0) return launch_chunk<F16>(a, stream);
  return launch_chunk<BF16>(a, stream);
}

}  // namespace ellm
