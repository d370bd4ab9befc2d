// Attention for the shapes the 128-wide 16-bit kernels do not take: any head size up to 256 and
// binary32 storage.  The reference's generic leaf (src/kernel/generic/flash_attention.rs:60-89)
// honours whatever `length` and element type its caller hands it, and its operator test runs in
// f32 (src/compiler/mul/attention.rs:262-330).  Same arguments, masks, position rules and
// log-sum-exp as the other kernels (ellm_attn_run / ellm_attn_run_ragged).  This file: the choice
// between the two kernels, their key splits, and the merge of a chunk's splits.
#include "attn_general.hpp"
#include "chunk_plan.hpp"

namespace ellm {
namespace gen {
namespace {

// Folds the partial rows of a chunk call: G lanes per (query row, four columns) take the row's
// splits in turn and combine through lane exchanges.  A row's live splits are those that start
// before the end of its workgroup's keys; one whose keys are all masked for this row left
// (-inf, 0) and weighs nothing.  Split 0 always holds key 0, so the reference is finite.
template <typename S, bool VEC, int G>
__global__ __launch_bounds__(256) void general_merge_kernel(GeneralArgs p, uint32_t planes, uint32_t pitch,
                                                            uint32_t tile_rows) {
  const uint32_t quads = pitch / 4;
  const size_t items = (size_t)planes * p.rows * quads;
  const size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t sub = gid % G;
  const bool valid = gid / G < items;
  const size_t item = valid ? gid / G : 0;   // idle groups keep their lanes in the exchanges
  const uint32_t dq = item % quads;
  const size_t prow = item / quads;
  const uint32_t r = prow % p.rows, plane = prow / p.rows;
  const uint32_t seq = plane / p.n_kv_heads, kvh = plane % p.n_kv_heads;
  const uint32_t last_row = min(p.rows, (r / tile_rows + 1) * tile_rows) - 1;
  const uint32_t end = start_position(p, seq) + last_row / p.group + 1;
  const uint32_t live = (end + p.split_len - 1) / p.split_len;
  const float* ml = p.part_ml + prow * p.n_split * 2;
  const float* po = p.part_o + prow * p.n_split * pitch + 4 * dq;
  float m = -INFINITY;
  for (uint32_t s = sub; s < live; s += G) m = fmaxf(m, ml[2 * s]);
#pragma unroll
  for (int x = 1; x < G; x <<= 1) m = fmaxf(m, __shfl_xor(m, x));
  float l = 0.0f;
  f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
  for (uint32_t s = sub; s < live; s += G) {
    const float ms = ml[2 * s];
    const float w = (ms == -INFINITY) ? 0.0f : fast_exp2(ms - m);
    l += w * ml[2 * s + 1];
    o += w * *(const f32x4*)(po + (size_t)s * pitch);
  }
#pragma unroll
  for (int x = 1; x < G; x <<= 1) {
    l += __shfl_xor(l, x);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] += __shfl_xor(o[e], x);
  }
  if (!valid || sub != 0) return;
  const size_t row = query_row(p, seq, kvh, r);
  const float inv = 1.0f / l;
  store_out4<S, VEC>(p, row, 4 * dq, f32x4{o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv});
  if (p.lse && dq == 0) p.lse[row] = (m + fast_log2(l)) * kLn2;
}

template <typename S, bool VEC>
hipError_t launch_merge(const GeneralArgs& p, uint32_t planes, uint32_t pitch, hipStream_t stream) {
  const size_t items = (size_t)planes * p.rows * (pitch / 4);
  auto go = [&](auto kernel, size_t lanes) {
    hipLaunchKernelGGL(kernel, dim3((uint32_t)((items * lanes + 255) / 256)), dim3(256), 0, stream, p, planes, pitch,
                       p.tile_rows);
    return hipGetLastError();
  };
  if (p.n_split > 8 && items * 8 <= ((size_t)1 << 21)) return go(general_merge_kernel<S, VEC, 8>, 8);
  return go(general_merge_kernel<S, VEC, 1>, 1);
}

uint32_t element_bytes(int dtype) { return dtype == 2 ? 4 : 2; }

}  // namespace
}  // namespace gen

GeneralWorkspace general_workspace(uint32_t max_interval, uint32_t batch_capacity, uint32_t n_q_heads,
                                   uint32_t n_kv_heads, uint32_t head_size, uint32_t n_cu) {
  GeneralWorkspace w;
  const uint32_t group = n_q_heads / n_kv_heads;
  w.pitch = 32 * (uint32_t)gen::head_blocks(head_size, false);   // (never below the pitch of the vector form)
  size_t rows = decode_workspace(batch_capacity, n_q_heads, n_kv_heads, n_cu).rows;
  const size_t chunk = prefill_workspace_rows(max_interval, batch_capacity, n_q_heads, n_cu);
  if (chunk > rows) rows = chunk;
  const size_t cap = (size_t)512 * n_cu * 128 / w.pitch;         // 68 MB on 256 units
  w.rows = rows < cap ? rows : cap;
  const uint32_t tiles = (group + gen::kGeneralStepRows - 1) / gen::kGeneralStepRows;
  w.counters = (size_t)batch_capacity * n_kv_heads * (tiles > 2 ? tiles : 2);
  return w;
}

hipError_t launch_attn_general(const AttnArgs& a, uint32_t head_size, hipStream_t stream) {
  gen::GeneralArgs p;
  p.q = a.q;
  p.k = a.k;
  p.v = a.v;
  p.out = a.out;
  p.lse = a.lse;
  p.positions = a.positions;
  p.seq_offsets = a.seq_offsets;
  p.seq_caps = a.seq_caps;
  p.kv_stride_seq = a.kv_stride_seq;
  p.kv_stride_head = a.kv_stride_head;
  p.kv_stride_pos = a.kv_stride_pos;
  p.batch_pitch = a.batch_pitch;
  p.n_q_heads = a.n_q_heads;
  p.n_kv_heads = a.n_kv_heads;
  p.group = a.group;
  p.head_size = head_size;
  p.position_index = a.position_index;
  p.interval = a.position_interval;
  const float c = a.scale * kLog2e;
  p.negate_q = c < 0.0f ? 1u : 0u;
  // scale == 0 (uniform attention): a tiny positive c keeps -inf * c == -inf for masked keys
  p.c = c < 0.0f ? -c : c > 0.0f ? c : 1e-37f;
  p.part_o = a.prefill_part_o;
  p.part_ml = a.prefill_part_ml;
  p.counters = a.counters;
  const size_t rows = (size_t)a.position_interval * a.group;
  const size_t planes_s = (size_t)a.batch * a.n_kv_heads;
  if (rows == 0 || planes_s == 0) return hipSuccess;
  if (head_size == 0 || head_size > (uint32_t)gen::kMaxHead || rows > 0x7fffffffu) return hipErrorInvalidValue;
  p.rows = (uint32_t)rows;
  const uint32_t planes = (uint32_t)planes_s;
  const uint32_t es = gen::element_bytes(a.dtype);
  // whole aligned 16-byte pieces: rows and planes of 16-byte multiples (a table of per-sequence
  // offsets lies on the device and may hold anything), 64 rows within a buffer descriptor's reach
  const bool vec = head_size * es % 16 == 0 && p.kv_stride_seq * es % 16 == 0 && p.kv_stride_head * es % 16 == 0 &&
                   p.kv_stride_pos * es % 16 == 0 && p.kv_stride_pos * es <= ((size_t)1 << 25) && !p.seq_offsets;
  const int nb = gen::head_blocks(head_size, vec);
  const uint32_t max_len = a.position_index + a.position_interval;
  const size_t room = p.part_o ? a.prefill_part_rows / ((size_t)planes * rows) : 1;

  // Few query rows per plane: the call is a stream of K and V.  Two workgroups of sixteen rows read a
  // plane twice (the second time from a cache); from 33 rows on the chunk kernel reads it once.
  if (p.interval == 1 || rows <= 2 * gen::kGeneralStepRows) {
    p.row_tiles = (p.rows + gen::kGeneralStepRows - 1) / gen::kGeneralStepRows;
    DecodePlan plan = decode_plan(max_len, planes * p.row_tiles, 1, a.n_cu);
    if (plan.n_split > room) {
      const uint32_t n = room > 1 ? (uint32_t)room : 1;
      plan.split_len = ((max_len + n - 1) / n + 63) / 64 * 64;
      plan.n_split = (max_len + plan.split_len - 1) / plan.split_len;
    }
    p.split_len = plan.split_len;
    p.n_split = plan.n_split;
    if ((size_t)planes * p.row_tiles * p.n_split > 0x7fffffffu) return hipErrorInvalidValue;
    return gen::launch_general_step(p, a.dtype, nb, vec, planes, stream);
  }

  const bool f32 = a.dtype == 2;
  auto tiles_of = [&](size_t n) { return (rows + n - 1) / n; };
  // Key groups put more waves on a row's keys: 64 rows and four groups while all workgroups find a
  // unit of their own (131 tokens on 378, 32 / 8 heads of 64: 15.2 -> 9.7 us), else 128 rows.  With
  // more workgroups than units, heads of 65 to 128 elements keep two small workgroups a unit, whose
  // starts and ends overlap (408 tokens x 4 on 152, 32 / 32 heads of 96: 26 us, 32 with two groups);
  // heads up to 64 leave room for two workgroups of two groups, and wider ones have one wave per SIMD
  // without them.  Up to 128 keys there is nothing to share (21 tokens: 5.8 against 6.2 us).
  p.tile_rows = 128;
  p.key_groups = 1;
  if (max_len > 128) {
    if (gen::chunk_key_groups(f32, nb, 2) > 1 && planes * tiles_of(64) <= a.n_cu) p.tile_rows = 64;
    const bool one_each = planes * tiles_of(p.tile_rows) <= a.n_cu;
    if (one_each || nb <= 2 || nb > 4) p.key_groups = (uint32_t)gen::chunk_key_groups(f32, nb, p.tile_rows / 32);
  }
  p.row_tiles = (uint32_t)tiles_of(p.tile_rows);
  if ((size_t)planes * p.row_tiles > 0x7fffffffu) return hipErrorInvalidValue;
  const uint32_t items = planes * p.row_tiles;
  const uint32_t tiles = (max_len + 63) / 64;
  p.n_split = 1;
  p.split_len = tiles * 64;
  p.turn_at = items <= 2 * a.n_cu && planes <= a.n_cu ? a.n_cu / planes : p.row_tiles;
  // too few workgroups to fill the part: split the key range, in pieces of at least 512 keys or, four
  // waves a workgroup, 256
  const uint32_t slots = (es == 2 && nb <= 4 && p.key_groups == 1 ? 2 : 1) * a.n_cu;
  if (2 * (size_t)items <= slots && tiles >= 8 && room > 1) {
    const double tile_us = (es == 4 ? 1.7 : 0.5) * nb;
    const double split_us = (double)planes * rows * (32 * nb + 2) * 8 / 4e6;
    const KeySplit ks = plan_key_split(tiles, items, slots, p.key_groups > 1 ? 8 : 4, (uint32_t)(room < 4096 ? room : 4096), split_us / tile_us);
    if (ks.n_split > 1) {
      p.n_split = ks.n_split;
      p.split_len = ks.split_tiles * 64;
    }
  }
  const hipError_t e = gen::launch_general_chunk(p, a.dtype, nb, vec, planes, stream);
  if (e != hipSuccess || p.n_split == 1) return e;
  const uint32_t pitch = 32 * (uint32_t)nb;
  if (a.dtype == 0)
    return vec ? gen::launch_merge<F16, true>(p, planes, pitch, stream) : gen::launch_merge<F16, false>(p, planes, pitch, stream);
  if (a.dtype == 1)
    return vec ? gen::launch_merge<BF16, true>(p, planes, pitch, stream) : gen::launch_merge<BF16, false>(p, planes, pitch, stream);
  return vec ? gen::launch_merge<gen::F32, true>(p, planes, pitch, stream) : gen::launch_merge<gen::F32, false>(p, planes, pitch, stream);
}

}  // namespace ellm
