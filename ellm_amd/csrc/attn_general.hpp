// Shared parts of the attention kernels for shapes other than 128-wide 16-bit heads: any head
// size up to 256 and binary32 storage (general_plan.hpp: which kernel, what cut; attn_general.hip:
// launches, merge and the row kernel; attn_general_chunk.hip: many query rows per K/V plane;
// attn_general_step.hip: few).
#pragma once

#include <type_traits>

#include "common.hpp"
#include "general_plan.hpp"
#include "kernels.hpp"

namespace ellm {
namespace gen {

constexpr int kMaxHead = 256;

struct F32 {};   // binary32 storage

// What a storage type is to the kernels: its element, how many make a 16-byte piece, and the
// exponent shift the soft-max weights carry on their way through the second product (binary16
// weights keep 2^-24 at the small end: moved up, weights down to 2^-31 of the largest count).
template <typename S>
struct Store;
template <>
struct Store<F16> {
  typedef uint16_t E;
  static constexpr int kPiece = 8;
  static constexpr float kShift = 7.0f;
  static constexpr uint32_t kExpMask = 0x7c007c00u;
};
template <>
struct Store<BF16> {
  typedef uint16_t E;
  static constexpr int kPiece = 8;
  static constexpr float kShift = 0.0f;
  static constexpr uint32_t kExpMask = 0x7f807f80u;
};
template <>
struct Store<F32> {
  typedef float E;
  static constexpr int kPiece = 4;
  static constexpr float kShift = 0.0f;
  static constexpr uint32_t kExpMask = 0x7f800000u;
};

template <typename S>
__device__ __forceinline__ float load_elem(const typename Store<S>::E* p) {
  if constexpr (std::is_same<S, F32>::value) return *p;
  else return Mfma<S>::to_float(*p);
}
template <typename S>
__device__ __forceinline__ void store_elem(typename Store<S>::E* p, float v) {
  if constexpr (std::is_same<S, F32>::value) *p = v;
  else *p = (uint16_t)(Mfma<S>::pack2(v, 0.0f) & 0xffffu);
}

struct GeneralArgs {
  const void* q;
  const void* k;
  const void* v;
  void* out;
  float* lse;
  const uint32_t* positions;     // single-token calls only
  const size_t* seq_offsets;
  const uint32_t* seq_caps;
  size_t kv_stride_seq, kv_stride_head, kv_stride_pos;
  uint32_t batch_pitch, n_q_heads, n_kv_heads, group, head_size;
  uint32_t position_index;       // first query's position, or the bound of the per-sequence positions
  uint32_t interval;
  uint32_t rows;                 // query rows of a plane: interval x group; row r = token r / group, head r % group
  uint32_t negate_q;             // scale < 0: the sign is folded into the query rows so that c > 0
  float c;                       // |scale| x log2(e), > 0
  float scale;
  // Key range split over workgroups: n_split pieces of split_len keys.  Partial row of plane row
  // r and split s: (plane x rows + r) x n_split + s of part_o [..][pitch] (weighted sums) and
  // part_ml [..][2] (reference exponent in log2 units, denominator).
  uint32_t n_split, split_len;
  uint32_t row_tiles;            // workgroups along the rows of a plane
  uint32_t tile_rows;            // query rows of a workgroup of the chunk kernel (64 or 128)
  uint32_t turn_at;              // ... and the row tile of the launch (longest first) from which the order turns
  uint32_t key_groups;           // groups of waves that share the keys of those rows
  uint32_t max_first;            // (host) which form of the chunk kernel: GeneralPlan
  float* part_o;
  float* part_ml;
  uint32_t* counters;            // arrivals per (plane, row tile); zero between launches
};

// Position of a plane's query row; for calls with per-sequence positions and capacities too.
__device__ __forceinline__ uint32_t start_position(const GeneralArgs& p, uint32_t seq) {
  uint32_t pos = p.position_index;
  if (p.positions) pos = min(p.positions[seq], p.position_index);
  if (p.seq_caps) pos = min(pos, p.seq_caps[seq] - 1);   // (shared ranges fit every sequence: checked on the host)
  return pos;
}

// Element offset of query row r of a plane in q / out (x head_size) and in lse.
__device__ __forceinline__ size_t query_row(const GeneralArgs& p, uint32_t seq, uint32_t kvh, uint32_t r) {
  return ((size_t)(r / p.group) * p.batch_pitch + seq) * p.n_q_heads + kvh * p.group + r % p.group;
}

__device__ __forceinline__ uint64_t scalar64(uint64_t v) {  // tells the compiler that v is wave-uniform
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | (uint64_t)lo;
}

// ---- pieces of K / V rows ------------------------------------------------------------------
// VEC: rows start on 16-byte boundaries and hold whole 16-byte pieces.  The pieces of a chunk of
// keys are fetched with buffer loads whose descriptor ends at the last key that counts, so later
// rows read as zeros; a piece past the head's end is given an offset no descriptor covers.
// Otherwise a piece is sixteen bytes from anywhere inside its row (global loads need no alignment): the
// row's last ones where the piece goes past the head, put right (settle_piece) when they have arrived, so
// that a step's loads are in flight together (element by element under the two bounds, each load was
// waited for: 64 tokens x 2, 4 / 4 heads of 129, binary16 32 us); heads shorter than a piece by elements.
constexpr uint32_t kNowhere = 0xf0000000u;
constexpr uint32_t kMaxRecords = 0x80000000u;   // 64 rows of at most 2^25 bytes

__device__ __forceinline__ __amdgpu_buffer_rsrc_t chunk_rsrc(uint64_t plane, uint64_t off, uint64_t valid) {
  // (both offsets below 2^63, told apart by the high word: the scalar unit has no ordered 64-bit compare)
  const uint64_t left = valid - off;
  const int32_t hi = (int32_t)(left >> 32);
  const uint32_t lo = (uint32_t)left;
  const uint32_t capped = hi < 0 ? 0u : hi > 0 || lo > kMaxRecords ? kMaxRecords : lo;
  return __builtin_amdgcn_make_buffer_rsrc((void*)(plane + off), 0, (uint32_t)__builtin_amdgcn_readfirstlane((int)capped), 0x00020000);
}

template <typename S>
__device__ __forceinline__ u32x4 gather_piece(const typename Store<S>::E* plane, size_t stride_pos, uint32_t key,
                                              uint32_t end, uint32_t e0, uint32_t head_size) {
  typedef u32x4 AnyPlace __attribute__((aligned(2)));
  constexpr uint32_t kPiece = Store<S>::kPiece;
  const typename Store<S>::E* row = plane + (size_t)min(key, end - 1) * stride_pos;
  if (head_size >= kPiece) return *(const AnyPlace*)(row + min(e0, head_size - kPiece));
  u32x4 w = {0, 0, 0, 0};
#pragma unroll
  for (uint32_t e = 0; e < kPiece; ++e) {
    const typename Store<S>::E x = row[min(e, head_size - 1)];
    if constexpr (std::is_same<S, F32>::value) w[e] = e < head_size ? __builtin_bit_cast(uint32_t, x) : 0u;
    else w[e >> 1] |= (e < head_size ? (uint32_t)x : 0u) << (16 * (e & 1));
  }
  return w;
}

// The piece that was asked for, of what gather_piece fetched: the row's last elements moved down to its
// start, zeros past the head and past the keys.
template <typename S>
__device__ __forceinline__ u32x4 settle_piece(u32x4 w, uint32_t key, uint32_t end, uint32_t e0, uint32_t head_size) {
  constexpr uint32_t kPiece = Store<S>::kPiece, kBits = 128 / kPiece;
  const uint32_t from = head_size >= kPiece ? min(e0, head_size - kPiece) : 0u;
  const uint32_t bits = (e0 - from) * kBits;
  uint64_t lo = (uint64_t)w[0] | (uint64_t)w[1] << 32, hi = (uint64_t)w[2] | (uint64_t)w[3] << 32;
  if (bits >= 64) {
    lo = hi;
    hi = 0;
  }
  const uint32_t rest = bits & 63;
  lo = lo >> rest | (hi << 1) << (63 - rest);
  hi >>= rest;
  const bool any = key < end && e0 < head_size;
  return any ? u32x4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)} : u32x4{0, 0, 0, 0};
}

// Query row piece: elements e0 .. of the row, zeros past the head's end, sign folded in.
template <typename S, bool VEC>
__device__ __forceinline__ u32x4 query_piece(const GeneralArgs& p, const typename Store<S>::E* row, uint32_t e0) {
  u32x4 w = {0, 0, 0, 0};
  if constexpr (VEC) {
    if (e0 < p.head_size) w = load16(row + e0);
  } else {
    w = settle_piece<S>(gather_piece<S>(row, 0, 0, 1, e0, p.head_size), 0, 1, e0, p.head_size);
  }
  if (p.negate_q) w ^= std::is_same<S, F32>::value ? 0x80000000u : 0x80008000u;
  return w;
}

// Whether a piece holds an element with all exponent bits set (infinity or NaN): one more in the exponent's last
// place carries into the sign's, and no further.
template <typename S>
__device__ __forceinline__ uint32_t exponent_carry(uint32_t x) {
  constexpr uint32_t m = Store<S>::kExpMask;
  return (x & m) + (m & ~(m << 1));
}
template <typename S>
__device__ __forceinline__ bool piece_not_finite(u32x4 w) {
  constexpr uint32_t sign = std::is_same<S, F32>::value ? 0x80000000u : 0x80008000u;
  return ((exponent_carry<S>(w[0]) | exponent_carry<S>(w[1]) | exponent_carry<S>(w[2]) | exponent_carry<S>(w[3])) & sign) != 0;
}

// Agent-scope accesses for partial rows that another workgroup of the same launch folds.
__device__ __forceinline__ void store_agent(float* p, float v) {
  __hip_atomic_store((uint32_t*)p, __builtin_bit_cast(uint32_t, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ uint32_t lane_number() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m);
  return v;
}

// One query row over keys [k0, end), by one wave and without matrix instructions, result into the
// output or the partial row.  The matrix kernels multiply every value row of a chunk
// by every query row, masked pairs with a weight of zero, and 0 x infinity is not 0; a query row
// must not see what the value rows of later positions hold, so a workgroup that meets a value
// that is not finite beyond its first row's position takes its rows through here instead.  So do rows
// whose sums are not finite (not_finite_sum).
template <typename S>
__device__ __forceinline__ void plain_row(const GeneralArgs& p, const typename Store<S>::E* kp,
                                                     const typename Store<S>::E* vp, size_t row, size_t prow,
                                                     uint32_t k0, uint32_t end, uint32_t pitch, bool partial, int lane) {
  typedef typename Store<S>::E E;
  constexpr int kPerLane = kMaxHead / kWave;
  const E* q = (const E*)p.q + row * p.head_size;
  float qv[kPerLane], o[kPerLane];
#pragma unroll
  for (int i = 0; i < kPerLane; ++i) {
    const uint32_t d = lane + 64 * i;
    qv[i] = d < p.head_size ? (p.negate_q ? -load_elem<S>(q + d) : load_elem<S>(q + d)) : 0.0f;
    o[i] = 0.0f;
  }
  float m = -INFINITY, l = 0.0f;
  for (uint32_t j = k0; j < end; ++j) {
    float part = 0.0f, vv[kPerLane];
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
      const uint32_t d = lane + 64 * i;
      const size_t at = (size_t)j * p.kv_stride_pos + d;
      part = d < p.head_size ? __builtin_fmaf(qv[i], load_elem<S>(kp + at), part) : part;
      vv[i] = d < p.head_size ? load_elem<S>(vp + at) : 0.0f;
    }
    const float s = wave_sum(part) * p.c;
    const float m_new = fmaxf(m, s), ref = m_new == -INFINITY ? 0.0f : m_new;
    const float alpha = fast_exp2(m - ref), w = fast_exp2(s - ref);
    l = l * alpha + w;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) o[i] = __builtin_fmaf(w, vv[i], o[i] * alpha);
    m = m_new;
  }
  if (partial) {
#pragma unroll
    for (int i = 0; i < kPerLane; ++i)
      if (lane + 64 * i < (int)pitch) store_agent(p.part_o + prow * pitch + lane + 64 * i, o[i]);
    if (lane == 0) {
      store_agent(p.part_ml + 2 * prow, m);
      store_agent(p.part_ml + 2 * prow + 1, l);
    }
  } else {
    E* out = (E*)p.out + row * p.head_size;
    const float inv = 1.0f / l;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i)
      if (lane + 64u * i < p.head_size) store_elem<S>(out + lane + 64 * i, o[i] * inv);
    if (p.lse && lane == 0) p.lse[row] = (m + fast_log2(l)) * kLn2;
  }
}

// Four consecutive elements d .. d + 3 of an output row.
template <typename S, bool VEC>
__device__ __forceinline__ void store_out4(const GeneralArgs& p, size_t row, uint32_t d, f32x4 v) {
  typedef typename Store<S>::E E;
  E* out = (E*)p.out + row * p.head_size + d;
  if constexpr (VEC) {
    if (d >= p.head_size) return;
    if constexpr (std::is_same<S, F32>::value) *(f32x4*)out = v;
    else *(u32x2*)out = u32x2{Mfma<S>::pack2(v[0], v[1]), Mfma<S>::pack2(v[2], v[3])};
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (d + e < p.head_size) store_elem<S>(out + e, v[e]);
  }
}

// Weights of two keys as operands of the second product.  A 16-bit value keeps 11 (binary16) or 8
// (bfloat16) significant bits; the weight goes in as two of them, the rounded value and what the
// rounding left, so that the product carries the weight to 2^-17 of it in bfloat16 and to 2^-22 in
// binary16, whose rest has steps of 2^-24 (2^-31 after kShift, of the reference weight of 1).  The
// output is rounded once, at the end.
template <typename S>
__device__ __forceinline__ void split_pair(float p0, float p1, uint32_t& hi, uint32_t& lo) {
  hi = Mfma<S>::pack2(p0, p1);
  lo = Mfma<S>::pack2(p0 - Mfma<S>::to_float((uint16_t)(hi & 0xffffu)), p1 - Mfma<S>::to_float((uint16_t)(hi >> 16)));
}

// leaf(First) + ... + leaf(First + N - 1), added pairwise.  Binary32 products sum in many short chains of
// matrix instructions: one chain over a head of 128 rounds 128 times at up to the size of the score, and
// that error alone is as large as all others of a row together.
template <int First, int N, typename F>
__device__ __forceinline__ auto pairwise_sum(F& leaf) {
  if constexpr (N == 1) return leaf(std::integral_constant<int, First>{});
  else return pairwise_sum<First, N / 2>(leaf) + pairwise_sum<First + N / 2, N - N / 2>(leaf);
}

// Whether a row with these sums needs plain_row.  largest: the largest magnitude among its weighted sums (NaN
// counts as the largest of all); l: the weights' sum (NaN, as from a key that is not a number: every way to add
// up gives NaN).  A weight in two 16-bit operands on an infinite value gives NaN where it should give the
// infinity, when its rest is 0 or negative (0 x inf, inf - inf), and then the sum is NaN to the end.
__device__ __forceinline__ bool not_finite_sum(float largest, float l) { return !(largest < INFINITY) && l == l; }
__device__ __forceinline__ float largest_of(float m, float a, float b) {   // one instruction
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, __builtin_fabsf(a)), __builtin_fabsf(b));
}

// Launchers of the two kernels (grid and workspace fields of the arguments set); nb = blocks of
// 32 elements of the padded head, vec as above.
hipError_t launch_general_chunk(const GeneralArgs& p, int dtype, int nb, bool vec, uint32_t planes, hipStream_t stream);
hipError_t launch_general_step(const GeneralArgs& p, int dtype, int nb, bool vec, uint32_t planes, hipStream_t stream);

// f(std::integral_constant<int, blocks>, std::bool_constant<vec>) for a value of head_blocks().
template <typename F>
inline hipError_t with_head_blocks(int nb, bool vec, F f) {
  using std::integral_constant;
  if (vec) {
    switch (nb) {
      case 1: return f(integral_constant<int, 1>{}, std::true_type{});
      case 2: return f(integral_constant<int, 2>{}, std::true_type{});
      case 3: return f(integral_constant<int, 3>{}, std::true_type{});
      case 4: return f(integral_constant<int, 4>{}, std::true_type{});
      case 6: return f(integral_constant<int, 6>{}, std::true_type{});
      case 8: return f(integral_constant<int, 8>{}, std::true_type{});
    }
  } else {
    switch (nb) {
      case 2: return f(integral_constant<int, 2>{}, std::false_type{});
      case 4: return f(integral_constant<int, 4>{}, std::false_type{});
      case 8: return f(integral_constant<int, 8>{}, std::false_type{});
    }
  }
  return hipErrorInvalidValue;
}

}  // namespace gen
}  // namespace ellm
