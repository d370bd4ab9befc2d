// Attention for the shapes the 128-wide 16-bit kernels do not take: any head size up to 256 and
// binary32 storage.  The reference's generic leaf (src/kernel/generic/flash_attention.rs:60-89)
// honours whatever `length` and element type its caller hands it, and its operator test runs in
// f32 (src/compiler/mul/attention.rs:262-330).  Same arguments, masks, position rules and
// log-sum-exp as the other kernels (ellm_attn_run / ellm_attn_run_ragged).  This file: the launches
// (general_plan.hpp chooses), the kernel for short walks, and the merge of a chunk's splits.
#include "attn_general.hpp"

namespace ellm {
namespace gen {
namespace {

// Folds the partial rows of a chunk call: G lanes per (query row, four columns) take the row's
// splits in turn and combine through lane exchanges.  A row's live splits are those that start
// before the end of its workgroup's keys; one whose keys are all masked for this row left
// (-inf, 0) and weighs nothing.  Split 0 always holds key 0, so the reference is finite.
template <typename S, bool VEC, int G, int TURN>
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
  float l;
  f32x4 o;
  const float m = fold_splits<G, TURN>(p.part_ml + prow * p.n_split * 2, p.part_o + prow * p.n_split * pitch + 4 * dq, pitch, sub,
                                 live, p.n_split, l, o);
  if (!valid || sub != 0) return;
  const size_t row = query_row(p, seq, kvh, r);
  const float inv = 1.0f / l;
  store_out4<S, VEC>(p, row, 4 * dq, f32x4{o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv});
  if (p.lse && dq == 0) p.lse[row] = (m + fast_log2(l)) * kLn2;
}

// One workgroup per (token, sequence, query head) row, without matrix instructions: for walks of a few turns,
// where a launch of the matrix kernels is mostly what their tiles cost whatever is in them, and for few rows of
// wide heads (general_plan() has the rule and the measured times).  The four waves take the row's keys in turns of four, a
// lane owns elements lane, lane + 64, ... of the head, scores are sums over the wave, the soft-max runs online
// and the waves' partial rows meet in LDS.  Bound by the chain of turns: four trips to memory's data, six lane
// exchanges a score, an exponential.
constexpr int kRowWaves = 4, kRowKeys = kRowTurn / kRowWaves;

template <typename S>
__global__ __launch_bounds__(kRowWaves* kWave) void general_rows_kernel(GeneralArgs p) {
  typedef typename Store<S>::E E;
  constexpr int kPerLane = kMaxHead / kWave;
  __shared__ float s_o[kRowWaves][kMaxHead];
  __shared__ float s_m[kRowWaves], s_l[kRowWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // longest rows first, the planes side by side
  const uint32_t hs = p.head_size, planes = gridDim.x / p.rows, plane = blockIdx.x % planes;
  const uint32_t r = p.rows - 1 - blockIdx.x / planes;
  const uint32_t seq = plane / p.n_kv_heads, kvh = plane % p.n_kv_heads;
  const uint32_t pos = start_position(p, seq) + r / p.group;
  const size_t row = query_row(p, seq, kvh, r);
  const E* q = (const E*)p.q + row * hs;
  const size_t plane_at = seq_plane_offset(p.seq_offsets, p.kv_stride_seq, seq) + (size_t)kvh * p.kv_stride_head;
  const E* kp = (const E*)p.k + plane_at;
  const E* vp = (const E*)p.v + plane_at;

  float qv[kPerLane], o[kPerLane];
#pragma unroll
  for (int i = 0; i < kPerLane; ++i) {
    const uint32_t d = lane + 64 * i;
    qv[i] = d < hs ? load_elem<S>(q + d) * p.scale : 0.0f;
    o[i] = 0.0f;
  }
  float m = -INFINITY, l = 0.0f;
  // wave w takes keys 16 n + 4 w .. + 3 (wave-uniform bounds: no lane leaves the reductions)
  for (uint32_t j0 = kRowKeys * wave; j0 <= pos; j0 += kRowTurn) {
    float kk[kRowKeys][kPerLane], vv[kRowKeys][kPerLane];
#pragma unroll
    for (int u = 0; u < kRowKeys; ++u) {
      const size_t at = (size_t)min(j0 + u, pos) * p.kv_stride_pos;   // keys past the row's own position are masked below
#pragma unroll
      for (int i = 0; i < kPerLane; ++i) {
        const uint32_t d = lane + 64 * i;
        kk[u][i] = d < hs ? load_elem<S>(kp + at + d) : 0.0f;
        vv[u][i] = d < hs ? load_elem<S>(vp + at + d) : 0.0f;
      }
    }
    float s[kRowKeys];
#pragma unroll
    for (int u = 0; u < kRowKeys; ++u) {
      float part = 0.0f;
#pragma unroll
      for (int i = 0; i < kPerLane; ++i) part = __builtin_fmaf(qv[i], kk[u][i], part);
      s[u] = (j0 + u <= pos) ? wave_sum(part) : -INFINITY;
    }
    float m_new = m;
#pragma unroll
    for (int u = 0; u < kRowKeys; ++u) m_new = fmaxf(m_new, s[u]);
    const float alpha = __expf(m - m_new);   // m = -inf on the first turn: exp(-inf) = 0
    l *= alpha;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) o[i] *= alpha;
#pragma unroll
    for (int u = 0; u < kRowKeys; ++u) {
      const float w = __expf(s[u] - m_new);  // masked keys: exp(-inf) = 0
      l += w;
#pragma unroll
      for (int i = 0; i < kPerLane; ++i) o[i] = __builtin_fmaf(w, vv[u][i], o[i]);
    }
    m = m_new;
  }
  // the four waves' partial rows meet in LDS (a wave without keys leaves max = -inf, sum = 0)
#pragma unroll
  for (int i = 0; i < kPerLane; ++i) s_o[wave][lane + 64 * i] = o[i];
  if (lane == 0) {
    s_m[wave] = m;
    s_l[wave] = l;
  }
  __syncthreads();
  float top = s_m[0];   // finite: wave 0 holds key 0
#pragma unroll
  for (int w = 1; w < kRowWaves; ++w) top = fmaxf(top, s_m[w]);
  float sum = 0.0f, wgt[kRowWaves];
#pragma unroll
  for (int w = 0; w < kRowWaves; ++w) {
    wgt[w] = __expf(s_m[w] - top);
    sum += wgt[w] * s_l[w];
  }
  const float inv = 1.0f / sum;
  E* out = (E*)p.out + row * hs;
  for (uint32_t d = threadIdx.x; d < hs; d += blockDim.x) {
    float acc = 0.0f;
#pragma unroll
    for (int w = 0; w < kRowWaves; ++w) acc += wgt[w] * s_o[w][d];
    store_elem<S>(out + d, acc * inv);
  }
  if (p.lse && threadIdx.x == 0) p.lse[row] = top + __logf(sum);
}

hipError_t launch_rows(const GeneralArgs& p, int dtype, uint32_t planes, hipStream_t stream) {
  const dim3 grid(planes * p.rows), block(kRowWaves * kWave);
  if (dtype == 0)
    hipLaunchKernelGGL(general_rows_kernel<F16>, grid, block, 0, stream, p);
  else if (dtype == 1)
    hipLaunchKernelGGL(general_rows_kernel<BF16>, grid, block, 0, stream, p);
  else
    hipLaunchKernelGGL(general_rows_kernel<F32>, grid, block, 0, stream, p);
  return hipGetLastError();
}

template <typename S, bool VEC>
hipError_t launch_merge(const GeneralArgs& p, uint32_t planes, uint32_t pitch, hipStream_t stream) {
  const size_t items = (size_t)planes * p.rows * (pitch / 4);
  auto go = [&](auto kernel, size_t lanes) {
    hipLaunchKernelGGL(kernel, dim3((uint32_t)((items * lanes + 255) / 256)), dim3(256), 0, stream, p, planes, pitch,
                       p.tile_rows);
    return hipGetLastError();
  };
  // (as in prefill.hip; 40 tokens on 1536, 32 / 8 heads of 64, 4 pieces 12.05 / 11.8 us)
  if (p.n_split > 8 && items * 8 <= kMergeLanes)
    return p.n_split > 16 ? go(general_merge_kernel<S, VEC, 8, 4>, 8) : go(general_merge_kernel<S, VEC, 8, 2>, 8);
  return p.n_split > 2 ? go(general_merge_kernel<S, VEC, 1, 4>, 1) : go(general_merge_kernel<S, VEC, 1, 2>, 1);
}

uint32_t element_bytes(int dtype) { return dtype == 2 ? 4 : 2; }

}  // namespace
}  // namespace gen

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
  p.scale = a.scale;
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
  gen::GeneralCall call;
  call.planes = planes;
  call.group = a.group;
  call.interval = a.position_interval;
  call.max_len = a.position_index + a.position_interval;
  call.n_cu = a.n_cu;
  call.head_size = head_size;
  call.f32 = a.dtype == 2;
  call.vec = vec;
  call.room = p.part_o ? a.prefill_part_rows / ((size_t)planes * rows) : 1;
  const gen::GeneralPlan plan = gen::general_plan(call);
  const int nb = plan.nb;
  p.row_tiles = plan.row_tiles;
  p.tile_rows = plan.tile_rows;
  p.key_groups = plan.key_groups;
  p.turn_at = plan.turn_at;
  p.max_first = plan.max_first;
  p.n_split = plan.n_split;
  p.split_len = plan.split_len;
  if (plan.kernel == gen::kGeneralRows) return gen::launch_rows(p, a.dtype, planes, stream);
  if ((size_t)planes * p.row_tiles * (plan.kernel == gen::kGeneralStep ? p.n_split : 1) > 0x7fffffffu) return hipErrorInvalidValue;
  if (plan.kernel == gen::kGeneralStep) return gen::launch_general_step(p, a.dtype, nb, vec, planes, stream);
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
