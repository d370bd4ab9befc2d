// Projections of at most 64 token rows (a single-token step over that many sequences, a short chunk):
// bound by the stream of the weights from memory.  Same arithmetic and epilogue as the tile kernels.
//
// A workgroup owns 8 W8 output columns, so that about one workgroup per compute unit covers the
// matrix, and all of K.  Its eight waves take K in chunks of 64 (one 128-byte line of every row) in
// turn, each a stream of its own with nothing to meet the others for until the end: the chunk's weight
// and token rows go memory -> registers (eight whole lines an instruction, several chunks in flight) ->
// the wave's slice of LDS (16-byte pieces permuted by (row >> 1) & 7: stores and operand reads both
// conflict-free) -> 16x16x32 MFMA operands, weights as the A operand.  The waves' sums meet in LDS.
//
// Columns that are not normalised (value heads, the output projection, the raw sums of a fused
// single-token step) are finished by their own workgroup.  A normalised head needs the sum of squares
// over its 128 columns, i.e. over several workgroups: each leaves its columns in a workspace
// (device-coherent stores) and counts itself in; the last of them to arrive reads the head back,
// normalises, rotates and stores it.  The counters reset themselves.
//
// Measured (us a call, weights from memory), against 16- or 32-column workgroups that fetched all of K in
// one burst and re-read the token rows from the caches in operand layout: raw sums of 2048 -> 5120, one
// row 7.6 -> 6.2, 2048 -> 5120 with finished heads, 1 / 16 / 64 rows 9.4 / 9.9 / 17.0 -> 8.3 / 9.1 / 14.6;
// 4096 -> 12288, 1 / 16 / 64 rows 24 / 29 / 62 -> 21 / 21 / 27; 8192 -> 10240, 1 / 16 / 64 rows 53 / 65 / 64 ->
// 31 / 32 / 42 (all before the workgroups walked K apart, below).  What is left beside the stream is about 6 us a launch:
// start, first data, the sums, the store.
#include "project_common.hpp"

namespace ellm {
using namespace proj;
namespace {

constexpr int kStWaves = 8;
constexpr int kStThreads = kStWaves * kWave;
constexpr int kChunkK = 64;
constexpr int kLine = kChunkK * 2;   // bytes of a row in a chunk
constexpr int kCachePolicySc1 = 16;  // device-coherent (what the compiler's own agent-scope atomic loads carry)

__device__ __forceinline__ void store_coherent64(float* p, float lo, float hi) {
  const uint64_t bits = (uint64_t)__builtin_bit_cast(uint32_t, lo) | ((uint64_t)__builtin_bit_cast(uint32_t, hi) << 32);
  __hip_atomic_store((uint64_t*)p, bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ f32x4 load_coherent128(__amdgpu_buffer_rsrc_t table, uint32_t off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(table, off, 0, kCachePolicySc1));
}
__device__ __forceinline__ void wait_vm_done() { __builtin_amdgcn_s_waitcnt(0x0F70); }

typedef __attribute__((address_space(3))) uint8_t LdsByte;
typedef __attribute__((address_space(3))) u32x4 LdsVec4;

// W8: eight-row pieces of weights per chunk (8 W8 columns a workgroup); TB: blocks of 16 token rows.
template <int W8, int TB>
struct StreamShape {
  static constexpr int kCols = 8 * W8, NB = (W8 + 1) / 2;
  static constexpr int kPieces = W8 + 2 * TB;
  // chunks a wave keeps in flight: what 128 registers hold, at most eight
  static constexpr int kDepth = 32 / kPieces > 8 ? 8 : 32 / kPieces < 2 ? 2 : 32 / kPieces;
  static constexpr int kWaveLds = (16 * NB + 16 * TB) * kLine;
  static constexpr int kRedPitch = 16 * NB + 4;   // floats per (wave, token) row of the sums
  static constexpr int kRedBytes = kStWaves * 16 * TB * kRedPitch * 4;
  static constexpr int kLds = kStWaves * kWaveLds > kRedBytes ? kStWaves * kWaveLds : kRedBytes;
  static constexpr int kQuads = kCols / 4;
  static constexpr int kItems = (16 * TB * kQuads + kStThreads - 1) / kStThreads;   // (token, four columns) per thread
};

template <typename S, int MODE, int W8, int TB>
__global__ __launch_bounds__(kStThreads, 2) void project_small_kernel(ProjectKernelArgs p, float* ws, uint32_t* counters) {
  using M = Mfma<S>;
  using X = StreamShape<W8, TB>;
  constexpr int NB = X::NB, kDepth = X::kDepth;
  __shared__ __attribute__((aligned(16))) uint8_t smem[X::kLds];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i16 = lane & 15, q4 = lane >> 4;
  const uint32_t K = p.K, n_chunks = K / kChunkK;
  const uint32_t col0 = blockIdx.x * X::kCols, n_cols = (p.heads0 + 2 * p.heads_kv) * kHeadDim;

  auto finalizes = [&](uint32_t head) { return head < p.heads0 ? p.finalize0 != 0 : head < p.heads0 + p.heads_kv; };
  auto start_of = [&](uint32_t b) { return p.positions ? min(p.positions[b], p.max_start) : p.position_index; };

  // eight columns never straddle two weight matrices (their widths are multiples of 128); pieces past
  // the last column are fetched through empty descriptors
  __amdgpu_buffer_rsrc_t w_rsrc[W8];
#pragma unroll
  for (int i = 0; i < W8; ++i) {
    const uint32_t col = col0 + 8 * i, kv0 = p.heads0 * kHeadDim, kv1 = kv0 + p.heads_kv * kHeadDim;
    const uint16_t* w = col < kv0 ? p.w[0] + (size_t)col * K
                                  : col < kv1 ? p.w[1] + (size_t)(col - kv0) * K : p.w[2] + (size_t)(col - kv1) * K;
    const bool real = col < n_cols;
    w_rsrc[i] = __builtin_amdgcn_make_buffer_rsrc((void*)uniform64(real ? w : p.w[0]), 0, real ? 8 * K * 2 : 0u, kBufFlags);
  }
  const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)uniform64(p.x), 0, p.rows * K * 2, kBufFlags);
  const int row8 = lane >> 3, piece = lane & 7;
  const uint32_t src = row8 * K * 2 + piece * 16, x_step = 8 * K * 2;
  u32x4 stg[kDepth][X::kPieces];
  // Every workgroup starts its walk along K one chunk further than its neighbour: rows lie a power of two apart with
  // the usual widths, and in step all of them would read the same few kilobytes of every row, that is, from a part of
  // the memory channels (one token, 64 / 8 heads on 8192: 65.2 -> 57.7 us, 32 / 32 on 4096 35.2 -> 33.6; sixteenths of the
  // row apart, or apart by XCD only, less: 61 to 64).
  const uint32_t rot = blockIdx.x % n_chunks;
  auto load_chunk = [&](uint32_t chunk, u32x4 (&st)[X::kPieces]) {
    chunk += rot;
    chunk = chunk >= n_chunks ? chunk - n_chunks : chunk;
#pragma unroll
    for (int i = 0; i < W8; ++i) st[i] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc[i], src, chunk * kLine, 2);   // 2: read once
#pragma unroll
    for (int i = 0; i < 2 * TB; ++i) st[W8 + i] = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, src + i * x_step, chunk * kLine, 0);
  };

  // the residual's pieces are requested ahead of everything else
  u32x2 rs[X::kItems];
#pragma unroll
  for (int n = 0; n < X::kItems; ++n) {
    rs[n] = u32x2{0u, 0u};
    if constexpr (MODE == kModeAdd) {
      const uint32_t item = tid + n * kStThreads, R = item / X::kQuads, col = col0 + 4 * (item % X::kQuads);
      if (R < p.rows && col < n_cols && R % p.batch_pitch < p.batch) rs[n] = *(const u32x2*)(p.residual + (size_t)R * p.ld0 + col);
    }
  }

  const uint32_t lds0 = (uint32_t)(uintptr_t)(LdsByte*)smem + wave * X::kWaveLds;
  const uint32_t st_even = lds0 + row8 * kLine + ((piece ^ (row8 >> 1)) << 4);        // rows 16 n + row8
  const uint32_t st_odd = lds0 + row8 * kLine + ((piece ^ (4 + (row8 >> 1))) << 4);   // rows 16 n + 8 + row8, less the 8 rows
  const uint32_t rd = lds0 + i16 * kLine, swz = (i16 >> 1) & 7;
  const uint32_t rd_s[2] = {rd + ((q4 ^ swz) << 4), rd + (((4 + q4) ^ swz) << 4)};
  f32x4 acc[NB][TB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) acc[nb][tb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto consume = [&](const u32x4 (&st)[X::kPieces]) {
#pragma unroll
    for (int i = 0; i < W8; ++i) *(LdsVec4*)((i & 1 ? st_odd : st_even) + 8 * i * kLine) = st[i];
#pragma unroll
    for (int i = 0; i < 2 * TB; ++i) *(LdsVec4*)((i & 1 ? st_odd : st_even) + (16 * NB + 8 * i) * kLine) = st[W8 + i];
  };
  auto multiply = [&]() {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      u32x4 a[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) a[nb] = *(const LdsVec4*)(rd_s[s] + 16 * nb * kLine);
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) {
        const u32x4 b = *(const LdsVec4*)(rd_s[s] + 16 * (NB + tb) * kLine);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[nb][tb] = M::m16x16x32(a[nb], b, acc[nb][tb]);
      }
    }
  };

  // wave w takes chunks w, w + 8, ...; chunk n of its own travels through register set n % kDepth
  const uint32_t mine = n_chunks > (uint32_t)wave ? (n_chunks - wave + kStWaves - 1) / kStWaves : 0;
#pragma unroll
  for (int d = 0; d < kDepth; ++d)
    if ((uint32_t)d < mine) load_chunk(wave + kStWaves * d, stg[d]);
  for (uint32_t n0 = 0; n0 < mine; n0 += kDepth) {
#pragma unroll
    for (int d = 0; d < kDepth; ++d) {
      if (n0 + d >= mine) break;
      consume(stg[d]);
      if (n0 + d + kDepth < mine) load_chunk(wave + kStWaves * (n0 + d + kDepth), stg[d]);
      __builtin_amdgcn_wave_barrier();
      multiply();
      __builtin_amdgcn_wave_barrier();
    }
  }

  // the waves' sums: red[wave][token][column]; lane (token i16, columns 16 nb + 4 q4 ..)
  __syncthreads();
  float* red = (float*)smem;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
      *(f32x4*)(red + (wave * 16 * TB + 16 * tb + i16) * X::kRedPitch + 16 * nb + 4 * q4) = acc[nb][tb];
  __syncthreads();
#pragma unroll
  for (int n = 0; n < X::kItems; ++n) {
    const uint32_t item = tid + n * kStThreads, R = item / X::kQuads, c4 = item % X::kQuads, col = col0 + 4 * c4;
    if (R >= p.rows || col >= n_cols || R % p.batch_pitch >= p.batch) continue;
    f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < kStWaves; ++w) v += *(const f32x4*)(red + (w * 16 * TB + R) * X::kRedPitch + 4 * c4);
    if constexpr (MODE == kModeRaw) {   // plain stores: the kernel that reads them is the next launch on the stream
      *(f32x4*)(ws + (size_t)R * n_cols + col) = v;
    } else if constexpr (MODE == kModeAdd) {
      v[0] += M::to_float((uint16_t)(rs[n][0] & 0xffffu));
      v[1] += M::to_float((uint16_t)(rs[n][0] >> 16));
      v[2] += M::to_float((uint16_t)(rs[n][1] & 0xffffu));
      v[3] += M::to_float((uint16_t)(rs[n][1] >> 16));
      *(u32x2*)(p.out0 + (size_t)R * p.ld0 + col) = u32x2{M::pack2(v[0], v[1]), M::pack2(v[2], v[3])};
    } else {
      const uint32_t head = col / kHeadDim;
      if (finalizes(head)) {
        store_coherent64(ws + (size_t)R * n_cols + col, v[0], v[1]);
        store_coherent64(ws + (size_t)R * n_cols + col + 2, v[2], v[3]);
      } else {
        uint16_t* to;
        if (head < p.heads0) {
          to = p.out0 + (size_t)R * p.ld0 + col;
        } else {   // (key heads are always normalised)
          const uint32_t b = R % p.batch_pitch, pos = R / p.batch_pitch + start_of(b);
          to = p.v_out + kv_row_offset(p, b, head - p.heads0 - p.heads_kv, pos) + col % kHeadDim;
        }
        *(u32x2*)to = u32x2{M::pack2(v[0], v[1]), M::pack2(v[2], v[3])};
      }
    }
  }
  if constexpr (MODE == kModeQkv) {
    // arrivals: every thread's stores acknowledged, then one count per normalised head the columns touch
    __shared__ uint32_t s_last[2];
    const uint32_t head0 = col0 / kHeadDim, last_col = min(col0 + X::kCols, n_cols) - 1;
    const uint32_t n_heads = last_col / kHeadDim - head0 + 1;   // one or two: at most 48 columns
    wait_vm_done();
    __syncthreads();
    if ((uint32_t)tid < n_heads) {
      const uint32_t head = head0 + tid;
      uint32_t last = 0;
      if (finalizes(head)) {
        const uint32_t expected = (head * kHeadDim + kHeadDim - 1) / X::kCols - head * kHeadDim / X::kCols + 1;
        const uint32_t old = __hip_atomic_fetch_add(counters + head, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = old + 1 == expected ? 1u : 0u;
        if (last) __hip_atomic_store(counters + head, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
      }
      s_last[tid] = last;
    }
    __syncthreads();
    // the head's last workgroup: thread -> token tid / 16 (+ 32 a turn), columns 8 c .. 8 c + 7
    const int c8 = tid & 15;
    const uint32_t one_zero = M::pack2(1.0f, 0.0f);
    // (the workspace of a handle stays far below 4 GB: byte offsets fit 32 bits)
    const __amdgpu_buffer_rsrc_t ws_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)uniform64(ws), 0, 0xffffffffu, kBufFlags);
    for (uint32_t h = 0; h < n_heads; ++h) {
      if (s_last[h] == 0) continue;
      const uint32_t head = head0 + h, hs = head < p.heads0 ? head : head - p.heads0;
      for (uint32_t R = tid >> 4; R < (p.rows + 15) / 16 * 16; R += kStThreads / 16) {
        const uint32_t at = (R * n_cols + head * kHeadDim + 8 * c8) * 4;
        const uint32_t b = R % p.batch_pitch;
        const bool live = R < p.rows && b < p.batch;
        f32x4 lo = {0.0f, 0.0f, 0.0f, 0.0f}, hi = {0.0f, 0.0f, 0.0f, 0.0f};
        u32x4 rr = {one_zero, one_zero, one_zero, one_zero};
        uint32_t pos = 0;
        if (live) {
          lo = load_coherent128(ws_rsrc, at);
          hi = load_coherent128(ws_rsrc, at + 16);
          pos = R / p.batch_pitch + start_of(b);
          rr = load16(p.rope + (size_t)pos * p.rope_pos_stride + (size_t)hs * p.rope_head_stride + 8 * c8);
        }
        const float o[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        float ss = squares8(o);
#pragma unroll
        for (int m = 1; m < 16; m <<= 1) ss += __shfl_xor(ss, m, 16);
        const u32x4 packed = scale_rotate_pack8<S>(o, inverse_rms(ss, p.eps), rr);
        if (live)
          store16((head < p.heads0 ? p.out0 + (size_t)R * p.ld0 + hs * kHeadDim : p.k_out + kv_row_offset(p, b, hs, pos)) + 8 * c8,
                  packed);
      }
    }
  }
}

template <typename S, int MODE, int W8>
hipError_t launch_rows(const ProjectKernelArgs& p, float* ws, uint32_t* counters, uint32_t n_cols, hipStream_t stream) {
  const dim3 grid((n_cols + 8 * W8 - 1) / (8 * W8)), block(kStThreads);
  if (p.rows <= 16)
    hipLaunchKernelGGL((project_small_kernel<S, MODE, W8, 1>), grid, block, 0, stream, p, ws, counters);
  else if (p.rows <= 32)
    hipLaunchKernelGGL((project_small_kernel<S, MODE, W8, 2>), grid, block, 0, stream, p, ws, counters);
  else if (p.rows <= 48)
    hipLaunchKernelGGL((project_small_kernel<S, MODE, W8, 3>), grid, block, 0, stream, p, ws, counters);
  else
    hipLaunchKernelGGL((project_small_kernel<S, MODE, W8, 4>), grid, block, 0, stream, p, ws, counters);
  return hipGetLastError();
}

template <typename S, int MODE>
hipError_t launch_cols(const ProjectKernelArgs& p, float* ws, uint32_t* counters, uint32_t n_cu, hipStream_t stream) {
  // Columns a workgroup: whole rounds of one workgroup per compute unit, as few rounds as 48 columns
  // allow (a workgroup takes in all token rows with its weights, and a unit 55-60 GB/s: fewer, wider
  // workgroups leave units idle, 160 of 256 with 32 columns of 5120; narrower ones re-read the tokens).
  const uint32_t n_cols = (p.heads0 + 2 * p.heads_kv) * kHeadDim;
  const uint32_t rounds = (n_cols + 48 * n_cu - 1) / (48 * n_cu);
  const uint32_t w8 = (n_cols + 8 * rounds * n_cu - 1) / (8 * rounds * n_cu);
  switch (w8) {
    case 1: return launch_rows<S, MODE, 1>(p, ws, counters, n_cols, stream);
    case 2: return launch_rows<S, MODE, 2>(p, ws, counters, n_cols, stream);
    case 3: return launch_rows<S, MODE, 3>(p, ws, counters, n_cols, stream);
    case 4: return launch_rows<S, MODE, 4>(p, ws, counters, n_cols, stream);
    case 5: return launch_rows<S, MODE, 5>(p, ws, counters, n_cols, stream);
    case 6: return launch_rows<S, MODE, 6>(p, ws, counters, n_cols, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace

namespace proj {

bool small_kernel_takes(uint32_t rows, uint32_t K) { return rows <= kSmallRowsMax && K >= 1024; }

hipError_t launch_project_small(const ProjectKernelArgs& p, float* ws, uint32_t* counters, uint32_t n_cu, int dtype,
                                 int mode, hipStream_t stream) {
  if (mode == kModeAdd)
    return dtype == 0 ? launch_cols<F16, kModeAdd>(p, ws, counters, n_cu, stream)
                      : launch_cols<BF16, kModeAdd>(p, ws, counters, n_cu, stream);
  if (mode == kModeRaw)
    return dtype == 0 ? launch_cols<F16, kModeRaw>(p, ws, counters, n_cu, stream)
                      : launch_cols<BF16, kModeRaw>(p, ws, counters, n_cu, stream);
  return dtype == 0 ? launch_cols<F16, kModeQkv>(p, ws, counters, n_cu, stream)
                    : launch_cols<BF16, kModeQkv>(p, ws, counters, n_cu, stream);
}

}  // namespace proj
}  // namespace ellm
