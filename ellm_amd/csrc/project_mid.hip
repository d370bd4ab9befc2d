// Projection tile kernel for a few hundred to a few thousand rows, where the 256 x 256
// tiles of project.hip leave most compute units without a workgroup (1536 rows, the
// reference's own serving shape of 64 positions x 24 sequences, src/serving/start copy.rs:30,
// make 6 x 20 of them for the fused Q/K/V projection and 6 x 8 for the output projection).
// The same tile code (project_mid_tile.hpp) at 128 or 256 tokens x one head.  Tiles this small move up to twice
// the LDS bytes per MFMA, and 128-bit LDS stores are slow (13 cycles an instruction against
// 4.7 for a read), one more reason why operands go from memory straight into LDS.
// Where even these tiles leave most units idle (79 rows of 4096 -> 2048: 16 of 256) several workgroups share a tile's K
// and leave their sums for project_fold_kernel (project_plan.hpp: when, and both sides measured).  What bounds that form
// is the second launch, 4 us, and the sums' way through the L2s; finishing a tile in the last workgroup to arrive would
// read all of them through one unit at 60 to 100 GB/s, 5 to 8 us for eight pieces.
#include "project_mid_tile.hpp"

namespace ellm {
namespace proj {
namespace {

template <typename S, int MODE, int MB, int WAVES, int CH = 1>
__global__ __launch_bounds__(64 * WAVES) void project_mid_kernel(ProjectKernelArgs p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t mid_smem[];
  // workgroup -> tile: ids that share id % 8 (one XCD, one L2) are made consecutive; a band of
  // p.band_m token tiles x all heads is walked token-first (mid_band)
  const uint32_t total = p.tiles_m * p.tiles_n;
  const uint32_t q = total >> 3, r = total & 7, xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
  const uint32_t pid = xcd * q + min(xcd, r) + idx;
  const uint32_t per_band = p.band_m * p.tiles_n;
  const uint32_t first_m = pid / per_band * p.band_m, in_band = pid % per_band;
  const uint32_t here = min(p.tiles_m - first_m, p.band_m);
  mid_tile<S, MODE, MB, WAVES, 1, CH>(p, (first_m + in_band % here) * MidShape<MB, WAVES, 1, CH>::kTokens, in_band / here, mid_smem);
}

// Sums of the pieces of K, in order, and what the tiles' epilogue does with a finished head: 16 lanes a (row, head),
// eight columns each.
template <typename S, int MODE>
__global__ __launch_bounds__(256) void project_fold_kernel(ProjectKernelArgs p) {
  using M = Mfma<S>;
  const uint32_t heads = p.heads0 + 2 * p.heads_kv, n_cols = heads * kHeadDim;
  const uint32_t item = blockIdx.x * 16 + threadIdx.x / 16, c8 = threadIdx.x % 16;
  const uint32_t R = item / heads, head = item % heads, b = R % p.batch_pitch;
  const bool live = R < p.rows && b < p.batch;
  const size_t step = (size_t)p.rows * n_cols;
  const float* from = p.part + (live ? (size_t)R * n_cols + head * kHeadDim + 8 * c8 : 0);
  const bool rotated = MODE == kModeQkv && (head < p.heads0 ? p.finalize0 != 0 : head < p.heads0 + p.heads_kv);
  const uint32_t hs = head < p.heads0 ? head : head < p.heads0 + p.heads_kv ? head - p.heads0 : head - p.heads0 - p.heads_kv;
  const uint32_t pos = R / p.batch_pitch + (MODE == kModeQkv && live && p.positions ? min(p.positions[b], p.max_start) : p.position_index);
  const uint32_t one_zero = M::pack2(1.0f, 0.0f);
  u32x4 extra = {one_zero, one_zero, one_zero, one_zero};   // rotary row or residual
  if (MODE == kModeAdd && live) extra = load16(p.residual + (size_t)R * p.ld0 + head * kHeadDim + 8 * c8);
  if (MODE == kModeQkv && live && rotated) extra = load16(p.rope + (size_t)pos * p.rope_pos_stride + (size_t)hs * p.rope_head_stride + 8 * c8);
  f32x4 lo = {0.0f, 0.0f, 0.0f, 0.0f}, hi = lo;
  for (uint32_t s = 0; s < p.k_split; s += 4) {   // (four pieces' loads at once)
    f32x4 a[4], c[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* at = from + min(s + i, p.k_split - 1) * step;
      a[i] = *(const f32x4*)at;
      c[i] = *(const f32x4*)(at + 4);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (s + i < p.k_split) {
        lo += a[i];
        hi += c[i];
      }
  }
  float o[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  u32x4 packed;
  if constexpr (MODE == kModeAdd) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      packed[e] = M::pack2(o[2 * e] + M::to_float((uint16_t)(extra[e] & 0xffffu)), o[2 * e + 1] + M::to_float((uint16_t)(extra[e] >> 16)));
  } else {
    float ss = squares8(o);
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) ss += __shfl_xor(ss, m, 16);
    if (rotated) {
      packed = scale_rotate_pack8<S>(o, inverse_rms(ss, p.eps), extra);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) packed[e] = M::pack2(o[2 * e], o[2 * e + 1]);
    }
  }
  if (!live) return;
  uint16_t* to = head < p.heads0 ? p.out0 + (size_t)R * p.ld0 + head * kHeadDim
                                 : (head < p.heads0 + p.heads_kv ? p.k_out : p.v_out) + kv_row_offset(p, b, hs, pos);
  store16(to + 8 * c8, packed);
}

template <int MB, int WAVES>
hipError_t prepare_shape() {
  const void* kernels[] = {(const void*)project_mid_kernel<F16, kModeQkv, MB, WAVES>,
                           (const void*)project_mid_kernel<BF16, kModeQkv, MB, WAVES>,
                           (const void*)project_mid_kernel<F16, kModeAdd, MB, WAVES>,
                           (const void*)project_mid_kernel<BF16, kModeAdd, MB, WAVES>,
                           (const void*)project_mid_kernel<F16, kModePart, MB, WAVES>,
                           (const void*)project_mid_kernel<BF16, kModePart, MB, WAVES>,
                           (const void*)project_mid_kernel<F16, kModePart, MB, 8, 8 / WAVES>,
                           (const void*)project_mid_kernel<BF16, kModePart, MB, 8, 8 / WAVES>};
  for (const void* k : kernels) {
    const hipError_t e =
        hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, MidShape<MB, WAVES, 1>::kLdsBytes);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// Token tiles per band: the eighth of the tiles that an XCD works on side by side is then about
// band x the heads that make up its number, and the operand rows it takes in from outside its L2,
// band x tokens + heads x 128 per chunk, are fewer than with all token tiles of a head side by side.
// Only where that saves a fifth or more: output projection 4096 -> 2048 of 1280 / 1536 (12 x 16 tiles, 24 an
// XCD: 10 row blocks instead of 14) / 2048 / 3072 rows (7 instead of 13) 31.7 / 34.0 / 40.3 / 58.6 -> 31.2 / 33.4 /
// 39.7 / 57.5 us (two runs of each side, 0.1 apart); 770 rows (8 instead of 9) no gain, not taken.
uint32_t mid_band(uint32_t tiles_m, uint32_t tiles_n, uint32_t tokens) {
  const uint32_t per_xcd = (tiles_m * tiles_n + 7) / 8;
  auto rows_with = [&](uint32_t band) {
    const uint32_t heads = (per_xcd + band - 1) / band, wide = (heads + tiles_n - 1) / tiles_n;   // wide: bands an XCD spans
    return band * wide * tokens + (wide > 1 ? tiles_n : heads) * kHeadDim;
  };
  uint32_t best = tiles_m, best_rows = rows_with(tiles_m) * 4 / 5;
  for (uint32_t bands = 2; bands <= tiles_m; ++bands) {
    const uint32_t band = (tiles_m + bands - 1) / bands, rows = rows_with(band);
    if (rows <= best_rows) {
      best_rows = rows;
      best = band;
    }
  }
  return best;
}

template <int MB, int WAVES>
hipError_t launch_shape(ProjectKernelArgs p, int dtype, bool add, hipStream_t stream) {
  using Shape = MidShape<MB, WAVES, 1>;
  p.tiles_m = (p.rows + Shape::kTokens - 1) / Shape::kTokens;
  p.tiles_n = p.heads0 + 2 * p.heads_kv;
  p.band_m = mid_band(p.tiles_m, p.tiles_n, Shape::kTokens);
  const uint32_t blocks = p.tiles_m * p.tiles_n;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(Shape::kThreads), Shape::kLdsBytes, stream, p);
    return hipGetLastError();
  };
  if (p.k_split > 1) {
    constexpr int kHalves = 8 / WAVES;   // (1: the same kernel)
    using Halves = MidShape<MB, 8, 1, kHalves>;
    static_assert(Halves::kTokens == Shape::kTokens && Halves::kRingBytes <= Shape::kLdsBytes, "the same tile");
    auto pieces = [&](auto kernel, uint32_t threads) {
      hipLaunchKernelGGL(kernel, dim3(blocks, p.k_split), dim3(threads), Shape::kLdsBytes, stream, p);
    };
    if (p.half_heads)
      dtype == 0 ? pieces(project_mid_kernel<F16, kModePart, MB, 8, kHalves>, Halves::kThreads)
                 : pieces(project_mid_kernel<BF16, kModePart, MB, 8, kHalves>, Halves::kThreads);
    else
      dtype == 0 ? pieces(project_mid_kernel<F16, kModePart, MB, WAVES>, Shape::kThreads)
                 : pieces(project_mid_kernel<BF16, kModePart, MB, WAVES>, Shape::kThreads);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const dim3 grid((p.rows * p.tiles_n + 15) / 16);
    auto fold = add ? (dtype == 0 ? project_fold_kernel<F16, kModeAdd> : project_fold_kernel<BF16, kModeAdd>)
                    : (dtype == 0 ? project_fold_kernel<F16, kModeQkv> : project_fold_kernel<BF16, kModeQkv>);
    hipLaunchKernelGGL(fold, grid, dim3(256), 0, stream, p);
    return hipGetLastError();
  }
  if (add)
    return dtype == 0 ? go(project_mid_kernel<F16, kModeAdd, MB, WAVES>) : go(project_mid_kernel<BF16, kModeAdd, MB, WAVES>);
  return dtype == 0 ? go(project_mid_kernel<F16, kModeQkv, MB, WAVES>) : go(project_mid_kernel<BF16, kModeQkv, MB, WAVES>);
}

}  // namespace

hipError_t mid_prepare() {
  const hipError_t e = prepare_shape<1, 4>();
  return e != hipSuccess ? e : prepare_shape<1, 8>();
}

// 32x32x16 instructions -> this tile code (us, Q/K/V | output projection): 2048 wide 100 rows 18.0 | 29.1 ->
// 17.1 | 27.1, 1536 rows 37.2 | 34.6 -> 31.9 | 31.6; 4096 wide 256 rows 39.7 | 30.5 -> 35.3 | 28.4; 8192 wide 768 rows
// 132 | 118 -> 116 | 104.  One wave a SIMD (128 tokens) issues 16x16x32 instructions as fast only while it has
// little else to issue: with a register sum per operand read and a descriptor select per load it took 19.0 | 30.4 at
// 100 rows, with neither 17.1 | 27.1.
hipError_t launch_project_mid(ProjectKernelArgs p, uint32_t token_blocks, int dtype, bool add,
                              hipStream_t stream) {
  if (token_blocks != 2) return launch_shape<1, 4>(p, dtype, add, stream);
  return launch_shape<1, 8>(p, dtype, add, stream);
}

}  // namespace proj
}  // namespace ellm
