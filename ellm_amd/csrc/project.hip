// Projections around the attention operator on gfx950 MFMA:
//   fused Q/K/V projection   C = X . [Wq; Wk; Wv]^T  with, per finished 128-wide head
//   row, RMS norm (weight 1) and rotary rotation for the query and key heads, the
//   query rows written to the Q scratch, key and value rows written straight to their
//   token coordinates of the cache; replaces MatMul3::run (reference:
//   src/compiler/mul/matmul3.rs:289-385, finalize :243-254 and :436-451);
//   output projection + residual   Y = A . Wo^T + R; replaces MatMulAdd::run
//   (src/compiler/mul/matmul_add.rs:128-232).
// Weights are row-major [N][K] as the reference keeps them ("W_nt"), activations are
// row-major [rows][K]; both operands are K-contiguous, which is what MFMA wants.
//
// Formulation: the product is computed transposed, C^T[n][token] = W . X^T, so that a
// lane of the 16x16 accumulator block owns one token and 4 of 16 output columns: a
// head row (128 columns) of a token then sits in four lanes, the sum of
// squares needs two cross-lane exchanges and the (even, odd) rotation pairs are
// register neighbours.
//
// A workgroup of 8 waves (two per SIMD) owns a tile of 256 tokens x 256 output columns (two heads): mid_tile in
// project_mid_tile.hpp, which also says what bounds it.  Before, four waves of 512 registers with 32x32x16
// instructions and tiles through registers (us, Q/K/V | output projection): 8000 rows 2048 wide 170 | 122 -> 146 | 106,
// 4096 wide 693 | 239 -> 624 | 210, 8192 wide 1108 | 888 -> 1003 | 811 (1.34 and 1.32 PFLOP/s); 2500 rows 2048 wide
// 59 | 53 -> 52 | 44.
// Calls with at most 64 rows go to the streaming kernel of project_small.hip, calls that would
// leave these tiles fewer than the compute units to the 128-token tiles of project_mid.hip.
#include "project_mid_tile.hpp"
#include "project_plan.hpp"

namespace ellm {
using namespace proj;
namespace {

constexpr int kTile = 256;                          // tokens, and output columns, per workgroup
using TileShape = MidShape<2, 8, 2>;
constexpr int kProjThreads = TileShape::kThreads;
constexpr int kProjLdsBytes = TileShape::kLdsBytes;   // the most of the three forms of a workgroup
static_assert(TileShape::kTokens == kTile && MidShape<1, 8, 1>::kLdsBytes <= kProjLdsBytes && MidShape<1, 4, 1>::kLdsBytes <= kProjLdsBytes,
              "forms of a workgroup");
constexpr int kGroupM = 4;                          // token tiles that take turns on one column tile


template <typename S, int MODE>
__global__ __launch_bounds__(kProjThreads) void project_kernel(ProjectKernelArgs p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t proj_smem[];
  // workgroup -> tile: ids that share id % 8 (one XCD, one L2) are made consecutive,
  // then kGroupM token tiles x all column tiles form a band that is walked token-first;
  // the tiles past whole_tiles (a multiple of the compute units, or all) go to tail_parts
  // workgroups each, likewise consecutive per XCD
  const bool whole = blockIdx.x < p.whole_tiles;
  uint32_t tm, tn, part = 0;
  {
    const uint32_t total = whole ? p.whole_tiles : (p.tiles_m * p.tiles_n - p.whole_tiles) * p.tail_parts;
    const uint32_t id = whole ? blockIdx.x : blockIdx.x - p.whole_tiles;
    const uint32_t q = total >> 3, r = total & 7, xcd = id & 7, idx = id >> 3;
    uint32_t pid = xcd * q + min(xcd, r) + idx;
    if (!whole) {
      part = pid % p.tail_parts;
      pid = p.whole_tiles + pid / p.tail_parts;
    }
    const uint32_t per_band = kGroupM * p.tiles_n;
    const uint32_t band = pid / per_band, in_band = pid % per_band;
    const uint32_t first_m = band * kGroupM;
    const uint32_t band_m = min(p.tiles_m - first_m, (uint32_t)kGroupM);
    tm = first_m + in_band % band_m;
    tn = in_band / band_m;
  }
  const uint32_t heads_total = p.heads0 + 2 * p.heads_kv;
  if (!whole) {   // one head of the tile, all of its tokens or half of them
    const uint32_t hh = 2 * tn + (part & 1), first = tm * kTile + (part >> 1) * (kTile / 2);
    if (hh >= heads_total || first >= p.rows) return;
    if (p.tail_parts == 2)
      mid_tile<S, MODE, 1, 8, 1>(p, first, hh, proj_smem);
    else if (threadIdx.x < MidShape<1, 4, 1>::kThreads)   // (four of the eight waves)
      mid_tile<S, MODE, 1, 4, 1>(p, first, hh, proj_smem);
    return;
  }
  mid_tile<S, MODE, 2, 8, 2>(p, tm * kTile, 2 * tn, proj_smem);
}

}  // namespace

// Compute units of the device the kernels were prepared on (project_prepare()).
static uint32_t g_n_cu = 256;

// Which kernel a call runs: the few-rows streaming kernel when the handle has its workspace
// and the shape fits it; else the smallest tile whose workgroups all fit the part at once, one
// per compute unit (128 tokens x one head, then 256 tokens x one head); else 256 x 256 tiles,
// whose traffic per flop is the lowest.  Measured on 256 compute units for 2048 -> 5120 (us, 128-token / 256-token /
// 256 x 256 tiles): 640 rows 20 / 25 / 46, 1024 rows 36 / 28 / 46, 1536 rows 42 / 32 / 47, 2048 rows 58 / 53 / 49.
// Where the 256 x 256 tiles would leave two fifths of the units without one and two rounds of 128-token
// tiles suffice, those are faster still (256 x 256 / 128-token tiles, bf16, us): 640 rows 4096 -> 12288 80 / 65, 520 rows
// 79 / 62, 600 rows 2048 -> 12288 45 / 37, 896 rows 7168 -> 9216 132 / 109, 1152 rows 4096 -> 7168 80 / 66, 300 rows 8192
// -> 18432 149 / 122, 384 rows 152 / 141 (thirteen such shapes, 1.08 to 1.28).
int project_path(uint32_t rows, uint32_t heads, uint32_t K, bool has_workspace) {
  if (has_workspace && small_kernel_takes(rows, K)) return kPathFewRows;
  if (((rows + 127) / 128) * heads <= g_n_cu) return kPathTiles128;
  if (((rows + 255) / 256) * heads <= g_n_cu) return kPathTiles256x1;
  if (((rows + 127) / 128) * heads <= 2 * g_n_cu && 5 * ((rows + 255) / 256) * ((heads + 1) / 2) <= 3 * g_n_cu) return kPathTiles128;
  return kPathTiles;
}

bool project_raw_takes(uint32_t rows, uint32_t heads, uint32_t K, bool has_workspace) {
  return project_path(rows, heads, K, has_workspace) == kPathFewRows;
}

hipError_t launch_project(const ProjectArgs& a, hipStream_t stream) {
  if (a.rows == 0) return hipSuccess;
  ProjectKernelArgs p;
  p.x = (const uint16_t*)a.x;
  p.w[0] = (const uint16_t*)a.w0;
  p.w[1] = (const uint16_t*)a.wk;
  p.w[2] = (const uint16_t*)a.wv;
  p.out0 = (uint16_t*)a.out0;
  p.residual = (const uint16_t*)a.residual;
  p.k_out = (uint16_t*)a.k_out;
  p.v_out = (uint16_t*)a.v_out;
  p.rope = (const uint16_t*)a.rope;
  p.positions = a.positions;
  p.seq_offsets = a.seq_offsets;
  p.seq_caps = a.seq_caps;
  p.kv_stride_seq = a.kv_stride_seq;
  p.kv_stride_head = a.kv_stride_head;
  p.kv_stride_pos = a.kv_stride_pos;
  p.ld0 = a.heads0 * kHeadDim;
  p.rope_pos_stride = a.rope_pos_stride;
  p.rope_head_stride = a.rope_head_stride;
  p.K = a.K;
  p.rows = a.rows;
  p.batch_pitch = a.batch_pitch;
  p.batch = a.batch;
  p.heads0 = a.heads0;
  p.heads_kv = a.heads_kv;
  p.tiles_m = (a.rows + kTile - 1) / kTile;
  p.tiles_n = (a.heads0 + 2 * a.heads_kv + 1) / 2;
  p.position_index = a.position_index;
  p.max_start = a.max_start;
  p.finalize0 = a.finalize0;
  p.eps = a.eps;
  p.k_split = 1;
  p.half_heads = 0;
  p.part = nullptr;
  const uint32_t heads = a.heads0 + 2 * a.heads_kv;
  const int path = project_path(a.rows, heads, a.K, a.ws && a.counters);
  if (a.raw_out) {
    if (path != kPathFewRows || a.residual) return hipErrorInvalidValue;   // (project_raw_takes() said otherwise)
    return launch_project_small(p, a.ws, a.counters, g_n_cu, a.dtype, kModeRaw, stream);
  }
  if (path == kPathFewRows)
    return launch_project_small(p, a.ws, a.counters, g_n_cu, a.dtype, a.residual ? kModeAdd : kModeQkv, stream);
  if (path == kPathTiles128 && a.part) {
    const ProjectSplit split = project_split(a.rows, heads, a.K, g_n_cu);
    if (split.k_split > 1 && split_floats(split, a.rows, heads) <= a.part_floats) {
      p.k_split = split.k_split;
      p.half_heads = split.half_heads;
      p.part = a.part;
      return launch_project_mid(p, split.token_blocks, a.dtype, a.residual != nullptr, stream);
    }
  }
  if (path == kPathTiles128 || path == kPathTiles256x1)
    return launch_project_mid(p, path == kPathTiles128 ? 1 : 2, a.dtype, a.residual != nullptr, stream);
  // A last round of tiles that would leave half of the compute units without one, or three
  // quarters, is cut into halves (256 tokens x one head) or quarters (128 x one head), one per unit:
  // a half takes 0.6 of a tile's time, a quarter 0.4, and what reads more of the L2 lines per flop
  // runs only where units would idle.  Attention block of a layer, whole tiles -> cut (us): 8000 tokens
  // 2048 wide, 32 / 4 heads (640 tiles, 128 cut) 741 -> 731; 4300 tokens (340 tiles) 348 -> 335; 1800
  // tokens 8192 wide, 64 / 8 heads (320 tiles) 619 -> 538; 3300 tokens (520 and 416 tiles) 1155 -> 1089.
  // More than half a round stays whole: its halves would need two rounds of 0.6.
  const uint32_t tiles = p.tiles_m * p.tiles_n, last = tiles % g_n_cu;
  p.whole_tiles = tiles;
  p.tail_parts = 1;
  if (tiles > g_n_cu && last && 2 * last <= g_n_cu) {
    p.whole_tiles = tiles - last;
    p.tail_parts = 4 * last <= g_n_cu ? 4 : 2;
  }
  const uint32_t blocks = p.whole_tiles + (tiles - p.whole_tiles) * p.tail_parts;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kProjThreads), kProjLdsBytes, stream, p);
    return hipGetLastError();
  };
  if (a.residual)
    return a.dtype == 0 ? go(project_kernel<F16, kModeAdd>) : go(project_kernel<BF16, kModeAdd>);
  return a.dtype == 0 ? go(project_kernel<F16, kModeQkv>) : go(project_kernel<BF16, kModeQkv>);
}

// The kernels' LDS needs exceed the default limit; raised here, on the current device, when
// a handle is created, not at launch (a launch may be recorded into a graph).  With every handle (2 us): a mark that
// it has been done once would outlive the device's reset.
hipError_t project_prepare() {
  const void* kernels[] = {(const void*)project_kernel<F16, kModeQkv>, (const void*)project_kernel<BF16, kModeQkv>,
                           (const void*)project_kernel<F16, kModeAdd>, (const void*)project_kernel<BF16, kModeAdd>};
  for (const void* k : kernels) {
    const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kProjLdsBytes);
    if (e != hipSuccess) return e;
  }
  int dev = 0, n_cu = 0;
  if (hipGetDevice(&dev) == hipSuccess &&
      hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n_cu > 0)
    g_n_cu = (uint32_t)n_cu;
  return mid_prepare();
}

size_t project_workspace_floats(uint32_t heads) { return (size_t)heads * kHeadDim * kSmallRowsMax; }
size_t project_part_floats(uint32_t heads, uint32_t K, size_t max_rows) { return project_split_room(heads, K, g_n_cu, max_rows); }

}  // namespace ellm
