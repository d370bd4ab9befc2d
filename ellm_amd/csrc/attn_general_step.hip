// Single-token steps (and chunks of at most 32 query rows per K/V plane) for head sizes other than
// 128 and for binary32 storage: a stream of K and V from memory, each row of a plane read by one
// workgroup per 16 query rows, the key range split over workgroups with the partial rows folded by
// the last workgroup of a plane inside the launch (the protocol of decode_common.hpp).
//
// Bound: memory.  A wave streams its own chunks (registers -> its own slice of LDS -> matrix operands,
// no barrier in the loop), sixteen query rows wide, so that binary32 products (256 flops a cycle and
// unit) stay at a third of the stream's time; the four waves of a workgroup take alternate chunks and
// meet once at the end.  Measured: 8 sequences x 4096 keys, 32 query / 4 key-value heads of 128 in
// binary32: 27.5 us (4.9 TB/s), where one workgroup per query row took 437 us; 2 x 11046 keys, 32 / 32
// heads of 256 in bfloat16: 112 us (6.5 TB/s; was 5450); 11 x 131 keys, heads of 96: 6.9 us (was 31).
// Binary32 products sum in short chains (see pairwise_sum): 11 x 2471 keys, 32 / 32 heads of 128, an error of
// 2.1e-7 against 64 bits in 160 us, where one chain over the head and one over all keys gave 6.1e-7 in 156;
// chains of eight throughout 2.1e-7 in 161 (11 x 290 keys 16.0 us, sixteen 15.5).
#include "attn_general.hpp"
#include "decode_common.hpp"

namespace ellm {
namespace gen {
namespace {

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * kWave;
constexpr int kRows = (int)kGeneralStepRows;

typedef __attribute__((address_space(3))) uint8_t LdsByte;
typedef __attribute__((address_space(3))) u32x4 LdsU32x4;
typedef __attribute__((address_space(3))) float LdsF32;
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 LdsI16x4;

template <typename S, int NB>
struct StepShape {
  static constexpr bool kF32 = std::is_same<S, F32>::value;
  static constexpr int kBytes = sizeof(typename Store<S>::E);
  static constexpr int kHead = 32 * NB;
  static constexpr int kRowBytes = kHead * kBytes;
  static constexpr int kPiecesRow = kRowBytes / 16;
  // Keys a wave requests together: MC blocks of 16, about 16 KB of K and V, one such request in
  // flight ahead of the one in LDS; two workgroups a compute unit keep 128 KB on their way.
  static constexpr int MC = kRowBytes <= 128 ? 4 : kRowBytes <= 256 ? 2 : 1;
  static constexpr int kKeys = 16 * MC;
  static constexpr int kPieces = kKeys * kPiecesRow / kWave;
  // K rows: 16 bytes a lane from 16 rows (pitch of 4 x odd words); V rows: the four 16-lane blocks of
  // a transposing read take 32 bytes from each of sixteen rows (8 x odd words), binary32 16 words of
  // rows four apart (4 x odd words).
  static constexpr int kKPitch = kRowBytes + 16;
  static constexpr int kVPitch = kRowBytes + (kF32 ? 16 : 32);
  static constexpr int kWaveLds = kKeys * (kKPitch + kVPitch);
  static constexpr int kRedPitch = kHead + 4;   // floats per (wave, row) of the wave merge
  static constexpr int kRedBytes = kWaves * kRows * kRedPitch * 4;
  static constexpr int kLds = kWaves * kWaveLds > kRedBytes ? kWaves * kWaveLds : kRedBytes;
  static constexpr int kOccupancy = kLds <= 80 * 1024 ? 2 : 1;   // workgroups per compute unit
};

template <typename S, int NB, bool VEC>
__global__ __launch_bounds__(kThreads, (StepShape<S, NB>::kOccupancy)) void general_step_kernel(GeneralArgs p) {
  typedef StepShape<S, NB> X;
  typedef typename Store<S>::E E;
  constexpr int MC = X::MC, kPieces = X::kPieces;
  constexpr int kQ = X::kPiecesRow / 4;      // query registers: pieces 4 s + g of the row
  constexpr float kShift = Store<S>::kShift;
  constexpr int kQuads = X::kHead / 4;
  __shared__ __attribute__((aligned(16))) uint8_t smem[X::kLds];
  __shared__ uint32_t s_bad, s_last;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const uint32_t split = blockIdx.x % p.n_split, unit = blockIdx.x / p.n_split;
  const uint32_t plane = unit / p.row_tiles, row0 = unit % p.row_tiles * kRows;
  const uint32_t seq = plane / p.n_kv_heads, kvh = plane % p.n_kv_heads;
  const uint32_t P0 = start_position(p, seq);
  const uint32_t rows_here = min(p.rows - row0, (uint32_t)kRows);
  const uint32_t total = P0 + (row0 + rows_here - 1) / p.group + 1;   // keys of the last row
  const uint32_t live = (total + p.split_len - 1) / p.split_len;
  if (split >= live) return;
  const uint32_t k0 = split * p.split_len, end = min(total, k0 + p.split_len);
  const uint32_t first_pos = P0 + row0 / p.group;
  const uint32_t n_chunks = (end - k0 + X::kKeys - 1) / X::kKeys;

  const uint32_t r = row0 + min((uint32_t)c, rows_here - 1);
  const uint32_t rowpos = P0 + r / p.group;
  const size_t plane_at = seq_plane_offset(p.seq_offsets, p.kv_stride_seq, seq) + (size_t)kvh * p.kv_stride_head;
  const E* kp = (const E*)p.k + plane_at;
  const E* vp = (const E*)p.v + plane_at;
  const uint64_t kplane = scalar64((uint64_t)kp), vplane = scalar64((uint64_t)vp);
  const uint64_t pos_bytes = (uint64_t)p.kv_stride_pos * sizeof(E);
  const uint64_t valid = scalar64((uint64_t)(end - 1) * pos_bytes + (uint64_t)p.head_size * sizeof(E));
  uint32_t off[kPieces];
  uint32_t lds_k[kPieces];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LdsByte*)smem + wave * X::kWaveLds;
#pragma unroll
  for (int i = 0; i < kPieces; ++i) {
    const uint32_t pi = lane + kWave * i, krow = pi / X::kPiecesRow, col = pi % X::kPiecesRow;
    if constexpr (VEC)
      off[i] = col * Store<S>::kPiece < p.head_size ? (uint32_t)(krow * pos_bytes) + 16 * col : kNowhere;
    else
      off[i] = krow | col * Store<S>::kPiece << 16;
    lds_k[i] = lds0 + krow * X::kKPitch + 16 * col;
  }
  u32x4 kst[kPieces], vst[kPieces];
  auto load_rows = [&](uint32_t kb, const E* rows, uint64_t plane_base, u32x4 (&st)[kPieces]) {
    if constexpr (VEC) {
      const __amdgpu_buffer_rsrc_t rs = chunk_rsrc(plane_base, (uint64_t)kb * pos_bytes, valid);
#pragma unroll
      for (int i = 0; i < kPieces; ++i) st[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, off[i], 0, 2);   // 2: read once
    } else {
#pragma unroll
      for (int i = 0; i < kPieces; ++i)
        st[i] = gather_piece<S>(rows, p.kv_stride_pos, kb + (off[i] & 0xffffu), end, off[i] >> 16, p.head_size);
    }
  };
  auto load_chunk = [&](uint32_t chunk) {
    load_rows(k0 + chunk * X::kKeys, kp, kplane, kst);
    load_rows(k0 + chunk * X::kKeys, vp, vplane, vst);
  };
  if ((uint32_t)wave < n_chunks) load_chunk(wave);

  u32x4 qreg[kQ];
  {
    const E* qrow = (const E*)p.q + query_row(p, seq, kvh, r) * p.head_size;
#pragma unroll
    for (int s = 0; s < kQ; ++s) qreg[s] = query_piece<S, VEC>(p, qrow, (4 * s + g) * Store<S>::kPiece);
  }
  float m_run = -INFINITY, l_run = 0.0f;
  f32x4 acc[2 * NB];
#pragma unroll
  for (int b = 0; b < 2 * NB; ++b) acc[b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  bool bad = false;

  const uint32_t k_read = lds0 + c * X::kKPitch + 16 * g;
  const uint32_t v_base = lds0 + X::kKeys * X::kKPitch;
  const uint32_t v_read = X::kF32 ? v_base + 4 * g * X::kVPitch + 4 * c
                                  : v_base + (4 * g + (c >> 2)) * X::kVPitch + 8 * (c & 3);
  for (uint32_t chunk = wave; chunk < n_chunks; chunk += kWaves) {
    const uint32_t kb = k0 + chunk * X::kKeys;
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      if constexpr (!VEC) {
        kst[i] = settle_piece<S>(kst[i], kb + (off[i] & 0xffffu), end, off[i] >> 16, p.head_size);
        vst[i] = settle_piece<S>(vst[i], kb + (off[i] & 0xffffu), end, off[i] >> 16, p.head_size);
      }
      *(LdsU32x4*)lds_k[i] = kst[i];
      // (the V row of a piece: same place in a table of another pitch)
      const uint32_t pi = lane + kWave * i;
      *(LdsU32x4*)(v_base + pi / X::kPiecesRow * X::kVPitch + pi % X::kPiecesRow * 16) = vst[i];
    }
    if (kb + X::kKeys - 1 > first_pos && p.interval > 1) {   // some row must not see some of these values
#pragma unroll
      for (int i = 0; i < kPieces; ++i) bad |= piece_not_finite<S>(vst[i]);
    }
    if (chunk + kWaves < n_chunks) load_chunk(chunk + kWaves);
    __builtin_amdgcn_wave_barrier();
    // S^T: lane (row c, group g) register r of block mc <-> key kb + 16 mc + 4 g + r
    f32x4 st[MC];
    if constexpr (X::kF32) {
#pragma unroll
      for (int mc = 0; mc < MC; ++mc) {
        // chains of sixteen products, of eight up to heads of 64 (131 keys: with sixteen 1.01 of the error of sums
        // over lanes, with eight 0.91)
        constexpr int kChain = NB <= 2 ? 2 : 4, kChains = 4 / kChain;
        auto chain_scores = [&](auto n_) __attribute__((always_inline)) {
          constexpr int s = decltype(n_)::value / kChains, first = decltype(n_)::value % kChains * kChain;
          const u32x4 a = *(const LdsU32x4*)(k_read + 16 * mc * X::kKPitch + 64 * s);
          f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int e = first; e < first + kChain; ++e)
            sum = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, (uint32_t)a[e]),
                                                       __builtin_bit_cast(float, (uint32_t)qreg[s][e]), sum, 0, 0, 0);
          return sum;
        };
        st[mc] = pairwise_sum<0, kQ * kChains>(chain_scores);
      }
    } else {
#pragma unroll
      for (int mc = 0; mc < MC; ++mc) st[mc] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < kQ; ++s)
#pragma unroll
        for (int mc = 0; mc < MC; ++mc) {
          const u32x4 a = *(const LdsU32x4*)(k_read + 16 * mc * X::kKPitch + 64 * s);
          st[mc] = Mfma<S>::m16x16x32(a, qreg[s], st[mc]);
        }
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int mc = 0; mc < MC; ++mc)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t key = kb + 16 * mc + 4 * g + e;
        st[mc][e] = (key <= rowpos && key < end) ? st[mc][e] : -INFINITY;
        tmax = fmaxf(tmax, st[mc][e]);
      }
    tmax = fmaxf(tmax, xor_shuffle(tmax, 16));
    tmax = fmaxf(tmax, xor_shuffle(tmax, 32));
    const float m_new = fmaxf(m_run, tmax * p.c);   // -inf while the row has seen none of its keys
    const float ref = m_new == -INFINITY ? 0.0f : m_new;
    const float alpha = fast_exp2(m_run - ref);
    float psum = 0.0f;
#pragma unroll
    for (int mc = 0; mc < MC; ++mc)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        st[mc][e] = fast_exp2(__builtin_fmaf(st[mc][e], p.c, kShift - ref));
        psum += st[mc][e];
      }
    l_run = l_run * alpha + psum;
    m_run = m_new;
    if constexpr (X::kF32) {   // a sum of its own per request, in chains of eight keys
#pragma unroll
      for (int b = 0; b < 2 * NB; ++b) {
        auto key_pair = [&](auto n_) __attribute__((always_inline)) {
          constexpr int mc = decltype(n_)::value / 2, e = decltype(n_)::value % 2 * 2;
          const uint32_t vs = v_read + (16 * mc + e) * X::kVPitch + 64 * b;
          const f32x4 sum = __builtin_amdgcn_mfma_f32_16x16x4f32(*(const LdsF32*)vs, st[mc][e],
                                                                 f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
          return __builtin_amdgcn_mfma_f32_16x16x4f32(*(const LdsF32*)(vs + X::kVPitch), st[mc][e + 1], sum, 0, 0, 0);
        };
        const f32x4 part = pairwise_sum<0, 2 * MC>(key_pair);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[b][e] = __builtin_fmaf(acc[b][e], alpha, part[e]);
      }
    } else {
#pragma unroll
      for (int b = 0; b < 2 * NB; ++b) acc[b] *= alpha;
#pragma unroll
      for (int mc = 0; mc < MC; ++mc) {
        const uint32_t vs = v_read + 16 * mc * X::kVPitch;
        u32x2 hi, lo;
        uint32_t h, l;
        split_pair<S>(st[mc][0], st[mc][1], h, l);
        hi[0] = h, lo[0] = l;
        split_pair<S>(st[mc][2], st[mc][3], h, l);
        hi[1] = h, lo[1] = l;
#pragma unroll
        for (int b = 0; b < 2 * NB; ++b) {
          const u32x2 a = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4*)(vs + 32 * b)));
          acc[b] = Mfma<S>::m16x16x16(a, hi, acc[b]);
          acc[b] = Mfma<S>::m16x16x16(a, lo, acc[b]);
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  l_run += xor_shuffle(l_run, 16);
  l_run += xor_shuffle(l_run, 32);

  if constexpr (!X::kF32) {
    float top[2] = {0.0f, 0.0f};
#pragma unroll
    for (int b = 0; b < 2 * NB; ++b)
#pragma unroll
      for (int e = 0; e < 4; e += 2) top[e >> 1] = largest_of(top[e >> 1], acc[b][e], acc[b][e + 1]);
    bad |= not_finite_sum(largest_of(top[0], top[1], 0.0f), l_run);
  }
  // the four waves' rows meet in LDS (the staging buffers are idle behind the barrier)
  if (tid == 0) s_bad = 0;
  __syncthreads();
  if (bad) s_bad = 1;
  float* red = (float*)smem;
  if ((uint32_t)c < rows_here) {
    float* rr = red + (wave * kRows + c) * X::kRedPitch;
#pragma unroll
    for (int b = 0; b < 2 * NB; ++b) *(f32x4*)(rr + 16 * b + 4 * g) = acc[b];
    if (g == 0) *(f32x2*)(rr + X::kHead) = f32x2{m_run == -INFINITY ? m_run : m_run - kShift, l_run};
  }
  __syncthreads();
  const size_t prow0 = ((size_t)plane * p.rows + row0) * p.n_split;
  auto emit = [&](uint32_t rr, uint32_t dq, f32x4 a, float l, float m) {   // a finished output quad
    const size_t row = query_row(p, seq, kvh, row0 + rr);
    const float inv = 1.0f / l;
    store_out4<S, VEC>(p, row, 4 * dq, f32x4{a[0] * inv, a[1] * inv, a[2] * inv, a[3] * inv});
    if (p.lse && dq == 0) p.lse[row] = (m + fast_log2(l)) * kLn2;
  };
  const uint32_t n_items = rows_here * kQuads;
  if (s_bad) {
    for (uint32_t rr = wave; rr < rows_here; rr += kWaves)
      plain_row<S>(p, kp, vp, query_row(p, seq, kvh, row0 + rr), prow0 + (size_t)rr * p.n_split + split, k0,
                   min(end, P0 + (row0 + rr) / p.group + 1), X::kHead, live > 1, lane);
  } else {
    for (uint32_t item = tid; item < n_items; item += kThreads) {
      const uint32_t rr = item / kQuads, dq = item % kQuads;
      f32x2 ml[kWaves];
      f32x4 part[kWaves];
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const float* src = red + (w * kRows + rr) * X::kRedPitch;
        ml[w] = *(const f32x2*)(src + X::kHead);
        part[w] = *(const f32x4*)(src + 4 * dq);
      }
      float m = -INFINITY;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) m = fmaxf(m, ml[w][0]);
      float l = 0.0f;
      f32x4 a = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const float wgt = ml[w][0] == -INFINITY ? 0.0f : fast_exp2(ml[w][0] - m);
        l += wgt * ml[w][1];
        a += wgt * part[w];
      }
      if (live == 1) {
        emit(rr, dq, a, l, m);
      } else {
        const size_t prow = prow0 + (size_t)rr * p.n_split + split;
        dec::store_coherent64(p.part_o + prow * X::kHead + 4 * dq, a[0], a[1]);
        dec::store_coherent64(p.part_o + prow * X::kHead + 4 * dq + 2, a[2], a[3]);
        if (dq == 0) dec::store_coherent64(p.part_ml + prow * 2, m, l);
      }
    }
  }
  if (live == 1) return;
  if (!dec::arrive(p.counters + unit, live, &s_last, tid)) return;
  // the last workgroup of these rows folds every split's partial rows, eight at a time
  const __amdgpu_buffer_rsrc_t parts = dec::table_rsrc(p.part_o);
  for (uint32_t item = tid; item < n_items; item += kThreads) {
    const uint32_t rr = item / kQuads, dq = item % kQuads;
    const size_t first = prow0 + (size_t)rr * p.n_split;
    const uint32_t at = (uint32_t)first * X::kHead * 4 + 16 * dq;
    float m = -INFINITY, l = 0.0f;
    f32x4 a = {0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t s0 = 0; s0 < live; s0 += 8) {
      f32x4 part[8];
      f32x2 ml[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t s = min(s0 + i, live - 1);
        part[i] = dec::load_coherent128(parts, at + s * (X::kHead * 4));
        ml[i] = __builtin_bit_cast(f32x2, dec::load_coherent64(p.part_ml + (first + s) * 2));
        if (s0 + i >= live) ml[i] = f32x2{-INFINITY, 0.0f};
      }
      float m_new = m;
#pragma unroll
      for (int i = 0; i < 8; ++i) m_new = fmaxf(m_new, ml[i][0]);
      const float ref = m_new == -INFINITY ? 0.0f : m_new;
      const float alpha = fast_exp2(m - ref);
      l *= alpha;
      a *= alpha;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float wgt = fast_exp2(ml[i][0] - ref);
        l += wgt * ml[i][1];
        a += wgt * part[i];
      }
      m = m_new;
    }
    emit(rr, dq, a, l, m);
  }
}

}  // namespace

hipError_t launch_general_step(const GeneralArgs& p, int dtype, int nb, bool vec, uint32_t planes, hipStream_t stream) {
  const dim3 grid(planes * p.row_tiles * p.n_split), block(kThreads);
  return with_head_blocks(nb, vec, [&](auto n, auto v) {
    constexpr int NB = decltype(n)::value;
    constexpr bool VEC = decltype(v)::value;
    if (dtype == 0)
      hipLaunchKernelGGL((general_step_kernel<F16, NB, VEC>), grid, block, 0, stream, p);
    else if (dtype == 1)
      hipLaunchKernelGGL((general_step_kernel<BF16, NB, VEC>), grid, block, 0, stream, p);
    else
      hipLaunchKernelGGL((general_step_kernel<F32, NB, VEC>), grid, block, 0, stream, p);
    return hipGetLastError();
  });
}

}  // namespace gen
}  // namespace ellm
