// Chunks of tokens (or any call with more than 32 query rows per K/V plane) for head sizes other
// than 128 and for binary32 storage: the formulation of prefill.hip (S^T = K.Q^T, O^T += V^T.P^T, a
// lane owns one query row, online soft-max in binary32) on 32x32 matrix tiles, templated over the
// storage type and the padded head size.
//
// A key group is two or four waves of 32 rows that share steps of 32 or 64 keys through LDS
// (double-buffered, one barrier a step, the next step's rows in registers meanwhile); up to four groups
// take the steps of the same rows in turn and merge their rows in LDS at the end.  Rows are the
// (token, head) pairs of a GQA group in order, so a group's heads share the K/V rows whatever the
// group size.  What bounds it: 16-bit, the vector instructions of the soft-max (13 a pair of scores,
// two of them quarter-rate exponentials; 7 matrix cycles beside them with heads of 64), and one
// wave issues a vector instruction only every six cycles or so, so that a SIMD wants several waves:
// two, from two groups or two workgroups, are the least, four the best where registers allow.
// Groups that take turns at a step's matrix and vector parts, as the 128-wide tile kernel's do, came out
// slower than groups side by side (a lone wave's vector part is 1.5 x as long as a shared one).
// Binary32 is bound by the matrix pipe (256 flops a cycle and unit) and keeps one group.  Its sums run in
// chains of eight products; the chains are added up behind the next one's matrix instructions, and that
// costs: 681 tokens x 3, 32 / 4 heads of 128, 135 us and an error of 2.1e-7 against 64 bits with chains of
// half a head and of a step's keys, 171 us and 1.3e-7 now (one workgroup per query row: 1673 us, 1.6e-7).
// Measured, one group before: 2048 tokens, 32 query / 8 key-value heads of 64, bfloat16: 46.0 -> 41.9 us
// (410 TFLOP/s); 341 tokens, 32 / 32 heads of 96: 16.2 -> 10.2; 603 tokens x 2, 32 / 4 heads of 192: 40.6 -> 29.1.
// Binary16 heads of 256 (one group: no registers for two): 1019 tokens, 32 / 4 heads 80 us.
// Operands of both products read ahead of their use, values looked at for infinities only in the steps whose keys some
// row must not see, a step's place worked out without vector compares; before -> with it: 2048 tokens, 32 / 8 heads of 64,
// bf16 40.0 -> 37.0 us; 512 x 4 on 7680 220 -> 208; 2048, 32 / 32 heads of 96, f16 64.2 -> 55.7; 512 x 4 on 7680, 32 / 8
// heads of 256, bf16 986 -> 895 (a step of 32 keys x 32 rows of 64: 126 vector instructions, 150 before).
#include "attn_general.hpp"

namespace ellm {
namespace gen {
namespace {

constexpr float kRescaleStep = 8.0f;     // log2 units

typedef __attribute__((address_space(3))) uint8_t LdsByte;
typedef __attribute__((address_space(3))) u32x4 LdsU32x4;
typedef __attribute__((address_space(3))) float LdsF32;
typedef __attribute__((address_space(3))) f32x4 LdsF32x4;
typedef __attribute__((address_space(3))) f32x2 LdsF32x2;
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 LdsI16x4;

// Shape of a kernel: NB blocks of 32 head elements, RB row blocks (waves) of a key group, KG key
// groups, MB blocks of 32 keys a step of a group.
template <typename S, int NB, int RB, int KG>
struct Shape {
  static constexpr bool kF32 = std::is_same<S, F32>::value;
  static constexpr int kBytes = sizeof(typename Store<S>::E);
  static constexpr int kHead = 32 * NB;
  static constexpr int kPiecesRow = kHead * kBytes / 16;
  static constexpr int kWaves = RB * KG, kThreads = kWaves * kWave;
  static constexpr int kGroupThreads = RB * kWave;
  static constexpr int kTileRows = 32 * RB;  // query rows of a workgroup
  static constexpr int MB = (!kF32 && NB <= 4 && KG <= 2 && !(NB == 2 && KG == 2)) ? 2 : 1;
  static constexpr int kKeys = 32 * MB;
  // 16-byte pieces of K (and of V) a thread moves per step
  static constexpr int kAllPieces = kKeys * kPiecesRow;
  static constexpr int kPieces = kAllPieces / kGroupThreads;
  static_assert(kPieces * kGroupThreads == kAllPieces, "every thread moves the same number of pieces");
  // a thread's pieces lie in one column, kRowStep keys apart (or anywhere: 0)
  static constexpr int kRowStep = kGroupThreads % kPiecesRow == 0 ? kGroupThreads / kPiecesRow : 0;
  static constexpr int kPlaces = kRowStep ? 1 : kPieces;
  // Row pitches in LDS, bytes.  K rows are read 16 bytes a lane from 32 rows: a pitch of 4 x odd
  // words spreads 16 of them over all banks.  V rows, 16-bit: a 16-lane block of the transposing read
  // takes 32 bytes from each of four rows and its neighbour the next 32, so four rows 16 x odd words
  // apart cover the banks; binary32: lanes 0-31 read 32 words of a row and lanes 32-63 the same
  // columns four rows on, which 8 x odd words put into the other half of the banks.
  static constexpr int kKPitch = kHead * kBytes + 16;
  static constexpr int kVWords = kHead * kBytes / 4;
  static constexpr int kVPitch = 4 * (kF32 ? kVWords + 8 : (kVWords % 32 == 16 ? kVWords : kVWords + 16));
  static constexpr int kKBuf = kKeys * kKPitch, kVBuf = kKeys * kVPitch;
  static constexpr int kGroupLds = 2 * (kKBuf + kVBuf);
  // The groups' results meet in the same memory, up to half of them at a time: a wave's
  // accumulators and, behind all of those, its rows' maxima and sums.
  static constexpr int kMergeWave = NB * 16 * kWave * 4;
  static constexpr int kMergeLds = KG / 2 * RB * (kMergeWave + 2 * kWave * 4);
  static constexpr int kLds = KG * kGroupLds > kMergeLds ? KG * kGroupLds : kMergeLds;
  static_assert(kLds + 16 <= 160 * 1024, "LDS of a compute unit");
  // Waves per SIMD the registers are planned for: queries, accumulators, scores, weights and the
  // pieces on their way to LDS are about 40 (32 x 32 x head / 64) registers and a few dozen more.
  // Heads of 64 with two groups take steps of 32 keys to fit twice on a unit.
  // Wider binary32 heads have no registers left to hold the next V rows beside the partial sums of the
  // scores: those are requested between the two products (4096 matrix cycles each with heads of 128).
  static constexpr bool kLateV = kF32 && NB >= 4;
  static constexpr int kOccupancy = KG == 2 && NB <= 2 ? 4 : KG > 1 ? kWaves / 4 : kF32 ? (NB <= 4 ? 2 : 1) : NB <= 2 ? 3 : NB <= 4 ? 2 : 1;
};

// (heads of 65 to 96 with the maximum every step: 160 registers, three workgroups a unit, which is what that form is for)
template <typename S, int NB, bool VEC, int RB, int KG, bool LAZY>
__global__ __launch_bounds__((Shape<S, NB, RB, KG>::kThreads),
                             (NB == 3 && KG == 1 && !LAZY && !Shape<S, NB, RB, KG>::kF32 ? 3 : Shape<S, NB, RB, KG>::kOccupancy))
void general_chunk_kernel(GeneralArgs p) {
  typedef Shape<S, NB, RB, KG> X;
  typedef typename Store<S>::E E;
  constexpr int MB = X::MB, kKeys = X::kKeys, kPieces = X::kPieces, kTileRows = X::kTileRows;
  constexpr int kQ = X::kPiecesRow / 2;      // query registers: pieces 2 s + g of the row
  constexpr float kShift = Store<S>::kShift;
  __shared__ __attribute__((aligned(16))) uint8_t smem[X::kLds];
  __shared__ uint32_t s_bad;                 // a value beyond the first row's position is not finite

  const int tid = threadIdx.x % X::kGroupThreads, lane = tid & 63;   // within the key group
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t kg = KG == 1 ? 0u : (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / X::kGroupThreads));
  const int j = lane & 31, g = lane >> 5;
  const uint32_t planes = gridDim.x / p.row_tiles;
  const uint32_t plane = blockIdx.x % planes;
  // longest rows first; the second workgroup of every unit, where two are resident and there are no
  // more, in the opposite order, so that the unit with the longest gets the shortest
  uint32_t order = blockIdx.x / planes;
  if (order >= p.turn_at) order = p.row_tiles - 1 - (order - p.turn_at);
  const uint32_t tile = p.row_tiles - 1 - order;
  const uint32_t seq = plane / p.n_kv_heads, kvh = plane % p.n_kv_heads;
  const uint32_t P0 = start_position(p, seq);
  const uint32_t row0 = tile * kTileRows;
  const uint32_t last_row = min(p.rows, row0 + kTileRows) - 1;
  const uint32_t k0 = blockIdx.y * p.split_len;
  // keys [k0, end): up to the last row's position, and to the end of this split
  const uint32_t end = min(P0 + last_row / p.group + 1, k0 + p.split_len);
  if (k0 >= end) return;   // (the merge derives the live splits the same way)
  const uint32_t first_pos = P0 + row0 / p.group;
  const uint32_t n_steps = (end - k0 + kKeys - 1) / kKeys;

  const uint32_t r = row0 + 32 * wave + j;
  const bool row_valid = r < p.rows;
  const uint32_t rc = row_valid ? r : last_row;
  const uint32_t rowpos = P0 + rc / p.group;
  const uint32_t wave_row0 = min(row0 + 32u * wave, last_row), wave_row1 = min(wave_row0 + 31u, last_row);
  const uint32_t wave_first = P0 + wave_row0 / p.group;    // chunks up to here need no mask,
  const uint32_t wave_last = P0 + wave_row1 / p.group;     // chunks past here are not this wave's
  const bool wave_has_rows = __builtin_amdgcn_readfirstlane((int)(row0 + 32u * wave <= last_row));
  // steps of this split that end beyond key x: from this one on
  auto steps_beyond = [&](uint32_t x) { return x + 1 > k0 ? (x + 1 - k0) / kKeys : 0u; };
  auto uniform = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
  const uint32_t wave_steps = uniform(wave_has_rows && wave_last >= k0 ? min(n_steps, (wave_last - k0) / kKeys + 1) : 0u);
  const uint32_t mask_from = uniform(min(steps_beyond(wave_first), (end - k0) / kKeys));   // some pair is masked: by position, or past the end
  const uint32_t look_from = uniform(steps_beyond(first_pos));

  u32x4 qreg[kQ];
  {
    const E* qrow = (const E*)p.q + query_row(p, seq, kvh, rc) * p.head_size;
#pragma unroll
    for (int s = 0; s < kQ; ++s) qreg[s] = query_piece<S, VEC>(p, qrow, (2 * s + g) * Store<S>::kPiece);
  }

  const size_t plane_at = seq_plane_offset(p.seq_offsets, p.kv_stride_seq, seq) + (size_t)kvh * p.kv_stride_head;
  const E* kp = (const E*)p.k + plane_at;
  const E* vp = (const E*)p.v + plane_at;
  const uint64_t kplane = scalar64((uint64_t)kp), vplane = scalar64((uint64_t)vp);
  const uint64_t pos_bytes = (uint64_t)p.kv_stride_pos * sizeof(E);
  const uint64_t valid = scalar64((uint64_t)(end - 1) * pos_bytes + (uint64_t)p.head_size * sizeof(E));
  uint32_t off0[X::kPlaces], lds_k0[X::kPlaces], lds_v0[X::kPlaces];
  const uint32_t lds_all = (uint32_t)(uintptr_t)(LdsByte*)smem, lds0 = lds_all + kg * X::kGroupLds;
#pragma unroll
  for (int i = 0; i < X::kPlaces; ++i) {
    const uint32_t pi = tid + X::kGroupThreads * i, krow = pi / X::kPiecesRow, col = pi % X::kPiecesRow;
    if constexpr (VEC)
      off0[i] = col * Store<S>::kPiece < p.head_size ? (uint32_t)(krow * pos_bytes) + 16 * col : kNowhere;
    else
      off0[i] = krow | col * Store<S>::kPiece << 16;
    lds_k0[i] = lds0 + krow * X::kKPitch + 16 * col;
    lds_v0[i] = lds0 + 2 * X::kKBuf + krow * X::kVPitch + 16 * col;
  }
  // of piece i (a step of 64 keys is at most 2^31 bytes: kNowhere plus its rows stays past every descriptor)
  const uint32_t row_step = VEC ? (uint32_t)(X::kRowStep * pos_bytes) : (uint32_t)X::kRowStep;
  auto off = [&](int i) { return X::kRowStep ? off0[0] + i * row_step : off0[i % X::kPlaces]; };
  auto lds_k = [&](int i) { return X::kRowStep ? lds_k0[0] + i * X::kRowStep * X::kKPitch : lds_k0[i % X::kPlaces]; };
  auto lds_v = [&](int i) { return X::kRowStep ? lds_v0[0] + i * X::kRowStep * X::kVPitch : lds_v0[i % X::kPlaces]; };
  u32x4 kst[kPieces], vst[kPieces];
  auto load_rows = [&](uint32_t step, const E* rows, uint64_t plane_base, u32x4 (&st)[kPieces]) {
    const uint32_t kb = k0 + step * kKeys;
    if constexpr (VEC) {
      const __amdgpu_buffer_rsrc_t rs = chunk_rsrc(plane_base, (uint64_t)kb * pos_bytes, valid);
#pragma unroll
      for (int i = 0; i < kPieces; ++i) st[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, off(i), 0, 0);
    } else {
#pragma unroll
      for (int i = 0; i < kPieces; ++i)
        st[i] = gather_piece<S>(rows, p.kv_stride_pos, kb + (off(i) & 0xffffu), end, off(i) >> 16, p.head_size);
    }
  };
  // (steps are asked for in order: kg, kg + KG, ...)
  uint64_t next_off = scalar64((uint64_t)(k0 + kg * kKeys) * pos_bytes);
  const uint64_t off_step = scalar64((uint64_t)(KG * kKeys) * pos_bytes);
  auto load_step = [&](uint32_t step) {
    if constexpr (VEC && !X::kLateV) {
      const __amdgpu_buffer_rsrc_t kr = chunk_rsrc(kplane, next_off, valid), vr = chunk_rsrc(vplane, next_off, valid);
      next_off += off_step;
#pragma unroll
      for (int i = 0; i < kPieces; ++i) kst[i] = __builtin_amdgcn_raw_buffer_load_b128(kr, off(i), 0, 0);
#pragma unroll
      for (int i = 0; i < kPieces; ++i) vst[i] = __builtin_amdgcn_raw_buffer_load_b128(vr, off(i), 0, 0);
    } else {
      load_rows(step, kp, kplane, kst);
      if constexpr (!X::kLateV) load_rows(step, vp, vplane, vst);
    }
  };
  auto store_rows = [&](uint32_t step, const u32x4 (&st)[kPieces], auto at, int bytes) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) *(LdsU32x4*)(at(i) + (step / KG & 1) * bytes) = st[i];
  };
  auto look_at = [&](uint32_t step) {
    if (step >= look_from) {   // some row of the workgroup must not see some of these values
      asm volatile("");   // (a branch, not a condition: few steps of a walk come here)
      bool bad = false;
#pragma unroll
      for (int i = 0; i < kPieces; ++i) bad |= piece_not_finite<S>(vst[i]);
      if (bad) s_bad = 1;
    }
  };
  auto store_step = [&](uint32_t step) {
    if constexpr (!VEC) {
      const uint32_t kb = k0 + step * kKeys;
#pragma unroll
      for (int i = 0; i < kPieces; ++i) {
        kst[i] = settle_piece<S>(kst[i], kb + (off(i) & 0xffffu), end, off(i) >> 16, p.head_size);
        vst[i] = settle_piece<S>(vst[i], kb + (off(i) & 0xffffu), end, off(i) >> 16, p.head_size);
      }
    }
    store_rows(step, kst, lds_k, X::kKBuf);
    store_rows(step, vst, lds_v, X::kVBuf);
    look_at(step);
  };

  float m_run = -INFINITY, l_run = 0.0f;
  f32x16 oacc[NB];
#pragma unroll
  for (int db = 0; db < NB; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) oacc[db][e] = 0.0f;

  // K as the A operand: key j of a block, the pieces the query registers hold
  const uint32_t k_read = lds0 + j * X::kKPitch + 16 * g;
  // V^T as the A operand: 16-bit through the transposing read (see prefill.hip), binary32 element by
  // element, keys in the order in which the soft-max leaves the weights in registers
  const uint32_t v_read = X::kF32 ? lds0 + 2 * X::kKBuf + 4 * g * X::kVPitch + 4 * j
                                  : lds0 + 2 * X::kKBuf + (4 * g + ((lane & 15) >> 2)) * X::kVPitch +
                                        2 * (16 * ((lane >> 4) & 1) + 4 * (lane & 3));

  // 16-bit: operand n of the second product, keys 16 (n / NB) .., columns 32 (n % NB) ..
  auto v_operand = [&](uint32_t vs, int n) __attribute__((always_inline)) {
    const uint32_t at = vs + 16 * (n / NB) * X::kVPitch + 64 * (n % NB);
    const i16x4 a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4*)at);
    const i16x4 a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4*)(at + 8 * X::kVPitch));
    const u32x2 w0 = __builtin_bit_cast(u32x2, a0), w1 = __builtin_bit_cast(u32x2, a1);
    return u32x4{w0[0], w0[1], w1[0], w1[1]};
  };
  // operand reads ahead of the products (three are what 168 registers hold)
  constexpr int kAheadMax = NB == 3 && KG == 1 && !LAZY ? 3 : 4, kAheadK = kQ * MB < kAheadMax ? kQ * MB : kAheadMax;
  constexpr int kAhead = 2 * MB * NB < kAheadMax ? 2 * MB * NB : kAheadMax;
  auto load_late = [&](uint32_t step) __attribute__((always_inline)) {
    if constexpr (X::kLateV)
      if (step < n_steps) load_rows(step, vp, vplane, vst);
  };
  auto compute = [&](uint32_t step, auto first_) __attribute__((always_inline)) {
    constexpr bool kFirst = decltype(first_)::value;   // the group's first step: no row has a reference maximum yet
    const uint32_t kb = k0 + step * kKeys, buf = step / KG & 1;
    if (step >= wave_steps) {
      load_late(step + KG);
      return;
    }
    const uint32_t ks = k_read + buf * X::kKBuf, vs = v_read + buf * X::kVBuf;
    f32x16 st[MB];
    u32x4 va[2 * MB * NB];
    f32x16 zero;
#pragma unroll
    for (int e = 0; e < 16; ++e) zero[e] = 0.0f;
    if constexpr (X::kF32) {
      // Eight products a chain, chains added up in kTotals sums.  A matrix instruction keeps the pipe
      // busy for 64 cycles: a quarter of the additions of the chain before goes behind each of them.
      constexpr int kTotals = NB <= 2 ? 4 : 2;   // (what the registers hold)
      f32x16 total[kTotals], before;
      u32x4 a = *(const LdsU32x4*)ks;
      static_for<kQ + 1>([&](auto s_) __attribute__((always_inline)) {
        constexpr int s = decltype(s_)::value;
        u32x4 next;
        if constexpr (s + 1 < kQ) next = *(const LdsU32x4*)(ks + 32 * (s + 1));
        f32x16 sum = zero;
        static_for<4>([&](auto e_) __attribute__((always_inline)) {
          constexpr int e = decltype(e_)::value;
          if constexpr (s < kQ)
            sum = __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_bit_cast(float, (uint32_t)a[e]),
                                                       __builtin_bit_cast(float, (uint32_t)qreg[s][e]), sum, 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (s > 0) {
#pragma unroll
            for (int x = 4 * e; x < 4 * e + 4; ++x) {
              if constexpr (s <= kTotals) total[(s - 1) % kTotals][x] = before[x];
              else total[(s - 1) % kTotals][x] += before[x];
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        });
        before = sum;
        if constexpr (s + 1 < kQ) a = next;
      });
      auto each = [&](auto n_) { return total[decltype(n_)::value]; };
      st[0] = pairwise_sum<0, kTotals>(each);
    } else {
      // (operands a few reads ahead of their products; those of the second product, as far as they fit the registers the
      // first one's leave, ahead of the soft-max, which their way out of LDS then lies behind)
      u32x4 ka[kQ * MB];
      auto k_operand = [&](int n) { return (u32x4) * (const LdsU32x4*)(ks + 32 * (n % MB) * X::kKPitch + 32 * (n / MB)); };
#pragma unroll
      for (int n = 0; n < kAheadK; ++n) ka[n] = k_operand(n);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < kQ * MB; ++n) {
        st[n % MB] = Mfma<S>::m32x32x16(ka[n], qreg[n / MB], n < MB ? zero : st[n % MB]);
        if (n + kAheadK < kQ * MB) ka[n + kAheadK] = k_operand(n + kAheadK);
      }
#pragma unroll
      for (int n = 0; n < kAhead; ++n) va[n] = v_operand(vs, n);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (step >= mask_from) {   // some pair of the step is masked
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const uint32_t key = kb + 32 * mb + 8 * (e >> 2) + 4 * g + (e & 3);
          st[mb][e] = (key <= rowpos && key < end) ? st[mb][e] : -INFINITY;
        }
    }
    load_late(step + KG);
    // LAZY (16-bit storage, heads up to 128): exponentials against the reference maximum the row already has, and
    // its true maximum looked for only where a lane's sum of them passes Mfma<S>::kMaxSum (below).  Else (wider heads
    // keep their pipe busy with products, binary32 its own way to add up, and chunk_max_first() says where heads of 65
    // to 96 are better off) the maximum first, every step.
    // Maximum first -> here (us): 2048 tokens, 32 / 8 heads of 64, bf16 42.0 -> 40.0; 1500 on 300, 32 / 4 of 80 57.0 ->
    // 52.2; 400 x 3 on 1000, 32 / 8 of 96 49.1 -> 45.5; heads of 192 and 256 1.3 % slower.  Short walks gain or lose
    // nothing (300 x 2, 32 / 8 of 80 11.0 -> 11.0, of 32 7.7 -> 7.6; 119 x 3 on 125, 32 / 32 of 64 7.4 -> 7.4), but only
    // because a group's first step, when no row has a reference, goes to the maximum at once: with a pass over
    // the weights before it they took 2 to 5 % longer (11.5, 8.0, 7.5).
    float neg_m = kShift - m_run;
    if constexpr (!LAZY) {
      float rmax = st[0][0];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int e = 0; e < 16; ++e) rmax = fmaxf(rmax, st[mb][e]);
      rmax = max_with_partner_half(rmax);
      const float tmax = rmax * p.c;
      const bool grow = tmax > m_run + kRescaleStep;
      if (__any(grow)) {
        const float m_new = grow ? tmax : m_run;
        const float alpha = grow ? fast_exp2(m_run - m_new) : 1.0f;
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int db = 0; db < NB; ++db) oacc[db] *= alpha;
      }
      neg_m = (m_run == -INFINITY) ? 0.0f : kShift - m_run;
    }
    float psum = 0.0f;
    if constexpr (X::kF32) {
#pragma unroll
      for (int e = 0; e < 16; ++e) st[0][e] = fast_exp2(__builtin_fmaf(st[0][e], p.c, neg_m));
      auto weight = [&](auto e_) { return st[0][decltype(e_)::value]; };
      psum = pairwise_sum<0, 16>(weight);
      // chains of eight keys, added up likewise: a block's four chains, then their sum to the row's
      f32x16 before, block;
      float v[4];
      auto rows_of = [&](int n, float (&to)[4]) __attribute__((always_inline)) {   // chain n: block n / 4, keys 8 (n % 4) ..
#pragma unroll
        for (int e = 0; e < 4; ++e) to[e] = *(const LdsF32*)(vs + (8 * (n & 3) + e) * X::kVPitch + 128 * (n >> 2));
      };
      rows_of(0, v);
      static_for<4 * NB + 2>([&](auto n_) __attribute__((always_inline)) {
        constexpr int n = decltype(n_)::value, done = n - 1;   // (the chain before)
        float next[4];
        if constexpr (n + 1 < 4 * NB) rows_of(n + 1, next);
        f32x16 sum = zero;
        static_for<4>([&](auto e_) __attribute__((always_inline)) {
          constexpr int e = decltype(e_)::value;
          if constexpr (n < 4 * NB) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(v[e], st[0][4 * (n & 3) + e], sum, 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int x = 4 * e; x < 4 * e + 4; ++x) {
            if constexpr (done > 0 && done % 4 == 0) oacc[done / 4 - 1][x] += block[x];
            if constexpr (done >= 0 && done < 4 * NB) block[x] = done % 4 == 0 ? before[x] : block[x] + before[x];
          }
          __builtin_amdgcn_sched_barrier(0);
        });
        before = sum;
        if constexpr (n + 1 < 4 * NB)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = next[e];
      });
    } else {
      f32x16 w[MB];
      auto weigh = [&](int cc, float shift) __attribute__((always_inline)) {   // keys 16 cc .. + 15
#pragma unroll
        for (int e = 8 * (cc & 1); e < 8 * (cc & 1) + 8; e += 2) {
          w[cc >> 1][e] = fast_exp2(__builtin_fmaf(st[cc >> 1][e], p.c, shift));
          w[cc >> 1][e + 1] = fast_exp2(__builtin_fmaf(st[cc >> 1][e + 1], p.c, shift));
          psum += w[cc >> 1][e] + w[cc >> 1][e + 1];
        }
      };
      if constexpr (LAZY && !kFirst) {
#pragma unroll
        for (int cc = 0; cc < 2 * MB; ++cc) weigh(cc, neg_m);
      }
      if constexpr (LAZY) {
        // (a row without a reference makes its sum infinite or NaN; a row moves by what its own two lanes saw)
        const uint64_t over = kFirst ? ~(uint64_t)0 : __ballot(!(psum <= Mfma<S>::kMaxSum));
        if (over) {
          float rmax = st[0][0];
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int e = 0; e < 16; ++e) rmax = fmaxf(rmax, st[mb][e]);
          rmax = max_with_partner_half(rmax);
          const bool moves = (((over >> j) | (over >> j >> 32)) & 1) != 0;
          const float m_new = moves ? fmaxf(m_run, rmax * p.c) : m_run;
          const float alpha = m_new == m_run ? 1.0f : fast_exp2(m_run - m_new);
          m_run = m_new;
          l_run *= alpha;
#pragma unroll
          for (int db = 0; db < NB; ++db) oacc[db] *= alpha;
          neg_m = (m_run == -INFINITY) ? 0.0f : kShift - m_run;
          psum = 0.0f;
#pragma unroll
          for (int cc = 0; cc < 2 * MB; ++cc) weigh(cc, neg_m);
        }
      }
      u32x4 hi[2 * MB], lo[2 * MB];
      auto split = [&](int cc) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const int e = 8 * (cc & 1) + 2 * x;
          uint32_t h, l;
          split_pair<S>(w[cc >> 1][e], w[cc >> 1][e + 1], h, l);
          hi[cc][x] = h;
          lo[cc][x] = l;
        }
      };
      auto product = [&](int n, const u32x4& weights) __attribute__((always_inline)) {
        oacc[n % NB] = Mfma<S>::m32x32x16(va[n], weights, oacc[n % NB]);
      };
      auto more_operands = [&](int n) __attribute__((always_inline)) {
        if (n + kAhead < 2 * MB * NB) va[n + kAhead] = v_operand(vs, n + kAhead);
      };
      if constexpr (NB <= kAhead) {
        // sixteen keys at a time: their products run beside the splitting of the next ones' weights, and none waits for
        // the one before it
#pragma unroll
        for (int cc = 0; cc < 2 * MB; ++cc) {
          if constexpr (!LAZY) weigh(cc, neg_m);
          split(cc);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int n = NB * cc; n < NB * cc + NB; ++n) product(n, hi[cc]);
#pragma unroll
          for (int n = NB * cc; n < NB * cc + NB; ++n) {
            product(n, lo[cc]);
            more_operands(n);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {   // (wide heads have products enough: in that order 2 to 8 % slower)
#pragma unroll
        for (int cc = 0; cc < 2 * MB; ++cc) {
          weigh(cc, neg_m);
          split(cc);
        }
#pragma unroll
        for (int n = 0; n < 2 * MB * NB; ++n) {
          product(n, hi[n / NB]);
          product(n, lo[n / NB]);
          more_operands(n);
        }
      }
    }
    l_run += psum;
  };

  // step s of the keys belongs to group s mod KG; every group passes every barrier
  if (threadIdx.x == 0) s_bad = 0;
  if (kg < n_steps) load_step(kg);
  load_late(kg);
  __syncthreads();
  if (kg < n_steps) store_step(kg);
  if (kg + KG < n_steps) load_step(kg + KG);
  __syncthreads();
  auto turn = [&](uint32_t step, auto first) __attribute__((always_inline)) {
    compute(step, first);
    if (step + KG < n_steps) {
      store_step(step + KG);
      if (step + 2 * KG < n_steps) load_step(step + 2 * KG);
    }
    __syncthreads();
  };
  // (the first turn apart where it skips a pass over the weights: a branch in the loop costs 2048 tokens 1.5 %)
  if constexpr (LAZY) turn(kg, std::true_type{});
  for (uint32_t first = LAZY ? KG : 0; first < n_steps; first += KG) turn(first + kg, std::false_type{});

  const size_t part_row0 = (size_t)plane * p.rows;
  if (s_bad) {   // (uniform: the last barrier is behind every write of it)
    for (uint32_t rr = row0 + kg * RB + wave; rr <= last_row; rr += X::kWaves)
      plain_row<S>(p, kp, vp, query_row(p, seq, kvh, rr), (part_row0 + rr) * p.n_split + blockIdx.y, k0,
                   min(end, P0 + rr / p.group + 1), X::kHead, p.n_split > 1, (int)lane_number());
    return;
  }
  // the groups' rows: the upper half of the groups hands its own over, until one group is left
#pragma unroll
  for (int groups = KG; groups > 1; groups = (groups + 1) / 2) {
    const uint32_t half = (groups + 1) / 2, pairs = groups - half;
    const bool gives = kg >= half && kg < (uint32_t)groups, takes = kg < pairs;
    const uint32_t slot = (gives ? kg - half : kg) * RB + wave;
    const uint32_t at = lds_all + slot * X::kMergeWave + 16 * lane;
    const uint32_t ml = lds_all + pairs * RB * X::kMergeWave + slot * (2 * kWave * 4) + 8 * lane;
    if (gives) {
#pragma unroll
      for (int db = 0; db < NB; ++db)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4)
          *(LdsF32x4*)(at + (4 * db + q4) * (16 * kWave)) =
              f32x4{oacc[db][4 * q4], oacc[db][4 * q4 + 1], oacc[db][4 * q4 + 2], oacc[db][4 * q4 + 3]};
      *(LdsF32x2*)ml = f32x2{m_run, l_run};
    }
    __syncthreads();
    if (takes) {
      const f32x2 other = *(const LdsF32x2*)ml;
      const float m_new = fmaxf(m_run, other[0]);
      const float wa = m_run == -INFINITY ? 0.0f : fast_exp2(m_run - m_new);
      const float wb = other[0] == -INFINITY ? 0.0f : fast_exp2(other[0] - m_new);
      m_run = m_new;
      l_run = l_run * wa + other[1] * wb;
#pragma unroll
      for (int db = 0; db < NB; ++db)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const f32x4 o = *(const LdsF32x4*)(at + (4 * db + q4) * (16 * kWave));
#pragma unroll
          for (int e = 0; e < 4; ++e) oacc[db][4 * q4 + e] = oacc[db][4 * q4 + e] * wa + o[e] * wb;
        }
    }
    if (groups > 2) __syncthreads();
  }
  if (KG > 1 && kg != 0) return;
  const float l = sum_with_partner_half(l_run);
  // Sums that are not finite: an infinite value under a weight in two operands, or weights above one (up to
  // 2^8 in bfloat16) on values less than that below the largest number.
  float top[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int db = 0; db < NB; ++db)
#pragma unroll
    for (int e = 0; e < 16; e += 2) top[e >> 2] = largest_of(top[e >> 2], oacc[db][e], oacc[db][e + 1]);
  if (__any(not_finite_sum(largest_of(top[0], top[1], largest_of(top[2], top[3], 0.0f)), l))) {
    for (uint32_t rr = row0 + 32 * wave; rr < min(row0 + 32 * wave + 32, last_row + 1); ++rr)
      plain_row<S>(p, kp, vp, query_row(p, seq, kvh, rr), (part_row0 + rr) * p.n_split + blockIdx.y, k0,
                   min(end, P0 + rr / p.group + 1), X::kHead, p.n_split > 1, (int)lane_number());
    return;
  }
  // (the lane's row again, from the lane's number: kept through the loop it costs registers that are not there)
  const uint32_t lane_again = lane_number(), g_again = lane_again >> 5, r_again = row0 + 32 * wave + (lane_again & 31);
  if (r_again >= p.rows) return;
  const size_t row_again = query_row(p, seq, kvh, r_again);
  if (p.n_split > 1) {
    const size_t part = (part_row0 + r_again) * p.n_split + blockIdx.y;
    float* orow = p.part_o + part * X::kHead;
#pragma unroll
    for (int db = 0; db < NB; ++db)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        *(f32x4*)(orow + 32 * db + 8 * q4 + 4 * g_again) =
            f32x4{oacc[db][4 * q4], oacc[db][4 * q4 + 1], oacc[db][4 * q4 + 2], oacc[db][4 * q4 + 3]};
    if (g_again == 0) *(float2*)(p.part_ml + part * 2) = float2{m_run == -INFINITY ? m_run : m_run - kShift, l};
  } else {
    const float inv = 1.0f / l;
#pragma unroll
    for (int db = 0; db < NB; ++db)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        store_out4<S, VEC>(p, row_again, 32 * db + 8 * q4 + 4 * g_again,
                           f32x4{oacc[db][4 * q4] * inv, oacc[db][4 * q4 + 1] * inv, oacc[db][4 * q4 + 2] * inv,
                                 oacc[db][4 * q4 + 3] * inv});
    if (p.lse && g_again == 0) p.lse[row_again] = (m_run - kShift + fast_log2(l)) * kLn2;
  }
}

}  // namespace

hipError_t launch_general_chunk(const GeneralArgs& p, int dtype, int nb, bool vec, uint32_t planes, hipStream_t stream) {
  const dim3 grid(planes * p.row_tiles, p.n_split);
  return with_head_blocks(nb, vec, [&](auto n, auto v) {
    constexpr int NB = decltype(n)::value;
    constexpr bool VEC = decltype(v)::value;
    auto go = [&](auto storage) {
      typedef decltype(storage) S;
      constexpr int kLong = chunk_key_groups(std::is_same<S, F32>::value, NB, 4);
      // (one key group: not with heads up to 64, whose walks are two steps then, and with NB 3 as the plan says)
      constexpr bool kLazy = !std::is_same<S, F32>::value && NB <= 4;
      constexpr int kShort = chunk_key_groups(std::is_same<S, F32>::value, NB, 2);
      if constexpr (kShort > 1)
        if (p.tile_rows == 64) {
          hipLaunchKernelGGL((general_chunk_kernel<S, NB, VEC, 2, kShort, kLazy>), grid, dim3(128 * kShort), 0, stream, p);
          return hipGetLastError();
        }
      if constexpr (kLong > 1)
        if (p.key_groups > 1) {
          hipLaunchKernelGGL((general_chunk_kernel<S, NB, VEC, 4, kLong, kLazy>), grid, dim3(256 * kLong), 0, stream, p);
          return hipGetLastError();
        }
      if constexpr (NB == 3 && kLazy)
        if (p.max_first) {
          hipLaunchKernelGGL((general_chunk_kernel<S, NB, VEC, 4, 1, false>), grid, dim3(256), 0, stream, p);
          return hipGetLastError();
        }
      hipLaunchKernelGGL((general_chunk_kernel<S, NB, VEC, 4, 1, (kLazy && NB > 2)>), grid, dim3(256), 0, stream, p);
      return hipGetLastError();
    };
    return dtype == 0 ? go(F16{}) : dtype == 1 ? go(BF16{}) : go(F32{});
  });
}

}  // namespace gen
}  // namespace ellm
