// MFMA tile kernel for paged prefill / chunked extend attention at head_dim 256 on gfx950.
// Replaces paged_prefill_attention<bfloat16, 256, 256>
// (mini-sglang-mlx-kernel/csrc/paged_prefill_attention.metal:382-640, instantiated at :647).
//
// Same products and data path as the head_dim 128 kernel (S^T = K Q^T and O^T += V^T P^T on
// mfma 32x32x16 with rows on N, K and V rows moved HBM -> LDS by global_load_lds, V^T operands
// from row-major V through ds_read_b64_tr_b16), re-cut for 512-byte rows:
//   workgroup  = 8 waves, two per SIMD, 128 rows of one (request, kv head), row = q_idx * group + head.
//                Two waves share 32 rows: each takes half of a step's 64 keys for the scores and half of the
//                dims for the output (64 registers of output tile, 64 of Q operand), and gets the other's row
//                maxima and P through LDS.
//   stage      = 32 keys.  One LDS-direct load moves two whole rows (lanes 0..31 one key,
//                lanes 32..63 the key 16 further on); unit u of a stage holds keys u and u + 16,
//                units sit 1040 B (K) or 1088 B (V) apart so that what LDS serves at a time (lanes
//                0-3, 12-15, 20-27 and so on of a 16-byte read, 32 lanes of an 8-byte one) falls into
//                different banks.  Four K stages and four V stages of LDS.
//   pipeline   = one step per 64 keys: the matrix pipe computes the scores of step i+1 and adds P V of
//                step i-1 (32 MFMAs a wave) while the VALU turns the scores of step i into P.
//                K of step i+2 and V of step i leave in the first half of step i and are waited for at its
//                end, where the workgroup barrier publishes them.
//   slot ids   = fetched a step ahead by loads issued before the step's moves and hidden from
//                the compiler's wait bookkeeping, so that the wait at the end of the step covers them and
//                nothing else waits.
// What bounds it: 32 keys take 1690-1770 cycles, of which the matrix pipe is busy 1024, at the 1.9 GHz that the
// power leaves (1.04 PFLOP/s on the requests below; 1.16 on one long request, where the kernel for head_dim 128
// reaches 1.23).  Whole rows to a wave, for comparison:
// one wave of 32 rows per SIMD issued 400 instructions per 32 keys at 5 cycles each (2380 cycles), two of 16 rows
// read K and V twice as often from LDS (2050).  4 requests of 512-1972 tokens on prefixes up to 8 K, 24 / 4
// heads: 837 us with the first, 775 with the second, 717 so.
// Beside its steps a block pays for its start: with Q by way of LDS, each row once, and no products for nothing in the
// first step 8 K cycles less than before: 23 prompts of 129-1833 tokens, 16 / 4 heads, 434 -> 397 us, 60 of up to 400
// 139 -> 125, 30 x 10-400 on up to 500 cached, 24 / 4, 150 -> 135, 9 x 700-2329 under a window of 300 196 -> 175.
// Where the workgroup stays (STAY, see kMinHalfRounds256) the next block's slot ids are under way while the last one's P V
// is added, its K and Q while the result is stored, straight from the registers: 12 K cycles from step to step.  There
// are no registers to go on from block to block as in the head_dim 128 kernel (256 in the steps, 22 of a lane's constants
// spilled around them), nor for steps that leave the scores of a block's last step out (105 spilled in them).
//
// Algorithmic flops: 4 * D per visible (query, key) pair and q head (QK^T + PV).
#include <type_traits>

#include "msgl_device.h"
#include "msgl_internal.h"
#include "prefill_params.h"
#include "prefill_tile_common.h"

namespace msgl {
namespace {

constexpr int kD = 256;
constexpr int kHalf = 32;                     // keys per stage
constexpr int kStep = 2 * kHalf;              // keys per pipeline step
constexpr int kNW = 8;                        // waves per workgroup
constexpr int kUnits = 16;                    // LDS-direct loads per stage (two 512-byte rows each)
constexpr int kUPW = kUnits / kNW;            // units each wave moves per stage: 2
constexpr int kGroups = kNW / 2;              // groups of 32 rows, two waves each
constexpr int kKUnit = 1024 + 16;             // bytes between K units
constexpr int kVUnit = 1024 + 64;             // bytes between V units
constexpr int kKStage = kUnits * kKUnit;      // 16640
constexpr int kVStage = kUnits * kVUnit;      // 17408
constexpr int kKStages = 4, kVStages = 4;
constexpr int kVBase = kKStages * kKStage;
constexpr int kPBase = kVBase + kVStages * kVStage;       // P of a step: 2 KB per wave
constexpr int kMaxBase = kPBase + kNW * 2048;             // row maxima: 256 B per wave
constexpr int kStageTotal = kMaxBase + kNW * 256;         // 154624
constexpr int kKSteps = kD / 16;              // k-steps of QK^T
constexpr int kDT = kD / 2 / 32;              // 32-dim tiles of a wave's half of O^T

// STAY: the workgroup takes the blocks of its list (see kMaxRounds), one after the other.
template <bool WIDE, bool STAY>
__global__ __launch_bounds__(kNW * 64) void prefill_tile256_kernel(PrefillParams p) {
  constexpr int kRows = kPrefillBlockRows256;
  static_assert(kRows == kGroups * 32, "one 32-row tile per two waves");
  constexpr int OROW = kD + 8;
  constexpr int O_BYTES = kRows * OROW * 2;
  constexpr int SMEM_BYTES = kStageTotal > O_BYTES ? kStageTotal : O_BYTES;
  __shared__ __attribute__((aligned(16))) unsigned char smem[SMEM_BYTES];
  using OffT = typename std::conditional<WIDE, uint64_t, uint32_t>::type;
  __shared__ BlockList list;
  const ClockProbe clock_probe_(p.clock_probe);

  const int tid = threadIdx.x;
  if constexpr (!STAY)
    if (store_rows_of_no_request<kNW * 64>(p, p.nt, p.n_kv * kD, tid)) return;
  auto uniform = [](int x) { return __builtin_amdgcn_readfirstlane(x); };  // the same in every lane: a scalar
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int h = lane >> 5;
  const int c32 = lane & 31;
  const int group_row = 32 * (w % kGroups);  // the first of the wave's 32 rows
  const int f = w / kGroups;                 // its half: of the keys of a step for the scores, of the dims for the output

  // ---- block -> (request, kv head, key split, q block): consecutive block ids go to different
  // XCDs, the q blocks of one (request, kv head, key split) read the same keys, share an XCD and
  // run heaviest first, requests in order of decreasing kv length (each block ranks the requests
  // itself from kv_indptr)
  // With ragged shares: block -> (unit = (request, share), kv head), see prefill_ragged_tiles().
  int b, kvh, split = 0, qblk, n_shares = 1, n_listed = 1;
  bool to_partial = p.n_ksplit > 1;  // leave a partial for the merge kernel, not the result
  int64_t part_at = 0;               // partial row of the block's row 0 (ragged shares)
  LengthBlock by_length{};
  RequestPlace place{};
  if constexpr (STAY) {
    n_listed = list_blocks<kNW * 64, kRows, kHalf>(p, list, tid);
    n_listed = drop_blank_blocks<kNW * 64, kD, kRows>(p, list, n_listed, tid);
    if (n_listed == 0) return;
    kvh = uniform(list.block[0].kvh);  // of all the XCD's blocks
    b = qblk = 0;                      // the list has them
  } else if (p.ragged_tiles > 0) {
    kvh = (int)(blockIdx.x % (unsigned)p.n_kv);
    const int u = (int)(blockIdx.x / (unsigned)p.n_kv);
    place = place_of<kNW * 64>(p, u, tid);
    if (!place.ok) return;
    const RaggedUnit& ru = place.unit;
    b = place.b;
    split = ru.share;
    qblk = 0;
    n_shares = ru.count;
    to_partial = ru.count > 1;
    part_at = ((int64_t)u * p.n_kv + kvh) * p.ragged_rows;
    if (ru.share == 0 && kvh == 0 && tid == 0 && p.req_units != nullptr) {
      p.req_units[2 * b] = ru.first;  // tells the merge kernel where the request's partials are
      p.req_units[2 * b + 1] = ru.count;
    }
  } else if (p.length_heads > 0) {
    by_length = LengthOrder<kRows>(p).find((int)(blockIdx.x >> 3));
    if (!by_length.ok) return;
    b = by_length.b;
    kvh = by_length.kvh;
    qblk = by_length.qblk;
  } else {
    const BlockWork work = prefill_block_work(p);
    if (!work.ok) return;
    const int pair = work.unit / p.n_ksplit;  // unit = (request, kv head, key split)
    split = work.unit - pair * p.n_ksplit;
    qblk = work.qblk;
    const int want_rank = pair / p.n_kv;
    kvh = pair - want_rank * p.n_kv;
    place = place_of<kNW * 64>(p, want_rank, tid);
    b = place.b;
  }

  int q_start, q_len, kv_start, kn, prefix, k_lo, k_hi;
  auto take_listed = [&](int i) {
    const ListedBlock& l = list.block[i];
    q_start = uniform(l.q_start);
    q_len = uniform(l.q_len);
    kv_start = uniform(l.kv_start);
    kn = uniform(l.kv_len);
    prefix = uniform(l.prefix);
    qblk = uniform(l.qblk);
    k_lo = uniform(l.k_lo);
    k_hi = uniform(l.k_hi);
  };
  if constexpr (STAY) {
    take_listed(0);
  } else if (by_length.ok) {  // they came with the block
    q_start = by_length.q_start;
    q_len = by_length.q_len;
    kv_start = by_length.kv_start;
    kn = by_length.kv_len;
    prefix = by_length.prefix;
  } else {
    q_start = uniform(place.q_start);
    q_len = min(uniform(place.q_len), p.max_len_extend);
    kv_start = uniform(place.kv_start);
    kn = uniform(place.kv_len);
    prefix = uniform(place.prefix);
  }
  int rows_total = q_len * p.group;
  int row0 = qblk * kRows;
  if constexpr (!STAY) {
    if (row0 >= rows_total) return;
    if (p.nt.out_loc != nullptr) store_request_rows<kNW * 64, kD>(p, q_start, uniform(place.q_len), kvh, tid);
    block_keys<kRows, kHalf>(p, prefix, kn, row0, rows_total, &k_lo, &k_hi);
    // key split `split` of n_ksplit: a whole number of steps each, the last takes the ragged end;
    // shares past the end are empty (they still leave a "nothing seen" partial)
    if (p.ragged_tiles > 0 || p.n_ksplit > 1) {
      const int shares = p.ragged_tiles > 0 ? n_shares : p.n_ksplit;  // ragged: the request's own count
      const int all_steps = (k_hi - k_lo + kStep - 1) / kStep;
      const int share = (all_steps + shares - 1) / shares * kStep;
      k_lo = min(k_lo + split * share, k_hi);
      k_hi = min(k_hi, k_lo + share);
    }
  }
  // a half past the end reads clamped keys and is fully masked
  int n_steps = (k_hi - k_lo + kStep - 1) / kStep;

  // ---- this lane's row: visibility bounds -----------------------------------------------
  int row_lo, row_hi;
  int w_lo_max, w_hi_min;
  auto row_bounds = [&] {
    int lane_row = c32;  // anew, see move_q()
    asm volatile("" : "+v"(lane_row));
    const int row = row0 + group_row + lane_row;
    const bool valid = row < rows_total;
    const int qpos = prefix + (valid ? row_to_query(p, row) : 0);
    row_lo = (p.window > 0) ? qpos - p.window + 1 : 0;
    // k_hi - 1 only binds under a key split: the pipeline settles one step past its share
    row_hi = min(p.is_cross ? kn - 1 : min(qpos, kn - 1), k_hi - 1);
    w_lo_max = valid ? row_lo : -0x7fffffff;
    w_hi_min = valid ? row_hi : 0x7fffffff;
    if (!valid) {
      row_lo = 1;
      row_hi = 0;
    }
    w_lo_max = wave_max(w_lo_max);
    w_hi_min = wave_min(w_hi_min);
  };

  f32x16_t oacc[kDT];
  float m_run, l_run;
  auto reset = [&] {
#pragma unroll
    for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) oacc[dt][i] = 0.f;
    m_run = kNegInf;
    l_run = 0.f;
  };
  reset();

  // ---- moving a stage: wave w owns units 2w, 2w+1; in a unit, lane l fetches 16-byte chunk
  // l % 32 of key (unit + 16 (l / 32)) ----------------------------------------------------
  const uint32_t lds0 = (uint32_t)(uintptr_t)MSGL_LDS_PTR(unsigned char, smem);
  kvh = uniform(kvh);
  const unsigned char* k_src = reinterpret_cast<const unsigned char*>(p.k_cache + (int64_t)kvh * kD);
  const unsigned char* v_src = reinterpret_cast<const unsigned char*>(p.v_cache + (int64_t)kvh * kD);
  const uint32_t k_row_bytes = (uint32_t)p.k_stride0 * 2u;
  const uint32_t v_row_bytes = (uint32_t)p.v_stride0 * 2u;
  const uint32_t chunk_off = (uint32_t)(lane & 31) * 16u;
  // Slot ids of a half: lane l wants the ids of keys 2w, 2w+1 (+16 for the upper half of the
  // wave).  They are fetched by vector loads the compiler does not see (it would answer the
  // first use of their result with a wait for every load in flight, the moves included); the
  // caller's next wait, which names the result registers, makes them valid.  One 8-byte
  // load when the half lies inside the request, element-wise clamped loads on its last,
  // partial half.
  const int32_t* idx_ptr;
  const int lane_key = w * kUPW + 16 * (lane >> 5);
  auto slot_load = [&](int base, u32x2_t& sl) {
    const int first = base + lane_key;
    if (base + (kNW - 1) * kUPW + 16 + kUPW <= kn) {  // uniform: the whole half is in range
      const uint32_t off = (uint32_t)first * 4u;
      asm volatile("global_load_dwordx2 %0, %1, %2" : "=v"(sl) : "v"(off), "s"(idx_ptr) : "memory");
    } else {
      uint32_t e[kUPW];
#pragma unroll
      for (int i = 0; i < kUPW; ++i) {
        const uint32_t off = (uint32_t)min(first + i, kn - 1) * 4u;
        asm volatile("global_load_dword %0, %1, %2" : "=v"(e[i]) : "v"(off), "s"(idx_ptr) : "memory");
      }
      sl = u32x2_t{e[0], e[1]};
    }
  };
  // slot ids are clamped to the pool before they become addresses: an id that is out of range
  // (or stale) then reads a wrong row instead of faulting
  auto lane_offset = [&](uint32_t slot, uint32_t row_bytes) -> OffT {
    slot = min(slot, p.max_slot);
    if constexpr (WIDE) return (uint64_t)slot * row_bytes + chunk_off;
    else return __umul24(slot, row_bytes) + chunk_off;  // both factors below 2^24 here
  };
  // slot ids of the two halves whose K leaves in this step, and of those whose V leaves in it
  // (`v_slot[parity]`: the ids those halves' K left with two steps ago)
  uint32_t k_slot[2][kUPW], v_slot[2][2][kUPW];
  auto move_k = [&](int half, int n, uint32_t slot) {
    lds_direct_b128(lds0 + (uint32_t)(half & 3) * kKStage + (uint32_t)(w * kUPW + n) * kKUnit, k_src, lane_offset(slot, k_row_bytes));
  };
  auto move_v = [&](int half, int n, uint32_t slot) {
    lds_direct_b128(lds0 + kVBase + (uint32_t)(half & 3) * kVStage + (uint32_t)(w * kUPW + n) * kVUnit, v_src,
                    lane_offset(slot, v_row_bytes));
  };

  // per-lane LDS read offsets inside a stage
  //   K operand of MFMA row c32 (key c32 of the half): unit c32 % 16, row c32 / 16
  const uint32_t k_lane = (uint32_t)(c32 & 15) * kKUnit + (uint32_t)(c32 >> 4) * 512u + (uint32_t)h * 16u;
  //   V^T operand: group lane/16 reads dims 16 ((lane/16) % 2) .. +15 of the wave's half, keys 4h .. 4h+3 (+8)
  const uint32_t v_lane = (uint32_t)(4 * h + ((lane & 15) >> 2)) * kVUnit + (uint32_t)f * 256u +
                          (uint32_t)((lane >> 4) & 1) * 32u + (uint32_t)(lane & 3) * 8u;
  const unsigned char* const k_smem = smem + k_lane;
  // The block's Q rows, in front of its first V, in the V stages: 32 rows lie like 32 keys of K.  (Every wave its rows from
  // memory into registers is 32 bytes each of 32 rows a load, and every row twice: 6 K cycles a block.)  Rows past the
  // request's last: the last again, never stored.
  auto move_q = [&] {
    // the lane's and the wave's numbers are taken anew: what follows from them alone would else be kept through the
    // steps, in registers that those need
    int half_row = h, chunk = (int)chunk_off, wave = w;
    asm volatile("" : "+v"(half_row), "+v"(chunk), "+s"(wave));
    const int qi0 = row_to_query(p, row0);
    const uint16_t* const base = p.q + ((int64_t)(q_start + qi0) * p.n_q + kvh * p.group) * kD;
#pragma unroll
    for (int j = 0; j < 2 * kGroups; ++j) {
      const int unit = 2 * kGroups * wave + j;
      const int row = min(row0 + 32 * (unit >> 4) + (unit & 15) + 16 * half_row, rows_total - 1);
      const int qi = row_to_query(p, row);
      lds_direct_b128(lds0 + kVBase + (uint32_t)unit * kKUnit, base, (uint32_t)((qi - qi0) * p.n_q + row - qi * p.group) * (kD * 2u) + chunk);
    }
  };
  auto q_operand = [&](int kstep) {
    return as_bf16x8(*reinterpret_cast<const u32x4_t*>(k_smem + kVBase + (w % kGroups) * kKStage + kstep * 32));
  };
  const unsigned char* const v_smem = smem + kVBase + v_lane;

  // ---- the pieces of one step -------------------------------------------------------------
  // S^T[key][row]: key = base + 8(i/4) + 4h + i%4, row = c32
  auto k_operand = [&](int half, int kstep) {
    return as_bf16x8(*reinterpret_cast<const u32x4_t*>(k_smem + (half & 3) * kKStage + kstep * 32));
  };
  // keys {16u + 4h + e} and {16u + 8 + 4h + e}, e = 0..3, of the half: the S^T rows that the
  // lane's accumulators 8u .. 8u+7 hold
  auto v_operand = [&](int half, int u, int dt) {
    const unsigned char* vs = v_smem + (half & 3) * kVStage + u * 512 + dt * 64;
    const u32x2_t lo = lds_read_tr16(vs);
    const u32x2_t hi = lds_read_tr16(vs + 8 * kVUnit);
    return as_bf16x8(u32x4_t{lo[0], lo[1], hi[0], hi[1]});
  };
  auto mask_in_place = [&](f32x16_t& s, int base) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = base + 8 * (i >> 2) + 4 * h + (i & 3);
      const float x = s[i] * p.scale_log2e;
      s[i] = (key < row_lo || key > row_hi) ? kNegInf : x;
    }
  };
  const f32x16_t zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  // Softmax state of a step's scores:
  //   mul     factor still to be applied to them: the softmax scale on interior halves (max commutes with a
  //           positive scale), 1 on boundary halves, which are scaled and masked in place
  //   m_safe  the (lazy) running row max the exponentials are taken against
  //   alpha   exp2(previous max - m_safe): what O and l must be multiplied by first
  // Both waves of a group come to the same m_run: each leaves the maximum of its half in LDS before the barrier
  // (`reach`) and takes the other's behind it (`settle`).
  const int other = w ^ kGroups;
  float* const my_max = reinterpret_cast<float*>(smem + kMaxBase + w * 256) + lane;
  const float* const other_max = reinterpret_cast<const float*>(smem + kMaxBase + other * 256) + lane;
  u32x4_t* const my_p = reinterpret_cast<u32x4_t*>(smem + kPBase + w * 2048) + lane;
  const u32x4_t* const other_p = reinterpret_cast<const u32x4_t*>(smem + kPBase + other * 2048) + lane;
  float mul = 0.f, m_own = kNegInf;
  auto reach = [&](f32x16_t& s, bool mask, int base) {
    mul = p.scale_log2e;
    if (mask) {  // boundary half
      asm volatile("" ::: "memory");  // keeps this a branch instead of 32 selects in every step
      mask_in_place(s, base);
      mul = 1.0f;
    }
    float mx = fmaxf(s[0], s[1]);
#pragma unroll
    for (int i = 2; i < 16; ++i) mx = fmaxf(mx, s[i]);
    m_own = max_across<32>(mx * mul);
    *my_max = m_own;
  };
  float m_safe = 0.f, alpha = 1.0f;
  auto settle = [&](float m_other) {
    const float m = fmaxf(m_own, m_other);
    alpha = 1.0f;
    // Usual case: no row's scores are more than kLazy above its reference, and all references stay.
    if (__any(m > m_run + kLazy)) {
      const float m_old = m_run;
      const float m_new = fmaxf(m_old, m);
      const float m_use = (m_new - m_old > kLazy) ? m_new : m_old;
      alpha = fast_exp2(m_old - ((m_use == kNegInf) ? 0.f : m_use));
      m_run = m_use;
    }
    m_safe = (m_run == kNegInf) ? 0.f : m_run;
  };
  // One step over 64 keys.  The 32 MFMAs (a chain of 16 for this wave's scores of step i+1, 16 independent
  // ones adding its dims of P V of step i-1) depend on nothing the VALU does in this step; they are spread over
  // eight slices, 2 + 2 each, and each slice requests the LDS operands of the next.  The VALU turns the
  // scores of step i into bf16 P and the row sum.  P V takes the wave's own half of the keys first, then the
  // other wave's, whose P comes from LDS.  Between slices 5 and 6 a barrier: every wave has its copy of the other's
  // P of step i-1, and P of step i goes over it.  Scheduling barriers separate the slices: inside one
  // the compiler interleaves freely, across them nothing moves.
  // Of a block's first step (FIRST) there is no P V.
  bf16x8_t qreg[kKSteps];
  auto step = [&](auto first, int i, f32x16_t& cur, f32x16_t& nxt, bool mask_nxt, int nxt_base, const bf16x8_t (&p_prev)[2],
                  bf16x8_t (&p_cur)[2], const uint32_t (&vs)[2][kUPW]) {
    constexpr bool FIRST = decltype(first)::value;
    bf16x8_t kq[2][2], vq[2][2], p_other[2];
    const int k_half = 2 * i + 2 + f, v_own = 2 * i - 2 + f, v_other = 2 * i - 1 - f;
    auto request = [&](int s) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        kq[s & 1][e] = k_operand(k_half, 2 * s + e);
        if constexpr (!FIRST) vq[s & 1][e] = v_operand(s < 4 ? v_own : v_other, (s >> 1) & 1, 2 * (s & 1) + e);
      }
    };
    const float m_other = *other_max;
    request(0);
    if constexpr (!FIRST) {
#pragma unroll
      for (int u = 0; u < 2; ++u) p_other[u] = as_bf16x8(other_p[64 * u]);
      if (__any(alpha != 1.0f)) {  // rare: some row's lazy max moved in the previous step
#pragma unroll
        for (int dt = 0; dt < kDT; ++dt) oacc[dt] *= alpha;
      }
    }
    settle(m_other);
    float psum = 0.f;
    auto exponential = [&](int n) {
      float e = fast_exp2(__builtin_fmaf(cur[n], mul, -m_safe));
      pin(e);  // keeps the arithmetic in its slice
      cur[n] = e;
    };
    auto pack = [&](int n) {
      uint32_t pw = pack_bf16x2(cur[2 * n], cur[2 * n + 1]);
      pin(pw);
      // row sum of the rounded weights, the ones that multiply V
      psum = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, pw), kOnes, psum, false);
      return pw;
    };
    u32x4_t packed[2];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      if (s < 7) request(s + 1);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        nxt = mfma_32x32x16(kq[s & 1][e], qreg[2 * s + e], (s == 0 && e == 0) ? zero16 : nxt);
        [[maybe_unused]] const int dt = 2 * (s & 1) + e;
        if constexpr (!FIRST) oacc[dt] = mfma_32x32x16(vq[s & 1][e], s < 4 ? p_prev[s >> 1] : p_other[(s >> 1) & 1], oacc[dt]);
      }
      if (s < 4) {
#pragma unroll
        for (int n = 4 * s; n < 4 * s + 4; ++n) exponential(n);
        if (s < 2) {
#pragma unroll
          for (int n = 0; n < kUPW; ++n) move_k(2 * i + 4 + s, n, k_slot[s][n]);
        } else {
#pragma unroll
          for (int n = 0; n < kUPW; ++n) move_v(2 * i + s - 2, n, vs[s - 2][n]);
        }
      } else if (s < 6) {
#pragma unroll
        for (int n = 0; n < 4; ++n) packed[s - 4][n] = pack(4 * (s - 4) + n);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {  // an MFMA, requests of the next slice, a share of the VALU work
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (e < 3) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (s == 5) {
        asm volatile("s_barrier" ::: "memory");
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          p_cur[u] = as_bf16x8(packed[u]);
          my_p[64 * u] = packed[u];
        }
      }
    }
    l_run = l_run * alpha + psum;
    reach(nxt, mask_nxt, nxt_base);
    __builtin_amdgcn_sched_barrier(0);
  };

  const bool general_scale = p.scale_log2e <= 0.f;  // the fast path needs a positive scale
  auto needs_mask = [&](int base) {  // some row of this wave sees only part of keys base .. base+31
    return general_scale || (base < w_lo_max) || (base + 31 > w_hi_min);
  };
  u32x2_t sl[2], first_slots[4];
  auto request_slots = [&] {
    idx_ptr = p.kv_indices + kv_start;
#pragma unroll
    for (int x = 0; x < 4; ++x) slot_load(k_lo + x * kHalf, first_slots[x]);
#pragma unroll
    for (int x = 0; x < 2; ++x) slot_load(k_lo + (4 + x) * kHalf, sl[x]);  // for the K moves of step 0
  };
  auto move_first_k = [&] {
    // one round trip for all six
    wait_all_vm();
    asm volatile(""
                 : "+v"(first_slots[0]), "+v"(first_slots[1]), "+v"(first_slots[2]), "+v"(first_slots[3]),
                   "+v"(sl[0]), "+v"(sl[1])
                 :
                 : "memory");
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int n = 0; n < kUPW; ++n) {
        v_slot[x >> 1][x & 1][n] = first_slots[x][n];
        move_k(x, n, first_slots[x][n]);
      }
  };
  // ---- prologue: the Q rows and K of halves 0..3 leave and are waited for.  K of half x lives in K stage x % 4, V of
  // half x in V stage x % 4.
  row_bounds();
  if (STAY || n_steps > 0) {
    request_slots();
    move_q();
    move_first_k();
    wait_all_vm();
  }
  for (int at = 0; STAY || n_steps > 0; ++at) {
    __syncthreads();
    f32x16_t sa = zero16, sb;
    bf16x8_t pa[2], pb[2];
#pragma unroll
    for (int kstep = 0; kstep < kKSteps; ++kstep) qreg[kstep] = q_operand(kstep);
#pragma unroll
    for (int kstep = 0; kstep < kKSteps; ++kstep) sa = mfma_32x32x16(k_operand(f, kstep), qreg[kstep], sa);
    reach(sa, needs_mask(k_lo + f * kHalf), k_lo + f * kHalf);
    // Step 0 refills K stages 0 and 1 and the V stages that hold Q (every later step refills stages whose readers passed the
    // barrier at the end of the step before): no wave may start those moves while another still reads them.
    __syncthreads();
    // Step i reads K of halves 2i+2, 2i+3 and V of halves 2i-2, 2i-1; it fills the K stages of halves 2i, 2i+1 with
    // 2i+4, 2i+5 and the V stages of halves 2i-4, 2i-3 with 2i, 2i+1, all in its first half, to be there at its end.
    auto one_step = [&](auto first, int i, f32x16_t& cur, f32x16_t& nxt, const bf16x8_t (&p_prev)[2], bf16x8_t (&p_cur)[2],
                        uint32_t (&vs)[2][kUPW]) {
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int n = 0; n < kUPW; ++n) k_slot[x][n] = sl[x][n];  // requested one step ago
#pragma unroll
      for (int x = 0; x < 2; ++x) slot_load(k_lo + (2 * i + 6 + x) * kHalf, sl[x]);
      const int base = k_lo + (i + 1) * kStep + f * kHalf;
      step(first, i, cur, nxt, needs_mask(base), base, p_prev, p_cur, vs);
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int n = 0; n < kUPW; ++n) vs[x][n] = k_slot[x][n];
      asm volatile("s_waitcnt vmcnt(0)" : "+v"(sl[0]), "+v"(sl[1]) : : "memory");
      __syncthreads();
    };
    one_step(std::true_type{}, 0, sa, sb, pb, pa, v_slot[0]);
    for (int i = 1; i < n_steps; i += 2) {
      one_step(std::false_type{}, i, sb, sa, pa, pb, v_slot[1]);
      if (i + 1 == n_steps) break;
      one_step(std::false_type{}, i + 1, sa, sb, pb, pa, v_slot[0]);
    }
    // What the block leaves behind while the next one begins
    const int last_half = 2 * n_steps - 2, done_q = q_start, done_rows = rows_total, done_row0 = row0;
    const bool more = STAY && at + 1 < n_listed;  // constant where it doesn't stay
    if (more) {
      take_listed(at + 1);
      rows_total = q_len * p.group;
      row0 = qblk * kRows;
      n_steps = (k_hi - k_lo + kStep - 1) / kStep;
      row_bounds();
      request_slots();
    }
    // the last step's P V is still owed
    if (__any(alpha != 1.0f)) {
#pragma unroll
      for (int dt = 0; dt < kDT; ++dt) oacc[dt] *= alpha;
    }
#pragma unroll
    for (int x = 0; x < 2; ++x)  // keys of half 0, keys of half 1
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const bf16x8_t pw = as_bf16x8((x == f ? my_p : other_p)[64 * u]);
#pragma unroll
        for (int dt = 0; dt < kDT; ++dt) oacc[dt] = mfma_32x32x16(v_operand(last_half + x, u, dt), pw, oacc[dt]);
      }
    if constexpr (STAY) {
      // Nobody reads the K stages any more, nor the maxima; the barrier frees the V stages.
      const float own = sum_across<32>(l_run);
      *my_max = own;
      if (more) move_first_k();
      __syncthreads();
      if (more) move_q();
      const float l = own + *other_max, inv = (l > 0.f) ? 1.0f / l : 0.f;
      // Lane (row c32, h) holds 4 of 8 adjacent dims.  Exchanges between lanes l and l + 32 give it all 8 of every second
      // group, exchanges between rows c and c + 16 then leave a store 64 bytes each of 16 rows (32 of 32 rows take 1 K cycles
      // more).  Every wave makes every store, whether or not a lane has a row: the wait below counts on it.
      int lane_row = c32, half = h;  // anew, see move_q()
      asm volatile("" : "+v"(lane_row), "+v"(half));
      uint16_t* dst[2];
      unsigned long long has[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int row = done_row0 + group_row + 16 * x + (lane_row & 15);
        has[x] = __ballot(row < done_rows);
        const int qi = row_to_query(p, row);  // of a row past the last: an address, which nothing is stored at
        dst[x] = p.out + ((int64_t)(done_q + qi) * p.n_q + kvh * p.group + row - qi * p.group) * kD + 128 * f + 16 * (lane_row >> 4) + 8 * half;
      }
#pragma unroll
      for (int dt = 0; dt < kDT; ++dt) {
        u32x4_t out[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          uint32_t d[4];
#pragma unroll
          for (int a = 0; a < 4; ++a) d[a] = pack_bf16x2(oacc[dt][4 * a + 2 * e] * inv, oacc[dt][4 * a + 2 * e + 1] * inv);
          const auto ab = __builtin_amdgcn_permlane32_swap(d[0], d[1], false, false), cd = __builtin_amdgcn_permlane32_swap(d[2], d[3], false, false);
          const auto lo = __builtin_amdgcn_permlane16_swap(ab[0], cd[0], false, false), hi = __builtin_amdgcn_permlane16_swap(ab[1], cd[1], false, false);
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            out[x][e] = lo[x];
            out[x][2 + e] = hi[x];
          }
        }
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          unsigned long long saved;
          // (wait states: the store still reads its data's registers, and the compiler does not look into the statement)
          asm volatile("s_mov_b64 %0, exec\n\ts_and_b64 exec, exec, %1\n\tglobal_store_dwordx4 %2, %3, off offset:%4\n\ts_mov_b64 exec, %0\n\ts_nop 1"
                       : "=&s"(saved)
                       : "s"(has[x]), "v"(dst[x]), "v"(out[x]), "n"(64 * dt)
                       : "memory", "scc");
        }
      }
      if (!more) return;
      reset();
      alpha = 1.0f;
      wait_vm_at_most<2 * kDT>();  // all but the stores
    }
    if constexpr (!STAY) break;
  }
  if constexpr (STAY) return;
  // both halves of the row sum
  float l = l_run;
  l = sum_across<32>(l);
  __syncthreads();
  *my_max = l;
  __syncthreads();
  l += *other_max;
  const float inv = (l > 0.f) ? 1.0f / l : 0.f;
  __syncthreads();  // the epilogue reuses the stages

  // accumulator i of O^T tile dt is dim 128f + 32dt + 8(i/4) + 4h + i%4 of query row c32
  if (to_partial) {
    // ---- key split: normalised fp32 partial and log-sum-exp (base 2) per row, from registers
    const int row = row0 + group_row + c32;
    if (row < rows_total) {
      const int qi = row_to_query(p, row);
      const int hh = row - qi * p.group;
      const int64_t at = p.ragged_tiles > 0 ? part_at + row
                                            : (int64_t)split * p.part_rows + (int64_t)(q_start + qi) * p.n_q + kvh * p.group + hh;
      if (h == 0 && f == 0) p.part_lse[at] = (l > 0.f) ? m_run + __log2f(l) : kNegInf;
      float* dst = p.part_o + at * kD + 128 * f + 4 * h;
#pragma unroll
      for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          f32x4_t v = {oacc[dt][4 * a] * inv, oacc[dt][4 * a + 1] * inv, oacc[dt][4 * a + 2] * inv,
                       oacc[dt][4 * a + 3] * inv};
          *reinterpret_cast<f32x4_t*>(dst + 32 * dt + 8 * a) = v;
        }
    }
    return;
  }
  // ---- epilogue: normalise, transpose through LDS, store whole rows ---------------------
  unsigned char* os = smem;
  {
    const int lrow = group_row + c32;
#pragma unroll
    for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        u32x2_t wv;
        wv[0] = pack_bf16x2(oacc[dt][4 * a] * inv, oacc[dt][4 * a + 1] * inv);
        wv[1] = pack_bf16x2(oacc[dt][4 * a + 2] * inv, oacc[dt][4 * a + 3] * inv);
        *reinterpret_cast<u32x2_t*>(os + (lrow * OROW + 128 * f + 32 * dt + 8 * a + 4 * h) * 2) = wv;
      }
  }
  __syncthreads();
  constexpr int ROWS_PER_PASS = kNW * 64 / 32;  // 32 lanes store one 512-byte row
  const int c = tid & 31;
#pragma unroll 4
  for (int pass = 0; pass < kRows / ROWS_PER_PASS; ++pass) {
    const int lrow = pass * ROWS_PER_PASS + (tid >> 5);
    const int row = row0 + lrow;
    if (row < rows_total) {
      const int qi = row_to_query(p, row);
      const int hh = row - qi * p.group;
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(os + (lrow * OROW + c * 8) * 2);
      st_stream_b128(p.out + ((int64_t)(q_start + qi) * p.n_q + kvh * p.group + hh) * kD + c * 8, v);
    }
  }
}

}  // namespace

int launch_prefill_tile256(const PrefillArgs& a, hipStream_t stream) {
  if (a.head_dim != kD) return MSGL_ERR_HEAD_DIM;
  PrefillParams p;
  int64_t n_blocks = 0;
  bool wide = false;
  const int rc = make_prefill_params(a, p, n_blocks, wide, kPrefillBlockRows256);
  if (rc != MSGL_OK || n_blocks == 0) return rc;
  if (p.nt.out_loc != nullptr) {
    p.nt.blocks = (uint32_t)n_blocks;
    n_blocks += kRestBlocks;
  }
  const dim3 grid((unsigned)n_blocks);
  auto* const kernel = p.length_rounds > 0 ? (wide ? prefill_tile256_kernel<true, true> : prefill_tile256_kernel<false, true>)
                                           : (wide ? prefill_tile256_kernel<true, false> : prefill_tile256_kernel<false, false>);
  const int launched = launch_kernel(kernel, grid, dim3(kNW * 64), stream, p);
  if (launched != MSGL_OK || (p.n_ksplit == 1 && p.ragged_tiles == 0)) return launched;
  return launch_prefill_merge(p, kD, stream);
}

}  // namespace msgl
