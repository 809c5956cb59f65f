// What the kernels for short query blocks share (paged_splitkv.hip: equal segments of the token
// stream; paged_shares.hip: shares of one request): launch parameters, a request's geometry, and
// one wave's walk over a range of keys with its columns' softmax state in registers.
#pragma once
#include "msgl_device.h"
#include "msgl_internal.h"

namespace msgl {

// How the pool's rows are read: with offsets of 32 bits, or kWide of 64 (a pool of 4 GiB or more); kStream: past the caches (streams() in
// paged_splitkv.hip), but those of keys that another request has as well (OtherSlots).
enum Walk { kNarrow = 0, kWide = 1, kStream = 2 };

struct SplitKvParams {
  const uint16_t* q;
  const uint16_t* k_cache;
  const uint16_t* v_cache;
  const int32_t* kv_indptr;
  const int32_t* kv_indices;
  const int32_t* qo_indptr;
  const int32_t* prefix_lens;
  uint16_t* out;
  float* part_o;        // [n_seg + batch][n_kv][D / 8][cols][8], fp32 or IEEE half: see partial_offset()
  float* part_lse;      // [n_seg + batch][n_kv][cols]
  int32_t* req_items;   // [batch][2] first segment holding the request, number of segments sharing it
  int64_t k_stride0, v_stride0;
  int64_t q_stride0;    // elements from one row of q to the next
  int32_t batch, n_q, n_kv, group;
  int32_t nwh;          // kv heads per workgroup
  int32_t head_groups;  // n_kv / nwh
  int32_t n_seg, min_seg, cols, max_len_extend;
  int32_t boundary;  // stream positions a request boundary is charged with (see stream_length)
  int32_t q_begin, q_cap;  // first query of every request in this launch; cap on a request's queries
  int32_t f16;             // elements are IEEE half instead of bf16
  int32_t is_cross, window;
  int32_t walk;  // Walk
  uint32_t max_slot;  // num_slots - 1: slot ids are clamped to it before they become addresses
  uint32_t per_group;  // ceil(2^16 / group), see query_of()
  float scale_log2e;
  long long* clock_probe;  // measurement aid, see ClockProbe; nullptr: off
  struct {  // a decode step's new tokens (new_token.h); k == nullptr: none
    const uint16_t *k, *v, *q_weight, *k_weight;
    const int32_t *positions, *out_loc;
    uint16_t *k_pool, *v_pool;
    int64_t k_stride0, v_stride0;
    int32_t rows;     // of k and v
    uint32_t blocks;  // workgroups in front of those of store_rows_of_no_request()
    float eps, log2_base;
  } nt;
};

// Everything but the workspace pointers and the cut (paged_splitkv.hip).
void fill_splitkv_params(const SplitKvArgs& a, SplitKvParams& p);

// Visible key range and query geometry of one request.
struct ReqInfo {
  int32_t kv_start, kv_len;  // CSR segment
  int32_t q_start, q_len;    // rows of q / out
  int32_t prefix;            // position of query 0
  int32_t lo, hi;            // keys [lo, hi) can be visible to some query of the request
  int32_t rows;              // of q, those that this launch does not cover included
};

// P: SplitKvParams, or what of it this takes.
template <typename P>
__device__ __forceinline__ void visible_range(const P& p, ReqInfo& r) {
  // first query has the lowest window floor, last query the highest causal limit
  r.lo = (p.window > 0) ? max(0, r.prefix - p.window + 1) : 0;
  r.lo &= ~15;
  r.hi = p.is_cross ? r.kv_len : min(r.kv_len, r.prefix + r.q_len);
  if (r.q_len <= 0 || r.hi <= r.lo) {
    r.lo = 0;
    r.hi = 0;
  }
}
template <typename P>
__device__ __forceinline__ ReqInfo request_info(const P& p, int b) {
  ReqInfo r;
  r.kv_start = p.kv_indptr[b];
  r.kv_len = p.kv_indptr[b + 1] - r.kv_start;
  if (r.kv_len < 0) r.kv_len = 0;
  if (p.qo_indptr == nullptr) {
    r.q_start = b;
    r.q_len = r.rows = 1;
    r.prefix = r.kv_len - 1;
  } else {
    // this launch covers queries q_begin .. q_begin + max_len_extend - 1 of every request
    const int q0 = p.qo_indptr[b];
    r.rows = p.qo_indptr[b + 1] - q0;
    const int q_all = min(r.rows, p.q_cap);
    r.q_start = q0 + p.q_begin;
    r.q_len = max(min(q_all - p.q_begin, p.max_len_extend), 0);
    r.prefix = p.prefix_lens[b] + p.q_begin;
  }
  visible_range(p, r);
  return r;
}
// The same with meanwhile() called once the loads are under way.  (A decode call loads its lengths again for what it has not:
// a branch around those loads would be waited in front of.)
template <typename P, typename Meanwhile>
__device__ __forceinline__ ReqInfo request_info(const P& p, int b, Meanwhile&& meanwhile) {
  ReqInfo r;
  const bool decode = p.qo_indptr == nullptr;
  const int32_t *qo_indptr = decode ? p.kv_indptr : p.qo_indptr, *prefix_lens = decode ? p.kv_indptr : p.prefix_lens;
  r.kv_start = p.kv_indptr[b];
  const int kv_end = p.kv_indptr[b + 1], q0 = qo_indptr[b], q_end = qo_indptr[b + 1], prefix = prefix_lens[b];
  meanwhile();
  r.kv_len = max(kv_end - r.kv_start, 0);
  r.rows = decode ? 1 : q_end - q0;
  r.q_start = decode ? b : q0 + p.q_begin;
  r.q_len = decode ? 1 : max(min(min(r.rows, p.q_cap) - p.q_begin, p.max_len_extend), 0);
  r.prefix = decode ? r.kv_len - 1 : prefix + p.q_begin;
  visible_range(p, r);
  return r;
}

// The query that a column belongs to, col / group: exact while col (group - 1) < 2^16 (160 columns at most; a division is 25 instructions).
__device__ __forceinline__ int query_of(const SplitKvParams& p, int col) { return (int)((uint32_t)col * p.per_group >> 16); }

template <int D>
struct KvTile {
  u32x4_t k[2][D / 32];   // [16-token sub-tile][32-wide slice of D]: MFMA A operand of S^T
  u32x4_t v[D / 128][8];  // [128-wide half of D][token j of the lane group]: raw V segments
};

// One wave's columns (NCT tiles of 16) against one range of keys: the Q operand, what each column
// may see, and the running softmax state with the unnormalised output O^T.
template <int D, int NCT>
struct Columns {
  // Two tiles of 256 dims leave no registers for Q beside the keys in flight: it is in LDS, a lane's 16 bytes 64 lanes apart.
  static constexpr bool kQInLds = D == 256 && NCT > 1;
  static constexpr int kQInts = kQInLds ? NCT * (D / 32) * kWave : 1;  // of 16 bytes
  typename std::conditional<kQInLds, __attribute__((address_space(3))) u32x4_t*, u32x4_t[NCT][D / 32]>::type q;
  int lo[NCT], hi[NCT];        // first and last visible key of this lane's column in each tile
  int all_lo, all_hi;          // a tile of keys is mask-free iff inside [all_lo, all_hi]
  float m[NCT], l[NCT];        // running maximum (base 2); this lane's part of the sum
  f32x4_t o[NCT][D / 128][8];  // o[ct][hf][n][i]: dim hf * 128 + 8 * (4 * (lane / 16) + i) + n
};

// Columns ct0 * 16 .. of kv head `kvh` of request `r`, for the keys before `t_end`.  LOAD_Q: the Q operand from memory
// (else it is left to the caller).  SMALL: the launch is one of shares (the long walks' kernels have no register to spare for query_of()).
template <int D, int NCT, bool LOAD_Q = true, bool SMALL = false>
__device__ __forceinline__ void start_columns(const SplitKvParams& p, const ReqInfo& r, int kvh, int ct0,
                                              int t_end, Columns<D, NCT>& c_) {
  constexpr int KS = D / 32, VH = D / 128;
  const int t16 = lane_id() & 15, g = lane_id() >> 4;
  const int ncols = r.q_len * p.group;
  int all_lo = 0, all_hi = 0x7fffffff;
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    const int col = (ct0 + ct) * 16 + t16;
    const bool valid = col < ncols;
    const int qi = !valid ? 0 : SMALL ? query_of(p, col) : col / p.group;
    const int hh = valid ? col - qi * p.group : 0;
    const uint16_t* qrow =
        p.q + (int64_t)(r.q_start + qi) * p.q_stride0 + (kvh * p.group + hh) * D + g * 8;
#pragma unroll
    for (int c = 0; c < KS; ++c) {
      u32x4_t raw = {0u, 0u, 0u, 0u};
      if (LOAD_Q && valid) raw = ld_global_b128(qrow + c * 32);
      if constexpr (Columns<D, NCT>::kQInLds) c_.q[(ct * KS + c) * kWave] = raw;
      else c_.q[ct][c] = raw;
    }
    const int qpos = r.prefix + qi;
    int lo = (p.window > 0) ? qpos - p.window + 1 : 0;
    int hi = p.is_cross ? r.kv_len - 1 : min(qpos, r.kv_len - 1);
    hi = min(hi, t_end - 1);
    if (valid) {
      all_lo = max(all_lo, lo);
      all_hi = min(all_hi, hi);
    } else {
      lo = 1;
      hi = 0;
    }
    c_.lo[ct] = lo;
    c_.hi[ct] = hi;
  }
  c_.all_lo = __builtin_amdgcn_readfirstlane(row_max16(all_lo));
  c_.all_hi = __builtin_amdgcn_readfirstlane(~row_max16(~all_hi));
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    c_.m[ct] = kNegInf;
    c_.l[ct] = 0.f;
#pragma unroll
    for (int hf = 0; hf < VH; ++hf)
#pragma unroll
      for (int n = 0; n < 8; ++n) c_.o[ct][hf][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
}

// Slot ids of a wave's first two tiles: lane l those of tokens l % 16 and 16 + l % 16 of each.
struct FirstIds {
  int a[2], b[2];
};
__device__ __forceinline__ FirstIds first_ids(const SplitKvParams& p, const ReqInfo& r, int t_begin, int t_end) {
  const int32_t* idx = p.kv_indices + r.kv_start;
  const int at = t_begin + (lane_id() & 15), last = t_end - 1;
  return FirstIds{{idx[min(at, last)], idx[min(at + 16, last)]}, {idx[min(at + 32, last)], idx[min(at + 48, last)]}};
}

// Requests with a common prefix have its keys in the same slots, and each finds in the caches what another has read.  Plain loads get
// 9-10 TB/s then, loads past the caches the 7 they always get: decode of 64 requests of 256 keys behind 4096 in common, 32 / 8 heads, 117.7 us
// and 165.0, of 128 of 512 behind 1024 96 and 118, verify of 32 x 8 of 512 behind 4096 78 and 94, shares of 5 of 1024 behind 16 K, 16 / 2 heads of
// 256, 32.1 and 34.8.  So a segment or share whose first key another request has in the same slot is read plainly.  Of the requests the 64 around
// its own are looked at, one to a lane.  With nothing in common decode of 64 requests of 1-8 K 200.3 -> 201.5, 24 of 127-4095, 16 / 2 heads of 256, 24.3 -> 24.5.
struct OtherKeys {  // of one of those requests; those of the request itself as none
  int start, len;
};
struct OtherSlots {
  bool has;
  int slot, own;
  // `at`: a key of request `r`, -1: none
  __device__ __forceinline__ OtherSlots(const SplitKvParams& p, const OtherKeys& other, const ReqInfo& r, int at) {
    has = at >= 0 && at < other.len;
    const int own_at = at >= 0 ? r.kv_start + at : 0;
    slot = p.kv_indices[has ? other.start + at : own_at];
    own = p.kv_indices[own_at];
  }
  __device__ __forceinline__ bool same() const { return has && slot == own; }
  __device__ __forceinline__ bool shared() const { return __ballot(same()) != 0; }  // all lanes must call
};

// A tile whose K rows came by whole lines (attend_keys): of the 16 rows of a sub-tile, lanes of t16 < 8 have even pieces of 64 bytes, of
// row t16 in slice 2 c and of row t16 + 8 in slice 2 c + 1, the others odd ones, of row t16 - 8 and of row t16.  Lane t16 gives
// lane t16 +- 8 what is of its row.
template <int D>
__device__ __forceinline__ void lines_to_operands(KvTile<D>& t) {
  constexpr int kRor8 = 0x128;  // DPP: from the lane 8 away in a row of 16; banks 0xc: written in its upper 8 lanes, 0x3 in the lower
#pragma unroll
  for (int sub = 0; sub < 2; ++sub)
#pragma unroll
    for (int c = 0; c < D / 32; c += 2)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int a = (int)t.k[sub][c][e], b = (int)t.k[sub][c + 1][e];
        t.k[sub][c][e] = (uint32_t)__builtin_amdgcn_update_dpp(a, b, kRor8, 0xf, 0xc, false);
        t.k[sub][c + 1][e] = (uint32_t)__builtin_amdgcn_update_dpp(b, a, kRor8, 0xf, 0x3, false);
      }
}

// The scores of a tile where Q is in LDS: S^T[token][col] for the two 16-token sub-tiles.
template <int D, int NCT, bool F16>
__device__ __forceinline__ void scores_from_lds(const KvTile<D>& t, const Columns<D, NCT>& c_, f32x4_t (&s)[2][NCT]) {
  constexpr int KS = D / 32;
  auto load = [&](int c, u32x4_t (&q)[NCT]) {
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) q[ct] = c_.q[(ct * KS + c) * kWave];
  };
  u32x4_t q[2][NCT];
  load(0, q[0]);
#pragma unroll
  for (int sub = 0; sub < 2; ++sub)
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) s[sub][ct] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < KS; ++c) {
    if (c + 1 < KS) load(c + 1, q[(c + 1) & 1]);
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) s[sub][ct] = mfma_16x16x32_raw<F16>(t.k[sub][c], q[c & 1][ct], s[sub][ct]);
    __builtin_amdgcn_sched_barrier(0);  // no more of Q in registers than the next step's
  }
}

// Keys tb .. tb + 31, in registers, for the columns in `c_`.  scored(): called when K is no longer wanted (Q in LDS)
struct NothingElse {
  __device__ __forceinline__ void operator()() const {}
};
template <int D, int NCT, bool F16, typename Scored = NothingElse>
__device__ __forceinline__ void compute_tile(const SplitKvParams& p, const KvTile<D>& t, int tb, Columns<D, NCT>& c_, Scored&& scored = {}) {
  constexpr bool kQInLds = Columns<D, NCT>::kQInLds;
  constexpr int KS = D / 32;   // k-steps of the QK product
  constexpr int VH = D / 128;  // 128-wide halves of D in the PV product
  const int g = lane_id() >> 4;
  // S^T[token][col] for the two 16-token sub-tiles
  f32x4_t s[2][NCT];
  if constexpr (kQInLds) {
    scores_from_lds<D, NCT, F16>(t, c_, s);
    scored();
    __builtin_amdgcn_sched_barrier(0);
  } else {
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) {
        f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < KS; ++c)
          acc = mfma_16x16x32_raw<F16>(t.k[sub][c], c_.q[ct][c], acc);
        s[sub][ct] = acc;
      }
  }
  const bool need_mask = (tb < c_.all_lo) || (tb + 31 > c_.all_hi);
  uint32_t pb[NCT][4];
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    float x[2][4];
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
#pragma unroll
      for (int i = 0; i < 4; ++i) x[sub][i] = s[sub][ct][i] * p.scale_log2e;
    if (need_mask) {
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int tok = tb + sub * 16 + 4 * g + i;
          if (tok < c_.lo[ct] || tok > c_.hi[ct]) x[sub][i] = kNegInf;
        }
    }
    float mx = fmaxf(fmaxf(fmaxf(x[0][0], x[0][1]), fmaxf(x[0][2], x[0][3])),
                     fmaxf(fmaxf(x[1][0], x[1][1]), fmaxf(x[1][2], x[1][3])));
    mx = max_across<32>(max_across<16>(mx));
    const float m_new = fmaxf(c_.m[ct], mx);
    const float m_safe = (m_new == kNegInf) ? 0.f : m_new;
    const float alpha = fast_exp2(c_.m[ct] - m_safe);
    c_.m[ct] = m_new;
    float psum = 0.f;
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[sub][i] = fast_exp2(x[sub][i] - m_safe);
        psum += x[sub][i];
      }
    c_.l[ct] = c_.l[ct] * alpha + psum;
    pb[ct][0] = pack_16x2<F16>(x[0][0], x[0][1]);
    pb[ct][1] = pack_16x2<F16>(x[0][2], x[0][3]);
    pb[ct][2] = pack_16x2<F16>(x[1][0], x[1][1]);
    pb[ct][3] = pack_16x2<F16>(x[1][2], x[1][3]);
    if (__any(alpha != 1.0f)) {
#pragma unroll
      for (int hf = 0; hf < VH; ++hf)
#pragma unroll
        for (int n = 0; n < 8; ++n) c_.o[ct][hf][n] *= alpha;
    }
  }
  if constexpr (kQInLds) __builtin_amdgcn_sched_barrier(0);
  // O^T += V^T P^T.  MFMA n of half hf produces d = hf*128 + 8*row + n on row = l%16.
#pragma unroll
  for (int hf = 0; hf < VH; ++hf)
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      u32x4_t vt;
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const uint32_t a = t.v[hf][2 * qd][n >> 1];
        const uint32_t c = t.v[hf][2 * qd + 1][n >> 1];
        vt[qd] = (n & 1) ? pack_hi16(a, c) : pack_lo16(a, c);
      }
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) {
        const u32x4_t pv = {pb[ct][0], pb[ct][1], pb[ct][2], pb[ct][3]};
        c_.o[ct][hf][n] = mfma_16x16x32_raw<F16>(vt, pv, c_.o[ct][hf][n]);
      }
      if constexpr (kQInLds) __builtin_amdgcn_sched_barrier(0);  // (and no more transposed V than one product's)
    }
}

// Keys [t_begin, t_end) of request `r`, in order, for the columns in `c_`; `first`: its first_ids(), asked for before
// the columns were made.
// SHORT: ranges of one tile are common, end behind it (in a long walk the test costs more than it saves).
// kStream: the loads past the caches take whole lines.  A row of V is 16 lanes' load as it is.  K's rows as operands are not, 64 bytes
// of 16 rows a load: long walks load 128 bytes of 8 rows and exchange them (lines_to_operands); in shares, where a wave waits
// for each of its few tiles, the exchange costs more than it gives and K is read the plain way.  us, plain / V past the caches / K too, as operands / by
// lines: decode 1253 MiB 225 / 207 / 234 / 202, 4718 MiB 810 / 738 / 837 / 725, verify 143.5 / 134.3 / 146 / 126, shares at head_dim 256
// 26.3 / 24.8 / 28.6 / 26.3, of a window 33.1 / 27.7 / 31.6 / 29.6.  A row that two waves read (col_split) is read the plain way: 64 columns 1.0-1.2x past the
// caches, at head_dim 256 1.0-1.3x.
// meanwhile(): called once the first tile has been asked for; may finish the columns' Q operand and put keys of its own
// into their state.
template <int D, int NCT, int WALK, bool F16, bool SHORT, typename Meanwhile>
__device__ __forceinline__ void attend_keys(const SplitKvParams& p, const ReqInfo& r, int kvh, int t_begin,
                                            int t_end, const FirstIds& first, Columns<D, NCT>& c_, Meanwhile&& meanwhile) {
  constexpr int KS = D / 32;   // k-steps of the QK product
  constexpr int VH = D / 128;  // 128-wide halves of D in the PV product
  constexpr bool LINES = (WALK & kStream) && !SHORT;
  const int lane = lane_id();
  const int t16 = lane & 15;
  const int g = lane >> 4;
  const unsigned char* kbase =
      reinterpret_cast<const unsigned char*>(p.k_cache + (int64_t)kvh * D + g * 8 + (LINES ? (t16 >> 3) * 32 : 0));
  const unsigned char* vbase =
      reinterpret_cast<const unsigned char*>(p.v_cache + (int64_t)kvh * D + t16 * 8);
  const uint32_t k_row_bytes = (uint32_t)p.k_stride0 * 2u;
  const uint32_t v_row_bytes = (uint32_t)p.v_stride0 * 2u;
  auto row_offset = [](int slot_id, uint32_t row_bytes) -> uint64_t {
    if constexpr (WALK != kNarrow) return (uint64_t)(uint32_t)slot_id * row_bytes;
    else return (uint64_t)((uint32_t)slot_id * row_bytes);
  };
  auto load = [](const unsigned char* from) {
    if constexpr (WALK & kStream) return ld_stream_b128(from);
    else return ld_global_b128(from);
  };
  const int32_t* idx_base = p.kv_indices + r.kv_start;
  const int last_tok = t_end - 1;

  // slot ids of the two K rows this lane loads in a 32-token tile starting at tb
  auto load_idx = [&](int tb, int& s0, int& s1) {
    s0 = (int)min((uint32_t)idx_base[min(tb + t16, last_tok)], p.max_slot);
    s1 = (int)min((uint32_t)idx_base[min(tb + 16 + t16, last_tok)], p.max_slot);
  };
  auto load_k = [&](KvTile<D>& t, int s0, int s1) {
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const int s = sub ? s1 : s0;
      if constexpr (LINES) {  // of 8 rows 128 bytes each: rows t16 % 8 and t16 % 8 + 8
        const unsigned char* row[2] = {kbase + row_offset(__builtin_amdgcn_update_dpp(s, s, 0x128, 0xf, 0xc, false), k_row_bytes),
                                       kbase + row_offset(__builtin_amdgcn_update_dpp(s, s, 0x128, 0xf, 0x3, false), k_row_bytes)};
#pragma unroll
        for (int c = 0; c < KS; ++c) t.k[sub][c] = load(row[c & 1] + (c >> 1) * 128);
      } else {
        const unsigned char* row = kbase + row_offset(s, k_row_bytes);
#pragma unroll
        for (int c = 0; c < KS; ++c) t.k[sub][c] = ld_global_b128(row + c * 64);
      }
    }
  };
  auto load_v = [&](KvTile<D>& t, int s0, int s1) {
    // V rows of this lane group: tokens 4g+j (j<4) of sub-tile 0, then of sub-tile 1;
    // their slot ids sit in lanes 4g+j of the K index registers.
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int src = 4 * g + (j & 3);
      const int slot = __shfl(j < 4 ? s0 : s1, src, kWave);
      const unsigned char* vrow = vbase + row_offset(slot, v_row_bytes);
#pragma unroll
      for (int hf = 0; hf < VH; ++hf) t.v[hf][j] = load(vrow + hf * 256);
    }
  };

  auto load_tile = [&](KvTile<D>& t, int s0, int s1) {
    load_k(t, s0, s1);
    load_v(t, s0, s1);
  };

  if constexpr (Columns<D, NCT>::kQInLds) {
    // ---- one register tile: the next one's K comes in beside the softmax and the PV product, its V beside the next scores
    // (and whatever comes meanwhile has a tile of its own: it comes first)
    meanwhile();
    __builtin_amdgcn_sched_barrier(0);
    KvTile<D> t;
    int i0 = (int)min((uint32_t)first.a[0], p.max_slot), i1 = (int)min((uint32_t)first.a[1], p.max_slot);
    load_tile(t, i0, i1);
    i0 = (int)min((uint32_t)first.b[0], p.max_slot);
    i1 = (int)min((uint32_t)first.b[1], p.max_slot);
    for (int tok = t_begin; tok < t_end; tok += 32) {
      if constexpr (LINES) lines_to_operands(t);
      const int v0 = i0, v1 = i1;
      compute_tile<D, NCT, F16>(p, t, tok, c_, [&] {
        load_k(t, v0, v1);
        load_idx(tok + 64, i0, i1);
      });
      load_v(t, v0, v1);
      __builtin_amdgcn_sched_barrier(0);
    }
    return;
  }
  // ---- tile loop: two register tiles, slot ids fetched two tiles ahead.  Every load in
  // the loop body is unconditional (tokens past the range clamp to its last token and
  // are masked), so the number of loads in flight at each wait is a compile-time
  // constant and the next tile stays in flight while the current one is computed. ----
  const int n_pairs = (t_end - t_begin + 63) / 64;
  KvTile<D> ta, tb_;
  int i0a = (int)min((uint32_t)first.a[0], p.max_slot), i0b = (int)min((uint32_t)first.a[1], p.max_slot);
  int i1a = (int)min((uint32_t)first.b[0], p.max_slot), i1b = (int)min((uint32_t)first.b[1], p.max_slot);
  load_tile(ta, i0a, i0b);
  load_idx(t_begin + 64, i0a, i0b);
  meanwhile();
  for (int pr = 0; pr < n_pairs; ++pr) {
    const int tok = t_begin + pr * 64;
    load_tile(tb_, i1a, i1b);
    load_idx(tok + 96, i1a, i1b);
    if constexpr (LINES) lines_to_operands(ta);
    compute_tile<D, NCT, F16>(p, ta, tok, c_);
    if (SHORT && tok + 32 >= t_end) break;
    load_tile(ta, i0a, i0b);
    load_idx(tok + 128, i0a, i0b);
    if constexpr (LINES) lines_to_operands(tb_);
    compute_tile<D, NCT, F16>(p, tb_, tok + 32, c_);
  }
}

}  // namespace msgl
