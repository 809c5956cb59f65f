// The new token of a decode step inside the attention launch (paged_shares.hip, paged_splitkv.hip).
//
// A step's own row of k and v goes into the pool in the launch that attends, by the wave whose range holds its
// request's last key.  That wave takes the row from its source and not from the pool, so nobody waits for the
// store: while its first tile is under way the new key makes the first state of the columns, and the walk
// ends in front of it.  (Where the request's last key is another slot, every wave of the request stores the row and
// waits for that before it reads the pool.)  (Put into the tile that the walk computes last, it cost registers: 124 bytes of
// spills and 6 us at head_dim 256.)  With norm weights every wave normalises and rotates its own q heads (and that
// one the new key) at that time, four heads at once: a lane finds sine and cosine of one or two of the head's
// angles and the wave exchanges them through LDS.  (At head_dim 256 all that goes in front of the first tile: there
// are no registers for both.)
#pragma once
#include "norm_rope.h"
#include "prefill_tile_common.h"
#include "splitkv_tiles.h"

namespace msgl {

// What a decode launch does with its requests' new tokens: they are in the pool already; they are stored; q and k
// are normalised and rotated, k and v stored.
// (kStoreRows: kStore for several new tokens per request, a prefill call's.)
enum NewMode { kStored = 0, kStore = 1, kNormRopeStore = 2, kStoreRows = 3 };
template <NewMode MODE>
using New = std::integral_constant<int, MODE>;

inline void fill_new_tokens(const NewTokens& n, SplitKvParams& p) {
  if (n.k == nullptr) return;
  p.nt.k = static_cast<const uint16_t*>(n.k);
  p.nt.v = static_cast<const uint16_t*>(n.v);
  p.nt.q_weight = static_cast<const uint16_t*>(n.q_weight);
  p.nt.k_weight = static_cast<const uint16_t*>(n.k_weight);
  p.nt.positions = n.positions;
  p.nt.out_loc = n.out_loc;
  p.nt.k_pool = const_cast<uint16_t*>(p.k_cache);
  p.nt.v_pool = const_cast<uint16_t*>(p.v_cache);
  p.nt.k_stride0 = n.k_stride0;
  p.nt.v_stride0 = n.v_stride0;
  p.nt.rows = (int32_t)n.rows;
  p.nt.eps = n.eps;
  p.nt.log2_base = n.q_weight ? log2f(n.rope_base) : 0.f;
}

template <bool F16>
__device__ __forceinline__ float value_of(uint32_t pair, int e) {  // of two 16-bit values the first or the second
  if constexpr (F16) return (float)__builtin_bit_cast(f16x2_t, pair)[e];
  else return __builtin_bit_cast(float, e ? pair & 0xffff0000u : pair << 16);
}
// The walk ends in front of the new token, whose place in the pool is read by nobody: a wave's first slot ids again,
// those from `tail` on `before`, the id in front of it (the last tile's rows repeat the last key walked; what has
// weight 0 still has to be a number).
__device__ __forceinline__ void end_ids(FirstIds& ids, int t_begin, int tail, int before) {
  const int at = t_begin + (lane_id() & 15);
  if (at >= tail) ids.a[0] = before;
  if (at + 16 >= tail) ids.a[1] = before;
  if (at + 32 >= tail) ids.b[0] = before;
  if (at + 48 >= tail) ids.b[1] = before;
}

template <int D>
struct HeadLds {  // NORM: of one wave
  uint16_t row[17][D];  // the new key, the heads of the columns
  float cosines[D / 2], sines[D / 2];
};
// Where the new token of request b goes and, with NORM, its position: asked for, in vector registers until they are taken
// (a value known to be the wave's would be waited for at once, to become a scalar).
template <bool NORM>
struct NewTokenIds {
  int32_t slot_, position_ = 0;
  __device__ __forceinline__ NewTokenIds(const SplitKvParams& p, int b) {
    uint32_t at = (uint32_t)b;
    pin(at);
    slot_ = p.nt.out_loc[at];
    if constexpr (NORM) position_ = p.nt.positions[at];
  }
  __device__ __forceinline__ uint32_t slot() const { return (uint32_t)__builtin_amdgcn_readfirstlane(slot_); }
  __device__ __forceinline__ int position() const { return __builtin_amdgcn_readfirstlane(position_); }
};
template <int D, bool NORM, bool F16>
struct NewToken {
  static constexpr int E = D / 32, KS = D / 32, VH = D / 128;
  static constexpr int kEarly = 2;  // trips of four heads whose rows are asked for before the first tile
  using Half = typename HalfRow<E>::type;
  const SplitKvParams& sp;
  Columns<D, 1>& columns;
  HeadLds<D>& lds;
  const uint16_t* q;  // the first of the columns' heads
  const uint16_t *k, *v;
  bool owner;         // the request's last key is this wave's (in a request without keys: the wave stores the rows)
  bool seen;          // and that key is the new token
  bool elsewhere;     // the request's last key is not the new token, which may be any other of its keys
  int kvh;
  int before;         // slot id of the key in front of the last
  uint32_t slot;
  float position;
  u32x4_t krow[KS], vrow[VH][4];  // lane group g: dims 32 c + 8 g .. (as operand), hf 128 + 32 g + 8 i .. (as output)
  Half lo[kEarly], hi[kEarly], qwl, qwh, kwl, kwh;

  __device__ __forceinline__ NewToken(const SplitKvParams& s, const ReqInfo& r, Columns<D, 1>& c, HeadLds<D>& l, const NewTokenIds<NORM>& ids, int b,
                                      int head, bool own)
      : sp(s), columns(c), lds(l), owner(own), kvh(head) {
    const int lane = lane_id();
    // one round trip for both, beside that of the first tile's slot ids
    const int32_t* last = r.kv_len > 0 ? sp.kv_indices + r.kv_start + r.kv_len - 1 : sp.nt.out_loc + b;
    const uint32_t last_id = (uint32_t)*last;
    before = *(r.kv_len > 1 ? last - 1 : last);
    slot = ids.slot();
    elsewhere = (r.kv_len > 0) & (slot <= sp.max_slot) & (last_id != slot);
    seen = owner & (r.kv_len > 0) & (slot <= sp.max_slot) & (last_id == slot);
    q = sp.q + (int64_t)b * sp.q_stride0 + kvh * sp.group * D;
    k = sp.nt.k + (int64_t)b * sp.nt.k_stride0 + kvh * D;
    if constexpr (NORM) {
      position = (float)ids.position();
#pragma unroll
      for (int i = 0; i < kEarly; ++i) head_of(i, lo[i], hi[i]);
      const int off = E * (lane & 15);
      qwl = *reinterpret_cast<const Half*>(sp.nt.q_weight + off);
      qwh = *reinterpret_cast<const Half*>(sp.nt.q_weight + D / 2 + off);
      kwl = *reinterpret_cast<const Half*>(sp.nt.k_weight + off);
      kwh = *reinterpret_cast<const Half*>(sp.nt.k_weight + D / 2 + off);
    }
    v = sp.nt.v + (int64_t)b * sp.nt.v_stride0 + kvh * D;
    if (owner) rows();  // in front of the first tile
  }
  __device__ __forceinline__ void rows() {
    const int g = lane_id() >> 4;
#pragma unroll
    for (int hf = 0; hf < VH; ++hf)
#pragma unroll
      for (int i = 0; i < 4; ++i) vrow[hf][i] = ld_global_b128(v + hf * 128 + g * 32 + i * 8);
    if constexpr (!NORM) {
#pragma unroll
      for (int c = 0; c < KS; ++c) krow[c] = ld_global_b128(k + c * 32 + g * 8);
    }
  }

  // Row 0 is the new key, row n the head of column n - 1; four rows a trip, 16 lanes each (past the last: the last).
  __device__ __forceinline__ int row_of(int trip) const { return min(4 * trip + (lane_id() >> 4), sp.group); }
  __device__ __forceinline__ void head_of(int trip, Half& l, Half& h) const {
    const int row = row_of(trip);
    const uint16_t* src = (row == 0 ? k : q + (row - 1) * D) + E * (lane_id() & 15);
    l = *reinterpret_cast<const Half*>(src);
    h = *reinterpret_cast<const Half*>(src + D / 2);
  }
  // The wave's own writes to LDS before its reads: no barrier
  __device__ __forceinline__ static void own_writes() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

  // Sines and cosines of the position, which is there before the slot ids of the first tile are (at head_dim 128).
  __device__ __forceinline__ void angles() {
    if constexpr (NORM) {
#pragma unroll
      for (int i = lane_id(); i < D / 2; i += kWave) {
        float sn, cs;
        sincosf(rope_angle<D>(position, i, sp.nt.log2_base), &sn, &cs);
        lds.cosines[i] = cs;
        lds.sines[i] = sn;
      }
    }
  }
  __device__ __forceinline__ void normalise() {
    const int lane = lane_id(), t16 = lane & 15, g = lane >> 4, off = E * t16;
    if constexpr (D != 128) angles();
    own_writes();
    float cs[E], sn[E];
#pragma unroll
    for (int e = 0; e < E; e += 4) {
      *reinterpret_cast<f32x4_t*>(cs + e) = *reinterpret_cast<const f32x4_t*>(&lds.cosines[off + e]);
      *reinterpret_cast<f32x4_t*>(sn + e) = *reinterpret_cast<const f32x4_t*>(&lds.sines[off + e]);
    }
    auto trip = [&](int i, Half l, Half h) {
      const int row = row_of(i);
      norm_rope_head<D>(l, h, row == 0 ? kwl : qwl, row == 0 ? kwh : qwh, cs, sn, sp.nt.eps);
      *reinterpret_cast<Half*>(&lds.row[row][off]) = l;
      *reinterpret_cast<Half*>(&lds.row[row][off + D / 2]) = h;
    };
    trip(0, lo[0], hi[0]);
    if (sp.group >= 4) trip(1, lo[1], hi[1]);
    for (int i = kEarly; 4 * i <= sp.group; ++i) {
      Half l, h;
      head_of(i, l, h);
      trip(i, l, h);
    }
    own_writes();
#pragma unroll
    for (int c = 0; c < KS; ++c) {
      krow[c] = *reinterpret_cast<const u32x4_t*>(&lds.row[0][c * 32 + g * 8]);
      if (t16 < sp.group) columns.q[0][c] = *reinterpret_cast<const u32x4_t*>(&lds.row[t16 + 1][c * 32 + g * 8]);
    }
  }

  // Once, before the wave reads a row of the pool: a new token that may be any key of its request is in the pool then,
  // stored by every wave of the request.
  __device__ __forceinline__ void check() {
    if (!elsewhere) return;
    if (!owner) rows();
    if constexpr (NORM) normalise();
    store();
    wait_all_vm();
  }
  __device__ __forceinline__ void operator()() {
    __builtin_amdgcn_sched_barrier(0);
    run();
    __builtin_amdgcn_sched_barrier(0);
  }
  __device__ __forceinline__ void run() {
    if constexpr (NORM) normalise();
    if (!owner) return;
    const int g = lane_id() >> 4;
    if (seen) {  // the columns' first key: its score the maximum, its weight 1
      float score = 0.f;
#pragma unroll
      for (int c = 0; c < KS; ++c)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          score = __builtin_fmaf(value_of<F16>(columns.q[0][c][e >> 1], e & 1), value_of<F16>(krow[c][e >> 1], e & 1), score);
      columns.m[0] = sum_across<32>(sum_across<16>(score)) * sp.scale_log2e;
      columns.l[0] = g == 0 ? 1.f : 0.f;
#pragma unroll
      for (int hf = 0; hf < VH; ++hf)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int n = 0; n < 8; ++n) columns.o[0][hf][n][i] = value_of<F16>(vrow[hf][i][n >> 1], n & 1);
    }
    store();
  }
  __device__ __forceinline__ void store() const {
    const int t16 = lane_id() & 15, g = lane_id() >> 4;
    if (slot > sp.max_slot) return;  // a slot id outside the pool stores nothing
    if (t16 == 0) {
      uint16_t* to_k = sp.nt.k_pool + (int64_t)slot * sp.k_stride0 + kvh * D + g * 8;
      uint16_t* to_v = sp.nt.v_pool + (int64_t)slot * sp.v_stride0 + kvh * D + g * 32;
#pragma unroll
      for (int c = 0; c < KS; ++c) st_global_b128(to_k + c * 32, krow[c]);
#pragma unroll
      for (int hf = 0; hf < VH; ++hf)
#pragma unroll
        for (int i = 0; i < 4; ++i) st_global_b128(to_v + hf * 128 + i * 8, vrow[hf][i]);
    }
  }
};

// The new rows of a request, from their source to the pool.
template <int D>
__device__ __forceinline__ void store_new_rows(const SplitKvParams& p, int b, int kvh) {
  const int lane = lane_id();
  const uint32_t slot = (uint32_t)p.nt.out_loc[b];
  if (slot > p.max_slot || lane >= D / 8) return;
  st_global_b128(p.nt.k_pool + (int64_t)slot * p.k_stride0 + kvh * D + 8 * lane,
                 ld_global_b128(p.nt.k + (int64_t)b * p.nt.k_stride0 + kvh * D + 8 * lane));
  st_global_b128(p.nt.v_pool + (int64_t)slot * p.v_stride0 + kvh * D + 8 * lane,
                 ld_global_b128(p.nt.v + (int64_t)b * p.nt.v_stride0 + kvh * D + 8 * lane));
}

// The same without norm weights for the long walks of paged_splitkv.hip, whose two tiles leave no registers for a state
// in front of them (140 bytes of spills at head_dim 128, 196 at 256): the rows go to LDS by themselves when the walk starts
// and the new key comes into the state behind it.  Against a store launch in front, us: one request of 29 K keys, 32 / 8
// heads, 24.2 -> 22.4; two of 408-2260, 24 / 4 heads of 256, 23.3 -> 20.9; 68 of 325-1056, 16 / 8, 38.2 -> 37.0
// (larger launches lose: msgl_decode_step_workspace_bytes has the line).
template <int D>
struct NewRowsLds {
  uint16_t k[D], v[D];
  uint16_t rest[512 - 2 * D];  // a load moves 1 KiB
};
template <int D, bool F16>
struct LateToken {
  static constexpr int KS = D / 32, VH = D / 128;
  const SplitKvParams& p;
  NewRowsLds<D>& lds;  // this wave's
  bool owner, seen;    // see NewToken
  int before;
  uint32_t slot;
  __device__ __forceinline__ LateToken(const SplitKvParams& params, const ReqInfo& r, NewRowsLds<D>& l, int b, int kvh, bool own)
      : p(params), lds(l), owner(own) {
    const int32_t *loc = p.nt.out_loc + b, *last = p.kv_indices + r.kv_start + r.kv_len - 1;
    slot = (uint32_t)*loc;
    const uint32_t last_id = (uint32_t)*last;
    before = *(r.kv_len > 1 ? last - 1 : last);
    seen = owner & (slot <= p.max_slot) & (last_id == slot);
    if ((slot <= p.max_slot) & (last_id != slot)) {  // any key of its request, maybe: see NewToken::check()
      store_new_rows<D>(p, b, kvh);
      wait_all_vm();
    }
    if (owner) {
      const int lane = lane_id(), at = lane & (2 * D / 8 - 1);
      const uint16_t* src = at < D / 8 ? p.nt.k + (int64_t)b * p.nt.k_stride0 + kvh * D + 8 * at
                                       : p.nt.v + (int64_t)b * p.nt.v_stride0 + kvh * D + 8 * at - D;
      lds_direct_b128(__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)MSGL_LDS_PTR(uint16_t, &lds.k[0])), nullptr,
                      (uint64_t)reinterpret_cast<uintptr_t>(src));
    }
  }
  // Behind the walk; `walked`: its waits have been waits for the rows too.
  __device__ __forceinline__ void finish(Columns<D, 1>& c, int kvh, bool walked) {
    if (!owner) return;
    if (!walked) wait_all_vm();
    const int lane = lane_id(), g = lane >> 4;
    asm volatile("" ::: "memory");
    if (seen) {
      float score = 0.f;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const u32x4_t k = *reinterpret_cast<const u32x4_t*>(&lds.k[s * 32 + g * 8]);
#pragma unroll
        for (int e = 0; e < 8; ++e)
          score = __builtin_fmaf(value_of<F16>(c.q[0][s][e >> 1], e & 1), value_of<F16>(k[e >> 1], e & 1), score);
      }
      score = sum_across<32>(sum_across<16>(score)) * p.scale_log2e;
      const float m = fmaxf(c.m[0], score);
      const float m_safe = m == kNegInf ? 0.f : m;
      const float alpha = fast_exp2(c.m[0] - m_safe), weight = fast_exp2(score - m_safe);
      c.m[0] = m;
      c.l[0] = c.l[0] * alpha + (g == 0 ? weight : 0.f);
#pragma unroll
      for (int hf = 0; hf < VH; ++hf)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const u32x4_t v = *reinterpret_cast<const u32x4_t*>(&lds.v[hf * 128 + g * 32 + i * 8]);
#pragma unroll
          for (int n = 0; n < 8; ++n)
            c.o[0][hf][n][i] = __builtin_fmaf(weight, value_of<F16>(v[n >> 1], n & 1), c.o[0][hf][n][i] * alpha);
        }
    }
    if (slot > p.max_slot || lane >= D / 8) return;
    st_global_b128(p.nt.k_pool + (int64_t)slot * p.k_stride0 + kvh * D + 8 * lane, *reinterpret_cast<const u32x4_t*>(&lds.k[8 * lane]));
    st_global_b128(p.nt.v_pool + (int64_t)slot * p.v_stride0 + kvh * D + 8 * lane, *reinterpret_cast<const u32x4_t*>(&lds.v[8 * lane]));
  }
};
// The new tokens of a prefill call's request (kStoreRows, paged_shares.hip): rows q0 .. q0 + n - 1 of k and v.  As a rule
// they are the request's last n keys and their slots stand there in kv_indices; then the waves walk the keys in front of
// them, and one of them (the last wave of the last share) takes the new ones from their source, a tile of 32 at a time
// while its first tile is under way, and stores them.  Against a store launch in front, us: 32 requests of 8 tokens on
// 2-8 K, window 1024, 32 / 8 heads, 31.5 -> 30.0; 52 of 16, the same window, 69.3 -> 67.4; three of 3 tokens on some
// hundred 11.2 -> 9.6; one of 5 tokens 16.0 -> 14.7.  Where the slots listed are others, or the tokens are not the
// last keys, every wave of the request stores its head's rows and waits for that before it reads the pool.
template <int D, int NCT>
struct NewRows {
  static constexpr int KS = D / 32, VH = D / 128;
  const SplitKvParams& p;
  const ReqInfo& r;
  Columns<D, NCT>& columns;
  int kvh, q0, n;
  int end;                // of the keys that are walked
  bool last_keys, owner;  // the new tokens are the request's last keys; this wave takes them
  bool listed;            // their slots are the ones listed
  bool stores;            // (of several workgroups on the request's columns one stores the listed)
  uint32_t slot, id;      // lane i: slot of row i; slot id listed for its place

  __device__ __forceinline__ NewRows(const SplitKvParams& params, const ReqInfo& req, Columns<D, NCT>& c, int head, bool stores_rows)
      : p(params), r(req), columns(c), kvh(head), owner(false), stores(stores_rows) {
    const int lane = lane_id();
    q0 = req.q_start;  // (a launch of shares covers the queries from the first on)
    n = req.rows;
    last_keys = n > 0 && n <= kWave && r.prefix >= 0 && r.prefix + n == r.kv_len && r.hi > r.lo;
    end = last_keys ? max(min(r.hi, r.prefix), r.lo) : r.hi;
    slot = lane < n ? (uint32_t)p.nt.out_loc[q0 + lane] : 0u;
    id = last_keys && lane < n ? (uint32_t)p.kv_indices[r.kv_start + r.prefix + lane] : slot;
  }
  // Once, before the wave reads a row of the pool.
  __device__ __forceinline__ void check() {
    listed = last_keys && __all(lane_id() >= n || (slot == id && slot <= p.max_slot));
    if (listed) return;
    for (int i = 0; i < n; ++i) store_row(i);
    wait_all_vm();
  }
  __device__ __forceinline__ void store_row(int i) const {
    const int at = 8 * lane_id();
    const uint32_t to = (uint32_t)p.nt.out_loc[q0 + i];
    if (to > p.max_slot || at >= D) return;  // a slot id outside the pool stores nothing
    st_global_b128(p.nt.k_pool + (int64_t)to * p.k_stride0 + kvh * D + at, ld_global_b128(p.nt.k + (int64_t)(q0 + i) * p.nt.k_stride0 + kvh * D + at));
    st_global_b128(p.nt.v_pool + (int64_t)to * p.v_stride0 + kvh * D + at, ld_global_b128(p.nt.v + (int64_t)(q0 + i) * p.nt.v_stride0 + kvh * D + at));
  }
  __device__ __forceinline__ void operator()() {
    if (!owner) return;
    const int t16 = lane_id() & 15, g = lane_id() >> 4;
    for (int i0 = 0; i0 < n; i0 += 32) {
      KvTile<D> t;
      // a row's place: in the source, or in the pool
      auto k_row = [&](int i) {
        const int64_t from = (int64_t)(q0 + i) * p.nt.k_stride0, in = (int64_t)min(__shfl(id, i, kWave), p.max_slot) * p.k_stride0;
        return (listed ? p.nt.k + from : p.k_cache + in) + kvh * D;
      };
      auto v_row = [&](int i) {
        const int64_t from = (int64_t)(q0 + i) * p.nt.v_stride0, in = (int64_t)min(__shfl(id, i, kWave), p.max_slot) * p.v_stride0;
        return (listed ? p.nt.v + from : p.v_cache + in) + kvh * D;
      };
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        const uint16_t* row = k_row(min(i0 + 16 * sub + t16, n - 1));
#pragma unroll
        for (int c = 0; c < KS; ++c) t.k[sub][c] = ld_global_b128(row + c * 32 + g * 8);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint16_t* row = v_row(min(i0 + (j < 4 ? 0 : 16) + 4 * g + (j & 3), n - 1));
#pragma unroll
        for (int hf = 0; hf < VH; ++hf) t.v[hf][j] = ld_global_b128(row + hf * 128 + t16 * 8);
      }
      if (listed && stores) {
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
          const int i = i0 + 16 * sub + t16;
          uint16_t* to = p.nt.k_pool + (int64_t)(uint32_t)__shfl(slot, min(i, n - 1), kWave) * p.k_stride0 + kvh * D + g * 8;
          if (i < n) {
#pragma unroll
            for (int c = 0; c < KS; ++c) st_global_b128(to + c * 32, t.k[sub][c]);
          }
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int i = i0 + (j < 4 ? 0 : 16) + 4 * g + (j & 3);
          uint16_t* to = p.nt.v_pool + (int64_t)(uint32_t)__shfl(slot, min(i, n - 1), kWave) * p.v_stride0 + kvh * D + t16 * 8;
          if (i < n) {
#pragma unroll
            for (int hf = 0; hf < VH; ++hf) st_global_b128(to + hf * 128, t.v[hf][j]);
          }
        }
      }
      compute_tile<D, NCT, false>(p, t, r.prefix + i0, columns);
    }
    // what the walk's last tile holds past the walk's end is not visible in it
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) columns.hi[ct] = min(columns.hi[ct], end - 1);
    columns.all_hi = min(columns.all_hi, end - 1);
  }
};

}  // namespace msgl
