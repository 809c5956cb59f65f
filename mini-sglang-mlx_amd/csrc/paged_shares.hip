// Paged attention for short query blocks (decode, verify) when the launch is small for the chip:
// one workgroup per share of a request's keys, no second launch.
//
// The segment kernel (paged_splitkv.hip) is made for launches that the memory system bounds: one
// round of equal segments, a merge launch behind it.  On a small launch what counts is the chain of
// round trips and the second launch: a decode step of 4 requests with 1.7 K tokens in all took
// 14 us of attention and 4 us of merge, one after the other, for 0.9 MB per layer and head group.
//
// Work decomposition
//   A request's visible keys are cut into ceil(keys / share_len) equal shares.  A workgroup takes one
//   share of `heads_wg` adjacent kv heads; `share_waves` waves cut the share of each head into
//   adjacent ranges, so a share is read with every load of its first tiles in flight at once.  The
//   waves of a head meet in LDS.  (The columns of small launches go to several workgroups, a tile or two to each: col_groups_of().)
//   The grid holds the largest number of shares the sizes allow; a workgroup finds its (request, share) with one
//   wave-wide prefix sum over kv_indptr and takes the request's geometry from the same registers; a workgroup past the last share ends.
//   A request with one share is written at once.  Otherwise the share's normalised fp32 partial and
//   its log-sum-exp go to the workspace, the workgroup counts itself in the request's count word, and
//   the one that counts last reads the others and writes the result: nobody waits for anybody.
//   Partials and counts travel at agent scope (they cross XCDs).  A count word is
//   launch number << 16 | shares done; any other word counts as zero, so the workspace
//   needs no clearing (launch_number.h: why no data is taken for one), and the last share puts the word back to zero, so a captured launch replays.
//
// A decode step's new tokens (NEW) are stored here, normalised and rotated before where the step asks for that
//   (new_token.h), instead of by a launch in front.  Norm, rotary embedding, store and attention of 4 requests of
//   36-1022 tokens, 16 / 8 heads: 3.5 + 8.9 us in two launches, 9.8 in one (8.1 since), and one launch's host time less (28 layers
//   359 -> 281 us, now 240); store and attention of 24 requests of 127-4095, 16 / 2 heads of 256: 4.5 + 25.0 us, 26.0 in one (25.6 since).
#include <algorithm>
#include <cmath>

#include "launch_number.h"
#include "new_token.h"

namespace msgl {
namespace {

struct ShareParams {
  SplitKvParams s;
  unsigned long long* counts;  // [batch][head_groups][col_groups]
  unsigned long long nonce;
  int32_t heads_wg, head_groups;
};

// What the way to a workgroup's share takes (see request_info()).  These are the kernel's first arguments, one by one, which
// the launch leaves in scalar registers (-amdgpu-kernarg-preload-count, build.py).  Read where they were needed, the parameters were
// some eight round trips of 0.2-0.5 us in a workgroup's 8 us, three of them in front of its first load; in registers, or fetched
// together behind that load, with divisions that are multiplications: 28 layers of a step of 4 requests of 36-1022 tokens 269.7 ->
// 246.2 us, 32 requests of 8 queries with a window of 1024 34.4 -> 33.5, 24 of 127-4095 tokens, 16 / 2 heads of 256, 27.1 -> 26.7.
struct ShareStart {
  const int32_t *kv_indptr, *qo_indptr, *prefix_lens;
  int32_t batch, share_len, window, max_len_extend, q_cap, is_cross;
  uint32_t len_magic, len_shift;  // x / share_len = high half of x * len_magic, >> len_shift
  static constexpr int q_begin = 0;
  __device__ __forceinline__ int shares_of(int keys) const {
    return (int)(__umulhi((uint32_t)(keys + share_len - 1), len_magic) >> len_shift);
  }
};
struct ShareShape {  // powers of two: waves on a head; head groups (kNoShift: they are none).  Column groups
  static constexpr uint32_t kNoShift = 255;
  uint32_t bits;
  __host__ __device__ ShareShape(uint32_t len_shift, uint32_t waves, uint32_t groups, uint32_t col_groups)
      : bits(len_shift | waves << 8 | groups << 16 | col_groups << 24) {}
  __host__ __device__ explicit ShareShape(uint32_t b) : bits(b) {}
  __device__ __forceinline__ uint32_t len_shift() const { return bits & 0xffu; }
  __device__ __forceinline__ uint32_t waves() const { return (bits >> 8) & 0xffu; }
  __device__ __forceinline__ uint32_t groups() const { return (bits >> 16) & 0xffu; }
  __device__ __forceinline__ uint32_t col_groups() const { return bits >> 24; }
};
// ceil(a / b) of scalars, b > 0 and the result below 2^20 (the compiler's division is twice as long)
__device__ __forceinline__ int ceil_div(int a, int b) {
  int q = __builtin_amdgcn_readfirstlane((int)((float)a * __builtin_amdgcn_rcpf((float)b)));
  const int rest = a - q * b;  // q is within one of a / b
  if (rest > 0) ++q;
  if (rest > b) ++q;
  if (rest <= -b) --q;
  return q;
}

__device__ __forceinline__ void st_agent(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long ld_agent(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// 16 bytes of the partials at agent scope.  (As two 8-byte accesses, the largest there are of atomics, each of them walks all
// the lines that the wave's 16-byte pieces lie in: 24 loads of a thread took 1.5 K cycles to be issued, 48 of head_dim 256 3.8 K.)
constexpr int kAgentScope = 16;  // sc1
struct Partials {
  __amdgpu_buffer_rsrc_t at;
  __device__ __forceinline__ Partials(float* from, uint32_t bytes) : at(__builtin_amdgcn_make_buffer_rsrc(from, 0, bytes, 0x00020000)) {}
  __device__ __forceinline__ f32x4_t load(uint32_t lane_at, uint32_t share_at) const {
    return __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(at, (int)lane_at, (int)share_at, kAgentScope));
  }
  __device__ __forceinline__ void store(uint32_t lane_at, f32x4_t v) const {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), at, (int)lane_at, 0, kAgentScope);
  }
};
template <typename F, int... I>
__device__ __forceinline__ void each(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

// Share number `item` of the launch: its request, which of the request's shares it is, of how many; a lane's `other`: one of the requests
// around it.  All lanes must call; false past the last share.  The launch's other parameters are fetched while the first requests' lengths are.
template <int PARAMETERS>
__device__ __forceinline__ bool find_share(const ShareStart& p, int item, ReqInfo* r, int* b, int* share, int* n_shares, OtherKeys* other) {
  const int lane = lane_id();
  int base = 0;
  for (int b0 = 0; b0 < p.batch; b0 += kWave) {
    const ReqInfo mine = request_info(p, min(b0 + lane, p.batch - 1), [&] {
      if (b0 != 0) return;
      __builtin_amdgcn_sched_barrier(0);
      fetch_parameters<PARAMETERS>();
      __builtin_amdgcn_sched_barrier(0);
    });
    // a request without visible keys has one empty share: its rows are zero
    const int n = b0 + lane < p.batch ? max(p.shares_of(mine.hi - mine.lo), 1) : 0;
    const int incl = wave_inclusive_scan(n);
    const int sum = __builtin_amdgcn_readlane(incl, kWave - 1);
    if (item < base + sum) {
      const int first = base + incl - n;
      const unsigned long long hit = __ballot(item >= first && item < first + n);
      const int src = __builtin_amdgcn_readfirstlane(__ffsll((long long)hit) - 1);
      r->kv_start = __builtin_amdgcn_readlane(mine.kv_start, src);
      r->kv_len = __builtin_amdgcn_readlane(mine.kv_len, src);
      r->q_start = __builtin_amdgcn_readlane(mine.q_start, src);
      r->q_len = __builtin_amdgcn_readlane(mine.q_len, src);
      r->prefix = __builtin_amdgcn_readlane(mine.prefix, src);
      r->lo = __builtin_amdgcn_readlane(mine.lo, src);
      r->hi = __builtin_amdgcn_readlane(mine.hi, src);
      r->rows = __builtin_amdgcn_readlane(mine.rows, src);
      *b = b0 + src;
      *share = item - __builtin_amdgcn_readlane(first, src);
      *n_shares = __builtin_amdgcn_readlane(n, src);
      *other = OtherKeys{mine.kv_start, lane == src || b0 + lane >= p.batch ? 0 : mine.kv_len};
      return true;
    }
    base += sum;
  }
  return false;
}

struct Nothing {
  template <typename... Args>
  __device__ __forceinline__ explicit Nothing(const Args&...) {}
};

template <int D, int NCT, int NW>
struct ShareLds {
  static constexpr int kCols = 16 * NCT;
  static constexpr int kBlock = kCols * 8 + 8;  // floats of one block of 8 dims: [col][8], padded
  __attribute__((aligned(16))) float part[NW][D / 8][kBlock];
  float2 state[NW][kCols];  // (maximum, sum) of a wave's columns
  int is_last;
};
// A wave's place: share `item` of the launch, number `share` of the `n_shares` of request b; its kv head, the number of that in the
// workgroup and the wave's of the `share_waves` on it; its keys; the request's columns that the workgroup has.
struct SharePlace {
  int item, b, share, n_shares, kvh, sub, sw, share_waves, t_begin, t_end, col0, ncols;
  unsigned long long* cnt;
  unsigned long long fresh;
};

// From a share's first slot ids on.  (All of it: a branch around the walk alone costs the kernel 20-40 spilled registers.)
template <int D, int NCT, int NW, int WALK, bool F16, int NEW, typename NewIds, typename Rows>
__device__ __forceinline__ void attend_share(const ShareParams& sp, const SplitKvParams& p, ShareLds<D, NCT, NW>& lds, const SharePlace& place, const ReqInfo& r,
                                             FirstIds& ids, Columns<D, NCT>& c, const NewIds& new_ids, Rows& new_rows) {
  constexpr int VH = D / 128;
  auto& part = lds.part;
  auto& state = lds.state;
  auto& is_last = lds.is_last;
  const int item = place.item, share = place.share, n_shares = place.n_shares, kvh = place.kvh, sub = place.sub, share_waves = place.share_waves;
  const int t_begin = place.t_begin, t_end = place.t_end, col0 = place.col0, ncols = place.ncols;
  unsigned long long* const cnt = place.cnt;
  const unsigned long long fresh = place.fresh;
  const int lane = lane_id();
  const int t16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if constexpr (NEW == kStored) {
    start_columns<D, NCT, true, true>(p, r, kvh, col0 >> 4, t_end, c);
    if (t_begin < t_end) attend_keys<D, NCT, WALK, F16, true>(p, r, kvh, t_begin, t_end, ids, c, [] {});
  } else if constexpr (NEW == kStoreRows) {
    new_rows.owner = new_rows.last_keys && share == n_shares - 1 && place.sw == share_waves - 1;
    start_columns<D, NCT, true, true>(p, r, kvh, col0 >> 4, new_rows.owner ? r.hi : t_end, c);
    new_rows.check();
    if (t_begin < t_end) attend_keys<D, NCT, WALK, F16, true>(p, r, kvh, t_begin, t_end, ids, c, new_rows);
    else new_rows();
  } else {
    static_assert(sizeof(HeadLds<D>) <= sizeof(part[0]), "a wave's heads have their place in its part of the partials");
    const int tail = r.kv_len - 1;
    const bool owner = r.kv_len > 0 ? t_begin <= tail && tail < t_end : share == 0 && place.sw == 0;
    NewToken<D, NEW == kNormRopeStore, F16> token(p, r, c, *reinterpret_cast<HeadLds<D>*>(&part[wave][0][0]), new_ids, place.b, kvh, owner);
    if constexpr (D == 128) token.angles();
    int walk_end = t_end;
    if (token.seen) {
      walk_end = tail;
      end_ids(ids, t_begin, tail, token.before);
    }
    token.check();
    start_columns<D, NCT, NEW != kNormRopeStore, true>(p, r, kvh, 0, walk_end, c);
    if constexpr (D == 256) {
      token();
      if (t_begin < walk_end) attend_keys<D, NCT, WALK, F16, true>(p, r, kvh, t_begin, walk_end, ids, c, [] {});
    } else {
      if (t_begin < walk_end) attend_keys<D, NCT, WALK, F16, true>(p, r, kvh, t_begin, walk_end, ids, c, token);
      else if (owner) token();
    }
  }

  // ---- the waves of a kv head meet in LDS ---------------------------------------------------
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    float l = c.l[ct];
    l = sum_across<16>(l);
    l = sum_across<32>(l);
    const int col = ct * 16 + t16;
    if (col >= ncols) continue;
    if (g == 0) state[wave][col] = float2{c.m[ct], l};
#pragma unroll
    for (int hf = 0; hf < VH; ++hf)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f32x4_t w0, w1;
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          w0[n] = c.o[ct][hf][n][i];
          w1[n] = c.o[ct][hf][4 + n][i];
        }
        float* dst = &part[wave][hf * 16 + 4 * g + i][col * 8];
        *reinterpret_cast<f32x4_t*>(dst) = w0;
        *reinterpret_cast<f32x4_t*>(dst + 4) = w1;
      }
  }
  __syncthreads();

  constexpr int kQuads = D / 4;  // a thread's unit of work: 4 dims of one column, the 16 bytes at 16 it of a share's rows
  const int threads = 64 * share_waves;
  const int64_t row0 = ((int64_t)item * p.n_kv + kvh) * p.cols + col0;
  const Partials own(p.part_o + row0 * D, (uint32_t)(ncols * D * 4));
  // Every wave's part of a quad is asked for before the first is used.  The lanes of a row of 16 work on one column: lane w has
  // wave w's maximum and sum, and its weight goes to the others by DPP.
  auto put_together = [&](auto waves) {
    constexpr int W = decltype(waves)::value;
    for (int it = threadIdx.x - sub * threads; it < ncols * kQuads; it += threads) {
      const int col = it / kQuads, d4 = (it - col * kQuads) * 4;
      float2 ml = state[sub * W + min(t16, W - 1)][col];
      f32x4_t o[W];
#pragma unroll
      for (int w = 0; w < W; ++w) o[w] = *reinterpret_cast<const f32x4_t*>(&part[sub * W + w][d4 >> 3][col * 8 + (d4 & 7)]);
      if (t16 >= W) ml = float2{kNegInf, 0.f};
      const float m = row_max16(ml.x), m_safe = (m == kNegInf) ? 0.f : m;
      const float e = fast_exp2(ml.x - m_safe);  // 0 for a wave without visible keys
      const float l = row_sum16(e * ml.y);
      f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
      each([&](auto w) { acc += of_row_lane<decltype(w)::value>(e) * o[decltype(w)::value]; }, std::make_integer_sequence<int, W>{});
      acc *= (l > 0.f) ? 1.0f / l : 0.f;
      if (n_shares == 1) {
        const int qi = query_of(p, col0 + col);
        uint16_t* dst = p.out + ((int64_t)(r.q_start + qi) * p.n_q + kvh * p.group + (col0 + col - qi * p.group)) * D + d4;
        *reinterpret_cast<u32x2_t*>(dst) = u32x2_t{pack_16x2<F16>(acc[0], acc[1]), pack_16x2<F16>(acc[2], acc[3])};
      } else {
        own.store(16u * (uint32_t)it, acc);
        if (d4 == 0)
          __hip_atomic_store(p.part_lse + row0 + col, (l > 0.f) ? m + __log2f(l) : kNegInf, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  };
  if (share_waves == NW) put_together(std::integral_constant<int, NW>{});
  else if (share_waves == NW / 2) put_together(std::integral_constant<int, NW / 2>{});
  else if (share_waves == NW / 4) put_together(std::integral_constant<int, NW / 4>{});
  else put_together(std::integral_constant<int, 1>{});
  if (n_shares == 1) return;

  // ---- the share that counts last puts the request together ------------------------------------
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's partials are where every CU sees them
  __syncthreads();
  if (threadIdx.x == 0) {
    // one addition where the word is this launch's already; an addition to a word that was not did
    // not count, and the loop counts this share whatever the others do meanwhile
    unsigned long long seen = __hip_atomic_fetch_add(cnt, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    unsigned long long want = seen + 1;
    if ((seen >> 16) != sp.nonce) {
      seen = ld_agent(cnt);
      do {
        want = ((seen >> 16) == sp.nonce ? seen : fresh) + 1;
      } while (!__hip_atomic_compare_exchange_strong(cnt, &seen, want, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT));
    }
    const bool last = (int)(want & 0xffff) == n_shares;
    if (last) st_agent(cnt, 0ull);
    is_last = last;
  }
  __syncthreads();
  if (!is_last) return;
  constexpr int I = NW == 4 ? 2 : 1;  // a thread's quads whose loads are in flight together
  const int64_t step = (int64_t)p.n_kv * p.cols;  // rows from one share to the next
  const int64_t first = row0 - share * step;
  const uint32_t step_bytes = (uint32_t)step * (D * 4);  // (share_plan() sees to it that a request's partials are below 2 GiB)
  const Partials all(p.part_o + first * D, (uint32_t)n_shares * step_bytes);
  const float* const lse_from = p.part_lse + first;
  const int quads = ncols * kQuads;
  // ... for as many shares as there are, by fours, or 16 (loads past the last one cost as much as the others:
  // 16 for all of four shares 9.3 -> 9.8 us; 8 for more than 8 in turns 11.6 us against 11.2 at two of 3000 tokens).
  // As above, the lanes of a row of 16 have a share's log-sum-exp each.
  auto merge = [&](auto in_flight) {
    constexpr int U = decltype(in_flight)::value;
    for (int it0 = threadIdx.x - sub * threads; it0 < quads; it0 += I * threads) {
      float m[I], l[I];
      f32x4_t acc[I];
      uint32_t at[I];
#pragma unroll
      for (int i = 0; i < I; ++i) {
        at[i] = (uint32_t)min(it0 + i * threads, quads - 1);  // past the end: the last quad again, not written
        m[i] = kNegInf;
        l[i] = 0.f;
        acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
      for (int s0 = 0; s0 < n_shares; s0 += U) {
        const int mine = min(s0 + min(t16, U - 1), n_shares - 1);
        float lse[I];
        f32x4_t o[I][U];
#pragma unroll
        for (int i = 0; i < I; ++i) {
          lse[i] = __hip_atomic_load(lse_from + mine * step + at[i] / kQuads, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
          for (int u = 0; u < U; ++u)  // shares past the last one: the last again, with weight 0
            o[i][u] = all.load(16u * at[i], (uint32_t)min(s0 + u, n_shares - 1) * step_bytes);
        }
#pragma unroll
        for (int i = 0; i < I; ++i) {
          if (t16 >= U || s0 + t16 >= n_shares) lse[i] = kNegInf;
          const float m_new = fmaxf(m[i], row_max16(lse[i]));
          const float m_safe = (m_new == kNegInf) ? 0.f : m_new;
          const float old = fast_exp2(m[i] - m_safe), e = fast_exp2(lse[i] - m_safe);
          acc[i] *= old;
          l[i] = l[i] * old + row_sum16(e);
          m[i] = m_new;
          each([&](auto u) { acc[i] += of_row_lane<decltype(u)::value>(e) * o[i][decltype(u)::value]; }, std::make_integer_sequence<int, U>{});
        }
      }
#pragma unroll
      for (int i = 0; i < I; ++i) {
        if (it0 + i * threads >= quads) break;
        const int col = col0 + (int)(at[i] / kQuads), qi = query_of(p, col);
        const f32x4_t o = acc[i] * ((l[i] > 0.f) ? 1.0f / l[i] : 0.f);
        uint16_t* dst = p.out + ((int64_t)(r.q_start + qi) * p.n_q + kvh * p.group + (col - qi * p.group)) * D + 4 * (at[i] % kQuads);
        *reinterpret_cast<u32x2_t*>(dst) = u32x2_t{pack_16x2<F16>(o[0], o[1]), pack_16x2<F16>(o[2], o[3])};
      }
    }
  };
  if (n_shares <= 4) merge(std::integral_constant<int, 4>{});
  else if (n_shares <= 8) merge(std::integral_constant<int, 8>{});
  else merge(std::integral_constant<int, 16>{});
}

// GROUPS: a request's columns go to several workgroups, kCols to each.
template <int D, int NCT, int NW, int WALK, bool F16, int NEW, bool GROUPS>
__global__ __launch_bounds__(64 * NW, (D == 128 && NCT == 1) ? 2 : 1) void share_attention_kernel(
    const int32_t* kv_indptr, const int32_t* qo_indptr, const int32_t* prefix_lens, int32_t batch, int32_t share_len, int32_t window,
    int32_t max_len_extend, int32_t q_cap, int32_t is_cross, uint32_t len_magic, uint32_t shape_bits, ShareParams params) {
  const ShareShape shape(shape_bits);
  const ShareStart start{kv_indptr, qo_indptr, prefix_lens, batch, share_len, window, max_len_extend, q_cap, is_cross, len_magic, shape.len_shift()};
  constexpr int kCols = 16 * NCT;
  __shared__ ShareLds<D, NCT, NW> lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int item, hg;
  uint32_t block = blockIdx.x, cg = 0;
  if (GROUPS) {  // the column groups of a share are on one XCD
    const uint32_t seq = block >> 3, base = seq / shape.col_groups();
    cg = seq - base * shape.col_groups();
    block = base * 8 + (block & 7);
  }
  if (shape.groups() == ShareShape::kNoShift) {
    item = block / params.head_groups;
    hg = block - item * params.head_groups;
  } else {
    item = block >> shape.groups();
    hg = block & ((1u << shape.groups()) - 1);
  }
  const int col0 = GROUPS ? (int)cg * kCols : 0;  // the first of this workgroup's columns
  const int share_waves = 1 << shape.waves();
  const int sub = wave >> shape.waves();  // which of the workgroup's kv heads
  const int sw = wave & (share_waves - 1);
  const int kvh = hg * (NW >> shape.waves()) + sub;

  ReqInfo r;
  int b, share, n_shares;
  OtherKeys other;
  constexpr int kParameters = 3 * 8 + 8 * 4 + sizeof(ShareParams);
  static_assert((3 * 8 + 8 * 4) % alignof(ShareParams) == 0, "where they are, see below");
  if (!find_share<kParameters>(start, item, &r, &b, &share, &n_shares, &other)) {  // the whole workgroup
    if constexpr (NEW == kStoreRows) (void)store_rows_of_no_request<64 * NW>(params.s, params.s.nt, params.s.n_kv * D, threadIdx.x);
    return;
  }
  // The rest of the parameters are read from here on, from lines that find_share() had fetched: loads of theirs in front of the search
  // would be waited for there (28 layers of four requests 240.3 -> 243.5 us).
  auto args = __builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(args));
  const ShareParams& sp = *reinterpret_cast<const ShareParams*>((const char*)args + (kParameters - sizeof(ShareParams)));
  const SplitKvParams& p = sp.s;
  // From here on, not from the kernel's beginning as elsewhere: the search is not in the interval.  (Stamps at the beginning cost every
  // launch 0.03 us, with a test of whether there is a probe 0.14.)
  const ClockProbe clock_probe_(p.clock_probe);
  // what the rest of the way begins with and only the request's number leads to
  const typename std::conditional<NEW == kStore || NEW == kNormRopeStore, NewTokenIds<NEW == kNormRopeStore>, Nothing>::type new_ids(p, b);
  __builtin_amdgcn_sched_barrier(0);
  const int ncols = GROUPS ? min(r.q_len * p.group - col0, kCols) : r.q_len * p.group;
  if (ncols <= 0) return;
  Columns<D, NCT> c;
  // the keys that are walked: all, but for a prefill call's own new ones
  typename std::conditional<NEW == kStoreRows, NewRows<D, NCT>, Nothing>::type new_rows(p, r, c, kvh, col0 == 0);
  int hi = r.hi;
  if constexpr (NEW == kStoreRows) hi = new_rows.end;
  const int vis = hi - r.lo;
  const int per = (ceil_div(vis, n_shares) + 31) & ~31;
  const int s_begin = min(r.lo + share * per, hi), s_end = min(s_begin + per, hi);
  const int per_wave = (((per + share_waves - 1) >> shape.waves()) + 31) & ~31;
  const int t_begin = min(s_begin + sw * per_wave, s_end), t_end = min(t_begin + per_wave, s_end);

  FirstIds ids{};
  if (t_begin < t_end) ids = first_ids(p, r, t_begin, t_end);
  const typename std::conditional<(WALK & kStream) != 0, OtherSlots, Nothing>::type other_slots(p, other, r, s_begin < s_end ? s_begin : -1);
  __builtin_amdgcn_sched_barrier(0);
  unsigned long long* const cnt = sp.counts + ((int64_t)b * sp.head_groups + hg) * (GROUPS ? shape.col_groups() : 1) + cg;
  const unsigned long long fresh = sp.nonce << 16;
  // The first share makes the count word this launch's, long before anybody counts.  Nothing waits
  // for it: whoever finds the word not made yet makes it (below).  (The last wave, which has the fewest keys or none.)
  if (n_shares > 1 && share == 0 && threadIdx.x == 64 * (NW - 1)) {
    unsigned long long seen = ld_agent(cnt);
    if ((seen >> 16) != sp.nonce)
      (void)__hip_atomic_compare_exchange_strong(cnt, &seen, fresh, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
  }
  const SharePlace place{item, b, share, n_shares, kvh, sub, sw, share_waves, t_begin, t_end, col0, ncols, cnt, fresh};
  if constexpr (WALK & kStream) {
    if (other_slots.shared())
      return attend_share<D, NCT, NW, WALK & kWide, F16, NEW>(sp, p, lds, place, r, ids, c, new_ids, new_rows);
  }
  attend_share<D, NCT, NW, WALK, F16, NEW>(sp, p, lds, place, r, ids, c, new_ids, new_rows);
}

// waves of a workgroup: two per SIMD where a wave fits 256 registers
int waves_of(int64_t head_dim, int nct) { return head_dim == 128 && nct == 1 ? 8 : 4; }

template <int D, int NCT, int NW, bool GROUPS>
int launch_shape(const ShareParams& sp, const SharePlan& plan, unsigned blocks, hipStream_t stream) {
  const int share_len = plan.share_len;
  auto log2_of = [](uint32_t x) { return 31u - (uint32_t)__builtin_clz(x); };
  // x / d for x < 2^31, d > 1: with 2^s the next power of two, m = ceil(2^(31 + s) / d), it is x m >> (31 + s)
  const uint32_t d = (uint32_t)share_len, s = log2_of(d - 1) + 1;
  const uint32_t magic = (uint32_t)(((1ull << (31 + s)) + d - 1) / d), groups = (uint32_t)sp.head_groups;
  const ShareShape shape(s - 1, log2_of((uint32_t)NW / (uint32_t)sp.heads_wg), (groups & (groups - 1)) == 0 ? log2_of(groups) : ShareShape::kNoShift,
                         (uint32_t)plan.col_groups);
  auto launch = [&](auto f16, auto mode_of) {
    constexpr bool F16 = decltype(f16)::value;
    constexpr int NEW = decltype(mode_of)::value;
    // (launches with column groups are small, 64 MiB at most, and stay in the caches)
    constexpr int kPast = GROUPS ? kNarrow : kStream;
    const auto kernel = sp.s.walk == kStream             ? share_attention_kernel<D, NCT, NW, kPast, F16, NEW, GROUPS>
                        : sp.s.walk == (kStream | kWide) ? share_attention_kernel<D, NCT, NW, kPast | kWide, F16, NEW, GROUPS>
                        : sp.s.walk == kWide             ? share_attention_kernel<D, NCT, NW, kWide, F16, NEW, GROUPS>
                                                         : share_attention_kernel<D, NCT, NW, kNarrow, F16, NEW, GROUPS>;
    return launch_kernel(kernel, dim3(blocks), dim3(64 * NW), stream, sp.s.kv_indptr, sp.s.qo_indptr, sp.s.prefix_lens,
                         sp.s.batch, (int32_t)share_len, sp.s.window, sp.s.max_len_extend, sp.s.q_cap, sp.s.is_cross, magic, shape.bits, sp);
  };
  if constexpr (NCT == 1 && !GROUPS) {  // IEEE half and new tokens exist for decode only (one column tile)
    const int mode = sp.s.nt.k == nullptr || sp.s.qo_indptr != nullptr ? kStored : sp.s.nt.q_weight == nullptr ? kStore : kNormRopeStore;
    if (sp.s.f16) {
      if (mode == kStored && sp.s.nt.k == nullptr)
        return launch(std::true_type{}, New<kStored>{});
      if (mode == kStore)
        return launch(std::true_type{}, New<kStore>{});
      return MSGL_ERR_DTYPE;
    }
    if (mode == kStore)
      return launch(std::false_type{}, New<kStore>{});
    if (mode == kNormRopeStore)
      return launch(std::false_type{}, New<kNormRopeStore>{});
  }
  if (sp.s.f16) return MSGL_ERR_DTYPE;
  if (sp.s.nt.k != nullptr)  // a prefill call's
    return launch(std::false_type{}, New<kStoreRows>{});
  return launch(std::false_type{}, New<kStored>{});
}

thread_local int64_t t_force = 0;  // benchmarking switch, see shares_force()

}  // namespace

void shares_force(int64_t v) { t_force = v; }

// (request, kv head) pairs no more than compute units: length and line from measured costs.
static bool heads_alone(int64_t batch, int64_t n_kv) { return batch * n_kv <= device_cus(); }

// Length of the shares there: of those (in steps of a third or a half from `least` on) that fit the chip in one round, requests of one
// length included, the one that costs least: its keys, what a share costs the one that puts the request together, and a round trip
// for every 16 of them, all in keys' worth of time.  Fitted to 4280 launches at head_dim 256 (decode and verify, 1-40 requests of 200-100 000
// keys, four head counts, every length that fits timed): within 1.0 % of the best length on average up to 8 columns, 1.4 % beyond; the shortest that
// fits with at most 16 shares to a request, from 256 on, and segments for fewer than 12 pairs: 16 and 11 %.
// The same costs hold at head_dim 128: 12 700 launches of up to 25 pairs within 0.3-3 % of the best, where the shortest that fits with at most 16
// shares to a request was 1-3 % from 12 pairs on, 3-44 % for 4 to 11 and up to 2x for fewer.
// Every decode step makes it twice, 28 layers of a step that the host's side bounds: the search is without divisions and ends where a length's own
// keys cost as much as the best.  A plan, eight kv heads of 128, by all lengths in floating point and by this, ns: one request of 2000 keys 52
// and 26, four of 300 34 and 22, eight of 1000 42 and 23, two of 20 K 64 and 27; two kv heads of 256, 24 of 2000, 49 and 29.
static int64_t cost_share_length(int64_t batch, int64_t keys, int64_t n_kv, int64_t cols, int64_t least, int64_t round) {
  // in a round beside half a share a request for the rounding and two standard deviations of that
  const double room = (double)round / (double)n_kv - 0.5 * (double)batch - 0.43 * std::sqrt((double)batch);
  const int64_t mean = keys / batch, most = round / (batch * n_kv);  // keys, and shares that fit the round, of a request of that length
  const int64_t put_together = cols > 8 ? 320 : 200;  // costs are in halves of a key
  bool thirds = (least & (least - 1)) != 0;  // a length is 2^shift or 3 2^shift
  int shift = 63 - __builtin_clzll((uint64_t)(thirds ? least / 3 : least));
  int64_t len = 0, lowest = 0;
  for (int64_t c = least; c < (1 << 20); c = (int64_t)(thirds ? 3 : 1) << shift) {
    const uint64_t up = (uint64_t)(mean + c - 1) >> shift;
    const int64_t of_one = std::max<int64_t>((int64_t)(thirds ? up / 3 : up), 1);
    if (of_one <= most && (double)keys <= (double)c * room) {
      const int64_t alone = std::min(2 * c, 3 * mean);
      if (len != 0 && alone + 8 >= lowest) break;
      const int64_t cost = alone + (of_one > 1 ? put_together : 0) + 8 * of_one + 200 * ((of_one + 15) / 16 - 1);
      if (len == 0 || cost < lowest) {
        len = c;
        lowest = cost;
      }
      if (c >= 2 * mean) break;
    }
    shift += thirds ? 2 : -1;
    thirds = !thirds;
  }
  return len > 0 ? len : 1 << 20;
}

// Columns in several workgroups, each of which reads all of a share's keys: for launches of one round and few keys, where the tile
// kernels' way (a block of 256 rows mostly empty, 13 us outside its loop, a merge launch) is longer.  2500 launches of 2-16 tokens a request, requests of
// up to 64 K keys with and without a window of 1024, this by that (geometric mean, worst of a bin).  head_dim 256, by keys times column groups for
// each compute unit: up to 64 0.72 (0.91), 181 0.72 (0.88), 256 0.77 (1.02), 362 0.86 (1.2), 512 0.96 (1.5), 724 1.09 (1.6); nine and ten groups 0.81 (0.94) up
// to 256, eleven and more 0.95 (1.06) and 1.2-1.7 beyond; up to 128 keys a request 0.95-1.05, more than a round of workgroups 1.1-2.
// head_dim 128, by the same, in groups of two tiles (col_groups_of() has those of one): 49-64 columns up to 256 0.73 (0.88), 512 0.82 (0.92), 724
// 0.98; 65-96 0.73 (1.04), 0.80 (0.97), 0.93 (1.11); 97-128 0.72 (0.98), 0.76 (0.96), 0.88 (1.1) (of three tiles 65-96 0.98 (1.2)); up to 192 keys a
// request 0.9-1.1, more than three quarters of a round 1.0 (1.2).  (us: 16 of 5 tokens,
// window 1024, 8 / 1 heads of 256, 34 -> 16; one of 1.7 K, 12 tokens, the same, 22 -> 12; two of 14 tokens, window 1024, 32 / 8 heads of 128, 25 -> 13.)
constexpr int64_t kXcds = 8;
static int64_t groups_keys(int64_t head_dim) { return head_dim == 256 ? 400 : 512; }  // for each compute unit
static bool groups_round(int64_t batch, int64_t keys, int64_t n_kv, int64_t slots, int64_t head_dim) {
  return head_dim == 256 ? batch * n_kv <= slots && keys > 128 * batch : 4 * batch * n_kv <= 3 * slots && keys > 192 * batch;
}

// (share, head group)s of a round, a compute unit to a workgroup; the column groups of one are on one XCD
static int64_t round_slots(int64_t col_groups) { return col_groups == 1 ? device_cus() : device_cus() / (kXcds * col_groups) * kXcds; }

// A request's columns by tiles of 16: workgroups on them, and the tiles of one (three fit a wave at head_dim 128, one at 256; of several
// workgroups two and one).  0: too many.  At head_dim 128 a workgroup to each tile where those are few enough for a round: eight waves instead of four, half
// or a third to put together.  600 launches of 17-48 columns, that by all tiles in one workgroup: two tiles 0.76-0.80 (0.91), beyond 256 keys for each
// compute unit 0.85 (1.08); three 0.60 (0.73) and 0.70 (0.83), in two workgroups 0.78 (0.93).  49-128 columns, a tile to each by two: up to
// 128 0.77 (0.85), 256 0.80 (0.89), 512 0.89 (1.03).  (us: one of 953 keys, 6 tokens, 64 / 8 heads, 18.8 -> 9.2; four of 5, window 1024, 32 / 4, 17.3
// -> 10.2; two of 722 keys in all, 10 tokens, 32 / 4, 12.8 -> 8.3.)
struct ColGroups {
  int groups, tiles;
};
static ColGroups col_groups_of(int64_t head_dim, int64_t cols, int64_t batch, int64_t keys, int64_t n_kv) {
  const bool d256 = head_dim == 256;
  const int tiles = (int)((cols + 15) / 16);
  if (tiles < 1 || tiles > (d256 ? 10 : 8)) return ColGroups{0, 0};
  const ColGroups together{1, tiles}, pairs{(tiles + 1) / 2, 2}, apart{tiles, 1};
  if (tiles == 1) return together;
  if (t_force > 0) return d256 ? apart : tiles <= 3 ? together : pairs;
  auto in_round = [&](const ColGroups& c) { return groups_round(batch, keys, n_kv, round_slots(c.groups), head_dim); };
  auto fits = [&](const ColGroups& c) { return in_round(c) && keys * n_kv * c.groups <= groups_keys(head_dim) * device_cus(); };
  if (fits(apart)) return apart;
  if (!d256 && tiles > 2 && fits(pairs)) return pairs;
  if (!d256 && tiles <= 3) return together;
  const ColGroups any = d256 ? apart : pairs;  // (too many keys, but a window, unknown where a workspace's size is asked for, may make them few)
  return in_round(any) ? any : ColGroups{0, 0};
}

SharePlan share_plan(int64_t batch, int64_t keys, int64_t each, int64_t n_kv, int64_t head_dim, int64_t cols) {
  SharePlan plan{};
  if (t_force < 0 || batch < 1) return plan;
  const auto [col_groups, nct] = col_groups_of(head_dim, cols, batch, keys, n_kv);
  if (col_groups == 0) return plan;
  const int64_t slots = round_slots(col_groups);
  const int nw = waves_of(head_dim, nct);
  int64_t heads = 1, len;
  if (t_force > 0) {
    len = std::max<int64_t>(t_force & 0xfffff, 2);
    heads = t_force >> 20;
    if (heads < 1 || heads > nw || n_kv % heads != 0 || nw % heads != 0) heads = 1;
  } else {
    // as many waves on one kv head as possible while the requests alone do not fill the chip
    while (batch * n_kv > slots * heads && 2 * heads <= nw && n_kv % (2 * heads) == 0) heads *= 2;
    // the shortest shares, in steps of a third or a half, that fit the chip in one round, and at most 16 of an
    // average request: the last of them reads the others' partials.  Rounding adds half a share per request
    // and scatters around that: with two standard deviations more, 9 requests of 102-713 keys, 64 / 8 heads, have 192 keys a share
    // and take 12.5 us, without it 128, a few workgroups more than compute units, and 16.6
    const bool alone = col_groups > 1 || heads_alone(batch, n_kv);
    len = nct == 3 ? 512 : (nw == 4 && heads == 1 && !(head_dim == 256 && alone)) ? 256 : 128;
    if (each > 0) {  // one length for all: as many equal shares as fit
      const int64_t n = std::min<int64_t>(std::max<int64_t>(slots * heads / (batch * n_kv), 1), 16);
      len = std::max(len, ((each + n - 1) / n + 31) & ~(int64_t)31);
    } else if (alone) {
      len = cost_share_length(batch, keys, n_kv, std::min<int64_t>(cols, 16 * nct), len, slots);
    } else {
      const int64_t spread = (int64_t)std::sqrt((double)batch / 3);
      auto fits = [&](int64_t c) {
        return std::max(batch, keys / c + batch / 2 + spread) * (n_kv / heads) <= slots && keys <= 16 * c * batch;
      };
      while (!fits(len) && len < (1 << 19)) len = (len & (len - 1)) ? len / 3 * 4 : len / 2 * 3;
    }
  }
  // The kernel's offsets inside one request's partials have 32 bits, its count of shares 16.  The lengths above keep to that by far
  // (128 MiB and some hundred shares), whatever the requests' number: under a window a request is one share, or a few.  One set
  // by hand is raised to what does.
  const int64_t visible = each > 0 ? each : keys, row_bytes = n_kv * cols * head_dim * 4;
  if (visible > 0xffff || visible * row_bytes > 0x7fffffffLL) {  // (else shares of one key would)
    const int64_t most_of_one = std::min<int64_t>(std::max<int64_t>(0x7fffffffLL / row_bytes, 1), 0xffff);
    len = std::max(len, (visible + most_of_one - 1) / most_of_one);
  }
  plan.share_len = (int32_t)len;
  plan.heads_wg = (int32_t)heads;
  plan.share_waves = nw / plan.heads_wg;
  plan.max_shares = keys / plan.share_len + batch;
  plan.col_groups = col_groups;
  plan.col_tiles = nct;
  return plan;
}

// Fewer visible keys make shorter shares, but never more of them than fit the chip in one round, or than requests
// where those alone are more: with n = one_round / batch, at least 1, share_plan() makes them of keys / (n batch) keys
// or more, so keys / share_len is at most n batch.
SharePlan with_any_window(SharePlan plan, int64_t batch, int64_t n_kv) {
  const int64_t one_round = device_cus() * plan.heads_wg / (n_kv * plan.col_groups);
  plan.max_shares = std::max(plan.max_shares, std::max(one_round, batch) + batch);
  return plan;
}

// head_dim 256, up to three pairs (six of one kv head), more than half a column tile: the last share's part, the others' partials, is long, and nothing
// else is left to run meanwhile.  Shares by segments, 700 launches of 1-11 pairs, geometric mean (worst): whole tiles, up to three
// pairs, decode and verify of 512-1024 keys 0.87 (0.99), 1024-2048 1.00 (1.16), to 16384 1.07 (1.24), beyond 0.85; with norm and rotary embedding,
// which go in a launch of their own then, 0.84, 0.93, 1.05 (1.23), 1.00; windows of 256 0.80, 1024 1.04 (1.10), 4096 1.11 (1.15).  9-12 columns: to 4096
// 0.85, to 16384 1.02 (1.12), beyond 0.92.  Four pairs and more 0.88 (1.16); of one kv head four to six whole tiles of 1500-2500 keys
// 1.00 (1.13), to 8000 1.06 (1.21), beyond 0.92, seven and eight to 8000 0.99.
bool few_pairs_in_segments(int64_t batch, int64_t n_kv, int64_t mean, int64_t head_dim, int64_t cols, bool windowed) {
  if (t_force > 0 || head_dim != 256 || cols <= 8) return false;
  if (batch * n_kv <= 3) return mean <= 16384 && mean > (cols <= 12 ? 4096 : windowed ? 1024 : 1536);
  return n_kv == 1 && batch <= 6 && cols > 12 && mean > 2500 && mean <= 8000;
}

// Short requests gain most against segments (a segment pays 8 us for each request boundary it crosses, us: 46 x 4-18 keys 42.1 -> 7.3,
// 64 x 20-200 18.9 -> 11.3, 4 x 37-1023 15.7 -> 9.1), and nothing any more where they fill the chip several times over.  The segments'
// fixed costs are the same for any number of bytes, while the shares' lengths vary and the longest decides: a launch beyond some
// MiB has to be one whose shares fill one round, requests of one length included.
bool shares_preferred(const SharePlan& plan, int64_t batch, int64_t keys, int64_t n_kv, int64_t head_dim, int64_t cols) {
  if (plan.share_len == 0) return false;
  if (t_force > 0) return true;
  const int64_t mb = keys * n_kv * head_dim * 4 >> 20, mean = keys / batch, units = batch * n_kv;
  if (plan.col_groups > 1) {
    // (and at head_dim 256, where a share is longer than two requests, few keys again, as below: eight requests, one of 2.7 K among 0.1 K, 24.3 us in
    // tiles and 40.3; 22 such launches 0.87 of tiles, worst 1.66, those from 200 keys for each compute unit on 1.1-1.66)
    const int64_t read = keys * n_kv * plan.col_groups, cus = device_cus();
    return read <= groups_keys(head_dim) * cus && (head_dim == 128 || plan.share_len <= 2 * mean || read <= 200 * cus);
  }
  if (mean <= 512) return mb <= 160;
  if (few_pairs_in_segments(batch, n_kv, mean, head_dim, cols, false)) return false;
  const int64_t len = plan.share_len;
  if (heads_alone(batch, n_kv)) {
    // What part of a round of shares as long as the longest they are, by MiB of keys and values; shares by segments (geometric mean,
    // worst).  head_dim 256: up to 64 0.65 (1.10), 64-128 0.76 (0.99), 128-256 from 0.5 on 0.83 (1.05) and 1.03 below, 256-420 from
    // 0.62 on 0.91 (1.07), 1.05 below, 512-724 from 0.75 on 0.95 (1.03), 0.97 (1.09) below, 1.04 below 0.62, 1024-1448 from 0.88 on 0.96
    // (0.98), 0.98 (1.07) below, 1.02 below 0.75.  (Two of 408-2260 keys, 24 / 4 heads, 21.8 -> 11.0 us; one of 51.8 K, 16 / 2, 51 -> 35.)
    const double of_round = (double)(keys * n_kv) / (std::min((double)len, 1.75 * (double)mean) * (double)device_cus());
    if (head_dim == 256) return mb <= 1400 && of_round >= 0.12 * std::log2((double)std::max<int64_t>(mb, 1)) - 0.39;
    // head_dim 128: where a share is as long as a request or longer the longest request decides, and it may be many times the mean (32 requests, one
    // of 9.7 K among 0.6 K, 27.5 us in segments and 50.4).  7700 launches, half with one or some requests 4 to 40 times the others, four sets
    // of keys in turn, by MiB and a share's length by the mean, shares by segments (the worst tenth): up to 56 0.81 (0.91); 56-104 up to 2
    // 0.84 (0.94), 1.01 (1.27) beyond; 104-128 up to 1.5 0.88 (0.98), 1.05 (1.2) beyond; 128-160 up to 0.75 0.93 (1.0), to 1.5 1.03 (1.2), 1.2 (1.45)
    // beyond; 160-190 up to 0.5 0.97 (1.05), to 1 1.04 (1.25), 1.24 (1.45) beyond; 190-256 0.97 (1.03), 1.02 from there on.
    // (One of 10 K keys, 48 / 6, 16.3 -> 15.5; two, 54 K in all, 42.1 -> 32.1; 13 of 1 K, 32 / 4, 16.6 -> 11.4.)  Few pairs with two or three tiles of
    // columns leave much to put together to the last share of each: from 16 MiB on up to five pairs 0.98-1.07 and 1.1-1.2, six to eleven of up to
    // 16 K 1.05-1.15 (1.3; one of eight 54 K, 32 columns, 24.9 and 37.9 us), of more 0.98, twelve to 15 of up to 8 K 1.07 (1.5), of more 0.93.
    if (cols > 16 && mb > 16 && (units < 6 || (units < 12 && mean <= 16384) || (units < 16 && mean <= 8192))) return false;
    // Two kinds of 56-128 MiB, 0.82-0.9 of segments as well, stay there: that a step with norm weights is refused for one request of 20 K keys, and
    // that four and five requests of 24 columns take a store in front, is what callers were told and tests hold.
    if (mb > 56 && mb <= 128 && ((units < 48 && cols > 16) || (mb <= 80 && units < 12 && mean > 12288))) return false;
    if (mb > 190) return mb <= 256 && of_round >= 0.72 + (double)(mb - 190) / 2000;
    return mb <= 56 || 48 * len <= mean * std::min<int64_t>(200 - mb, 96);
  }
  // Several heads to a workgroup.
  const int64_t head_groups = n_kv / plan.heads_wg;
  if (head_dim == 256) {
    if (mb <= 128) return true;
    const bool even_fit = batch * ((mean + len - 1) / len) * head_groups <= device_cus();  // requests of one length go in one round
    const double shares = (double)keys / (double)len + 0.5 * (double)batch + std::sqrt((double)batch / 3);  // see share_plan()
    return even_fit && shares * (double)head_groups <= device_cus() && len * plan.heads_wg <= 1024 && mb <= 256;
  }
  // 230 of the launches above: 80-128 MiB 0.95 (1.15), 128-160 1.06 (1.35), 160-190 1.17 (1.4); of lengths that differ little 0.9, 0.93 and 1.09.
  return mb <= 128;
}

size_t share_workspace_bytes(const SharePlan& plan, int64_t batch, int64_t n_kv, int64_t head_dim, int64_t cols) {
  // (under a window a request's columns may go to more workgroups, as many as tiles)
  const size_t counts = (size_t)(batch * (n_kv / plan.heads_wg) * ((cols + 15) / 16)) * sizeof(unsigned long long);
  const size_t rows = (size_t)plan.max_shares * (size_t)(n_kv * cols);
  return ((counts + 255) / 256 + (rows * (size_t)(head_dim + 1) * sizeof(float) + 255) / 256) * 256;
}

int launch_shares(const SplitKvArgs& a, const NewTokens& n, const SharePlan& plan, hipStream_t stream) {
  const int64_t group = a.n_q / a.n_kv, cols = group * a.max_len_extend;
  const int64_t head_groups = a.n_kv / plan.heads_wg;
  const bool rows = n.k != nullptr && a.qo_indptr != nullptr;  // kStoreRows
  const int64_t of_keys = plan.col_groups == 1 ? plan.max_shares * head_groups : (plan.max_shares * head_groups + 7) / 8 * 8 * plan.col_groups;
  const int64_t blocks = of_keys + (rows ? kRestBlocks : 0);
  if (blocks > 0x7fffffffLL || a.total_kv > 0x7fffffffLL) return MSGL_ERR_SHAPE;
  ShareParams sp{};
  fill_splitkv_params(a, sp.s);
  char* ws = static_cast<char*>(a.workspace);
  sp.counts = reinterpret_cast<unsigned long long*>(ws);
  ws += ((size_t)(a.batch * head_groups * plan.col_groups) * sizeof(unsigned long long) + 255) / 256 * 256;
  sp.s.part_o = reinterpret_cast<float*>(ws);
  sp.s.part_lse = sp.s.part_o + (size_t)plan.max_shares * (size_t)(a.n_kv * cols * a.head_dim);
  sp.nonce = next_launch_number();
  sp.heads_wg = plan.heads_wg;
  sp.head_groups = (int32_t)head_groups;
  fill_new_tokens(n, sp.s);
  sp.s.nt.blocks = (uint32_t)of_keys;
  const int nct = plan.col_tiles;
  const unsigned grid = (unsigned)blocks;
  if (a.head_dim == 256) return plan.col_groups > 1 ? launch_shape<256, 1, 4, true>(sp, plan, grid, stream) : launch_shape<256, 1, 4, false>(sp, plan, grid, stream);
  if (plan.col_groups > 1)
    return nct == 1 ? launch_shape<128, 1, 8, true>(sp, plan, grid, stream) : launch_shape<128, 2, 4, true>(sp, plan, grid, stream);
  if (nct == 1) return launch_shape<128, 1, 8, false>(sp, plan, grid, stream);
  return nct == 2 ? launch_shape<128, 2, 4, false>(sp, plan, grid, stream) : launch_shape<128, 3, 4, false>(sp, plan, grid, stream);
}

}  // namespace msgl
