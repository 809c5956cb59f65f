// LDS-direct loads, counted waits and transposing LDS reads shared by the prefill tile kernels.
#pragma once
#include <type_traits>

#include "msgl_device.h"
#include "prefill_params.h"

namespace msgl {

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));
constexpr bf16x2_t kOnes = {(__bf16)1.0f, (__bf16)1.0f};
#define MSGL_LDS_PTR(T, p) ((__attribute__((address_space(3))) T*)(p))

// 64 lanes x 16 bytes: lane l's 16 bytes at `saddr + voff` land at LDS byte lds_addr + 16 l.
// The compiler does not see the LDS write: callers wait on vmcnt and pass a barrier before
// anyone reads the destination.  M0 is written without telling the compiler (it cannot be
// named as a clobber); nothing else in these kernels uses M0.
__device__ __forceinline__ void lds_direct_b128(uint32_t lds_addr, const void* saddr, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds_addr), "v"(voff), "s"(saddr)
               : "memory");
}
__device__ __forceinline__ void lds_direct_b128(uint32_t lds_addr, const void* saddr, uint64_t voff) {
  const unsigned char* a = static_cast<const unsigned char*>(saddr) + voff;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :
               : "s"(lds_addr), "v"(a)
               : "memory");
}
// 64 lanes x 4 bytes: lane l's dword at `saddr + voff` lands at LDS byte lds_addr + 4 l.
__device__ __forceinline__ void lds_direct_b32(uint32_t lds_addr, const void* saddr, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
               :
               : "s"(lds_addr), "v"(voff), "s"(saddr)
               : "memory");
}
// s_waitcnt vmcnt(0) (expcnt and lgkmcnt fields left at their maxima).  Issued through the
// builtin so that the compiler's own wait bookkeeping sees it.
__device__ __forceinline__ void wait_all_vm() {
  __builtin_amdgcn_s_waitcnt(0x0F70);
  asm volatile("" ::: "memory");
}

// s_waitcnt vmcnt(N): returns once at most N of this wave's vector-memory loads are still in
// flight.  Loads complete in issue order, so this waits for everything older than the last N.
template <int N>
__device__ __forceinline__ void wait_vm_at_most() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit field");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
  asm volatile("" ::: "memory");
}

// Lane i of each 16-lane group receives element (i % 4) of the 8 bytes addressed by lanes
// i/4, 4 + i/4, 8 + i/4, 12 + i/4 of its group.
__device__ __forceinline__ u32x2_t lds_read_tr16(const unsigned char* p) {
  const s16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(MSGL_LDS_PTR(s16x4_t, p));
  return __builtin_bit_cast(u32x2_t, v);
}

// row / group, a multiplication: with 2^shift the power of two that holds the group, magic = ceil(2^(31 + shift) / group)
// has 32 bits and the quotient is exact for rows below 2^31 (a division is 35 instructions; eight of them where a block's rows leave
// were 1-2 % of a small launch: five prompts of 34-392 tokens 22.5 -> 22.0 us, 13 of 10-18 at head_dim 256 11.4 -> 11.0).
__device__ __forceinline__ int row_to_query(const PrefillParams& p, int row) {
  return (int)(__umulhi((uint32_t)row << 1, p.group_magic) >> p.group_shift);
}

// Workgroup id -> (unit = (request rank, kv head, key split), query block), heaviest query block
// (latest rows) first; `ok` is false for the ids that pad the grid.  Consecutive ids go to
// different XCDs.
struct BlockWork {
  int unit, qblk;
  bool ok;
};
__device__ __forceinline__ BlockWork prefill_block_work(const PrefillParams& p) {
  const int xcd = blockIdx.x & 7;
  const int seq = blockIdx.x >> 3;
  const int n_units = p.n_pairs * p.n_ksplit;
  const int whole_rows = n_units >> 3;  // rows of 8 units, one unit per XCD
  BlockWork w;
  if (seq < whole_rows * p.n_qblk) {  // all query blocks of a unit on one XCD, back to back
    w.unit = (seq / p.n_qblk) * 8 + xcd;
    w.qblk = p.n_qblk - 1 - (seq % p.n_qblk);
    w.ok = true;
  } else {  // the left-over units: each on xcds_per_unit XCDs
    const int side_by_side = 8 / p.xcds_per_unit;
    const int u = xcd % side_by_side;
    const int j = (seq - whole_rows * p.n_qblk) * p.xcds_per_unit + xcd / side_by_side;
    w.unit = whole_rows * 8 + u;
    w.qblk = p.n_qblk - 1 - j;
    w.ok = w.unit < n_units && j < p.n_qblk;
  }
  return w;
}

// Workgroup id -> query block and its request's geometry, in order of length (see prefill_by_length()).
// Lengths count in steps of an eighth to a quarter of the longest: within a step a request's blocks stay
// together, because those that run at the same time then read the same keys (strictly by length, 11 prompts
// of 3637 tokens took 1415 us instead of 1345).  The length of block i of a request does not fall with i, so
// the number of its blocks of at least T steps is a division; a wave holds a request per lane, finds the T at
// which its XCD's blocks of at least T steps pass its own number by bisection, and its place among those of
// T steps by a prefix sum.  Every wave does this for itself: one memory round trip,
// no LDS, no barrier.
// (The length is the causal one; under a window it is cut off, so that the order stays the same for all
// masks.  It decides the order only: any order is correct.)
struct LengthBlock {
  int b, kvh, qblk;
  int q_start, q_len, kv_start, kv_len, prefix;
  bool ok;
};
// STAY: see kMaxRounds
template <int ROWS, bool STAY = false>
struct LengthOrder {
  const PrefillParams& p;
  int xcd, q_start, q_len, kv_start, kv_len, prefix;  // the lane's request
  int rows, kn, first_of, blocks, in_all, longest, shift;
  __device__ __forceinline__ explicit LengthOrder(const PrefillParams& params) : p(params) {
    const int lane = lane_id();
    xcd = blockIdx.x & 7;
    // the XCDs take 8 >> length_log2_xcds kv heads side by side
    const int part = xcd >> (3 - p.length_log2_xcds), mask = (1 << p.length_log2_xcds) - 1;
    q_start = q_len = kv_start = kv_len = prefix = 0;
    if (lane < p.batch) {
      q_start = p.qo_indptr[lane];
      q_len = p.qo_indptr[lane + 1];
      kv_start = p.kv_indptr[lane];
      kv_len = p.kv_indptr[lane + 1];
      prefix = p.prefix_lens[lane];
    }
    q_len = min(q_len - q_start, p.max_len_extend);
    kv_len = max(kv_len - kv_start, 0);
    rows = q_len * p.group;
    kn = min(kv_len, p.window > 0 ? p.window + ROWS / p.group + 1 : 0x7fffffff);
    first_of = (part + lane) & mask;  // this XCD's blocks: first_of, first_of + XCDs per head, ...
    blocks = rows > 0 ? (rows + ROWS - 1) / ROWS : 0;
    in_all = in_class(blocks);
    longest = wave_max(kn);
    // 4 to 8 steps, whole key tiles; two tiles where a workgroup's blocks are laid down
    shift = STAY ? 7 : max(31 - __builtin_clz(max(longest, 1)) - 2, 6);
  }
  __device__ __forceinline__ int in_class(int below) const {  // this XCD's blocks among the first `below`
    return below > first_of ? ((below - first_of - 1) >> p.length_log2_xcds) + 1 : 0;
  }
  __device__ __forceinline__ int at_least(int steps) const {  // this XCD's blocks of the request of at least `steps` steps
    if (steps <= 0) return in_all;
    const int keys = ((steps - 1) << shift) + 1;
    const int row = p.is_cross ? 0 : max(keys - 1 - prefix, 0) * p.group;  // first row that sees so many
    return in_all - in_class(kn >= keys && row < rows ? row / ROWS : blocks);
  }
  __device__ __forceinline__ int count(int steps) const { return wave_sum(at_least(steps)) * p.length_heads; }
  // Block number `seq` of the XCD.
  __device__ __forceinline__ LengthBlock find(int seq) const {
    LengthBlock w{};
    // count(lo) > seq >= count(hi)
    int lo = 0, hi = (longest >> shift) + 2;
    if (seq >= count(0)) return w;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (count(mid) > seq) lo = mid;
      else hi = mid;
    }
    const int longer = at_least(lo + 1), equal = (at_least(lo) - longer) * p.length_heads;
    const int left = seq - wave_sum(longer) * p.length_heads;  // its number among the blocks of exactly `lo` steps
    const int incl = wave_inclusive_scan(equal), before = incl - equal;
    const int src = __builtin_amdgcn_readfirstlane(__ffsll((long long)__ballot(left >= before && left < incl)) - 1);
    const int mine = left - __builtin_amdgcn_readlane(before, src);
    const int from_top = __builtin_amdgcn_readlane(longer, src) + mine / p.length_heads;
    w.b = src;
    w.kvh = (xcd & ((8 >> p.length_log2_xcds) - 1)) + 8 * (mine % p.length_heads);
    w.qblk = __builtin_amdgcn_readlane(first_of, src) + ((__builtin_amdgcn_readlane(in_all, src) - 1 - from_top) << p.length_log2_xcds);
    w.q_start = __builtin_amdgcn_readlane(q_start, src);
    w.q_len = __builtin_amdgcn_readlane(q_len, src);
    w.kv_start = __builtin_amdgcn_readlane(kv_start, src);
    w.kv_len = __builtin_amdgcn_readlane(kv_len, src);
    w.prefix = __builtin_amdgcn_readlane(prefix, src);
    w.ok = true;
    return w;
  }
};

// Keys that some row of a block sees: row0 its first row, `floor` the granularity of the first key.
template <int ROWS, int FLOOR>
__device__ __forceinline__ void block_keys(const PrefillParams& p, int prefix, int kn, int row0, int rows_total, int* lo, int* hi) {
  const int qi_lo = row0 / p.group;
  const int qi_hi = min(rows_total - 1, row0 + ROWS - 1) / p.group;
  *hi = p.is_cross ? kn : min(kn, prefix + qi_hi + 1);
  *lo = (p.window > 0) ? max(0, prefix + qi_lo - p.window + 1) : 0;
  *lo &= ~(FLOOR - 1);
  if (*hi < *lo) *hi = *lo;
}

// The blocks of a workgroup that stays (see kMaxRounds), found by its waves side by side.
struct ListedBlock {
  int kvh, qblk, q_start, q_len, kv_start, kv_len, prefix;
  int k_lo, k_hi, n_tiles;  // keys that some row of the block sees, from a whole tile on
};
struct BlockList {
  ListedBlock block[kMaxRounds];
  int count, blank;  // blocks; whether one has no keys
};
// How many there are, those without keys among them.  All threads of the workgroup.
template <int THREADS, int ROWS, int TILE>
__device__ __forceinline__ int list_blocks(const PrefillParams& p, BlockList& list, int tid) {
  constexpr int NW = THREADS / kWave;
  const int w = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid & (kWave - 1);
  if (tid == 0) list.count = list.blank = 0;
  const LengthOrder<ROWS, true> order(p);
  const int r = (int)(blockIdx.x >> 3), rounds = p.length_rounds;
  __syncthreads();
  for (int i = w; i < rounds; i += NW) {
    constexpr int kPerXcd = kComputeUnits / 8;
    const int seq = i * kPerXcd + ((i & 1) ? kPerXcd - 1 - r : r);
    const LengthBlock x = order.find(seq);
    if (!x.ok) break;
    ListedBlock l{x.kvh, x.qblk, x.q_start, x.q_len, x.kv_start, x.kv_len, x.prefix, 0, 0, 0};
    block_keys<ROWS, TILE>(p, l.prefix, l.kv_len, l.qblk * ROWS, l.q_len * p.group, &l.k_lo, &l.k_hi);
    l.n_tiles = (l.k_hi - l.k_lo + kBN - 1) / kBN;
    if (lane == 0) {
      list.block[i] = l;
      atomicMax(&list.count, i + 1);
      if (l.n_tiles == 0) list.blank = 1;
    }
  }
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(list.count);
}
// The list of `n_listed` goes on without the blocks that have no keys: their rows are zero.  How many are left.
template <int THREADS, int D, int ROWS>
__device__ __forceinline__ int drop_blank_blocks(const PrefillParams& p, BlockList& list, int n_listed, int tid) {
  if (__builtin_amdgcn_readfirstlane(list.blank) != 0) {
    constexpr int kPerRow = THREADS / ROWS;
    static_assert(D / kPerRow == 64, "a thread writes 64 values of a row");
    for (int i = 0; i < n_listed; ++i) {
      const ListedBlock& l = list.block[i];
      const int row = l.qblk * ROWS + tid / kPerRow, total = l.q_len * p.group;
      if (l.n_tiles == 0 && row < total) {
        const int qi = row_to_query(p, row);
        const int at = (l.q_start + qi) * p.n_q + l.kvh * p.group + row - qi * p.group;
        uint16_t* dst = p.out + (int64_t)at * D + 64 * (tid % kPerRow);
#pragma unroll
        for (int e = 0; e < 8; ++e) st_global_b128(dst + 8 * e, u32x4_t{0u, 0u, 0u, 0u});
      }
    }
    __syncthreads();
    if (tid == 0) {
      int n = 0;
      for (int i = 0; i < n_listed; ++i)
        if (list.block[i].n_tiles > 0) list.block[n++] = list.block[i];
      list.count = n;
    }
    __syncthreads();
    n_listed = __builtin_amdgcn_readfirstlane(list.count);
  }
  return n_listed;
}

// ---- ragged shares: which (request, share) is unit `u`? ------------------------------------------
// Shares of a request, from the visible keys of its only query block (rows 0 .. q_len * group - 1), the
// floor rounded down to a tile: the kernels compute the same for their block.
__device__ __forceinline__ int ragged_shares(const PrefillParams& p, int q_len, int kn, int prefix) {
  const int hi = p.is_cross ? kn : min(kn, prefix + q_len);
  const int lo = ((p.window > 0) ? max(0, prefix - p.window + 1) : 0) & ~(kBN - 1);
  return q_len > 0 ? max(1, ((max(hi - lo, 0) + kBN - 1) / kBN + p.ragged_tiles - 1) / p.ragged_tiles) : 0;
}
struct RaggedUnit {
  int request, share, count, first;  // count = shares of the request, first = its first unit
  bool ok;                           // false: `u` lies past the last unit
};
// Every thread of the workgroup calls it.  A request with rows has at least one share (which
// writes zeros if it sees no key); a request without rows has none.
template <int THREADS>
__device__ __forceinline__ RaggedUnit ragged_unit(const PrefillParams& p, int u, int tid) {
  constexpr int kChunks = kRaggedMaxBatch / kWave;
  __shared__ int count[kRaggedMaxBatch];
  __shared__ int chunk_sum[kChunks];  // shares of requests 64 c .. 64 c + 63
  __shared__ int found[4];
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  if (tid == 0) found[0] = -1;
  for (int i = tid; i < p.batch; i += THREADS) {
    count[i] = ragged_shares(p, min(p.qo_indptr[i + 1] - p.qo_indptr[i], p.max_len_extend),
                             max(p.kv_indptr[i + 1] - p.kv_indptr[i], 0), p.prefix_lens[i]);
  }
  __syncthreads();
  const int n_chunks = (p.batch + kWave - 1) / kWave;
  for (int c = wave; c < n_chunks; c += THREADS / kWave) {
    const int i = c * kWave + lane;
    int v = i < p.batch ? count[i] : 0;
    v = wave_sum(v);
    if (lane == 0) chunk_sum[c] = v;
  }
  __syncthreads();
  int base = 0, c = 0;  // the chunk that holds unit u: the same for every thread
  for (; c < n_chunks; ++c) {
    const int sum = chunk_sum[c];
    if (u < base + sum) break;
    base += sum;
  }
  if (c < n_chunks && wave == 0) {
    const int i = c * kWave + lane;
    const int v = i < p.batch ? count[i] : 0;
    const int first = base + wave_inclusive_scan(v) - v;
    if (v > 0 && u >= first && u < first + v) {
      found[0] = i;
      found[1] = u - first;
      found[2] = v;
      found[3] = first;
    }
  }
  __syncthreads();
  RaggedUnit r;
  r.request = found[0];
  r.share = found[1];
  r.count = found[2];
  r.first = found[3];
  r.ok = found[0] >= 0;
  return r;
}

// ---- gang ranges: which parts of which units does this workgroup take? ---------------------------
// (prefill_gangs() in prefill_params.h says what they are for.)  Workgroup id -> XCD id % 8, gang
// (id / 8) / n_qblk, member (id / 8) % n_qblk = its query block in every unit.  The XCD's units are
// (request rank, kv head) pairs number i * 8 + xcd, i = 0 .. U - 1, longest requests first; unit i
// is `len` key tiles long (those the member's query block sees).  The units' tiles laid end to end
// are cut at multiples of ceil(total / gangs); a cut that falls within `gang_snap` tiles of either
// end of a unit moves to that end.  The workgroups of one member compute the same plan in every gang.
struct GangPlan {
  int first_unit, last_unit;  // units that overlap this gang's range (first > last: none)
  int lo, hi;                 // the gang's range [lo, hi) in tiles of the XCD's unit stream
};
struct GangLds {
  int order[kRankedBatch];           // request of rank r
  int kv_start[kRankedBatch], kv_len[kRankedBatch], q_start[kRankedBatch], q_len[kRankedBatch],
      prefix[kRankedBatch];          // per request (q_len capped by max_len_extend)
  int len[kGangMaxUnits];            // tiles of unit i
  int start[kGangMaxUnits + 1];      // its place in the stream; start[U] = total
  int cuts[kComputeUnits / 8 + 1];   // cuts[g] .. cuts[g + 1]: range of gang g
  int nonempty_before[kGangMaxUnits + 1];  // units with tiles in front of unit i
  int first_unit, last_unit;
  int cost_at;
};
constexpr int kGangUnitCost = 5;
// Every thread of the workgroup calls it (it holds barriers).
template <int THREADS>
__device__ __forceinline__ GangPlan gang_plan(const PrefillParams& p, GangLds& L, int xcd, int gang, int member,
                                              int block_rows, int tid) {
  __shared__ __attribute__((aligned(16))) int lens[kRankedBatch];
  const int padded = (p.batch + 3) & ~3;
  // every request's geometry in one round trip; the parts of the launch read it from here
  for (int i = tid; i < padded; i += THREADS) {
    int len = (int)0x80000000;
    if (i < p.batch) {
      const int k0 = p.kv_indptr[i], k1 = p.kv_indptr[i + 1], q0 = p.qo_indptr[i], q1 = p.qo_indptr[i + 1];
      len = k1 - k0;
      L.kv_start[i] = k0;
      L.q_start[i] = q0;
      L.q_len[i] = min(q1 - q0, p.max_len_extend);
      L.prefix[i] = p.prefix_lens[i];
    }
    lens[i] = len;
  }
  if (tid == 0) {
    L.first_unit = 0x7fffffff;
    L.last_unit = -1;
  }
  __syncthreads();
  for (int i = tid; i < p.batch; i += THREADS) {  // rank of request i: longer ones, and equal ones before it
    const int len_i = lens[i];
    int rank = 0;
    for (int j = 0; j < padded; j += 4) {
      const i32x4_t l4 = *reinterpret_cast<const i32x4_t*>(&lens[j]);
#pragma unroll
      for (int e = 0; e < 4; ++e) rank += (l4[e] > len_i) || (l4[e] == len_i && j + e < i);
    }
    L.order[rank] = i;
    L.kv_len[i] = max(len_i, 0);
  }
  __syncthreads();
  const int n_units = p.n_pairs / 8;
  for (int i = tid; i < n_units; i += THREADS) {
    const int b = L.order[(i * 8 + xcd) / p.n_kv];
    const int ql = L.q_len[b];
    const int kn = L.kv_len[b];
    // the tiles this workgroup's own query block sees: the members of a gang cut the same unit at
    // (slightly) different tiles, each so that its own work is level with that of its peers in
    // the other gangs (a cut by the longest block would leave the later blocks of every unit,
    // which see more keys, up to n_qblk - 1 tiles per unit behind)
    const int q_hi = min(ql, ((member + 1) * block_rows + p.group - 1) / p.group);  // past its last query
    const int hi = p.is_cross ? kn : min(kn, L.prefix[b] + q_hi);
    // a block with rows but no visible key still has to write its zeros: one (empty) tile
    L.len[i] = member * block_rows < ql * p.group ? max(1, (hi + kBN - 1) / kBN) : 0;
  }
  __syncthreads();
  if (tid < kWave) {  // exclusive prefix sums, 64 units at a time
    int base = 0, base_n = 0;
    for (int i0 = 0; i0 < n_units; i0 += kWave) {
      const int i = i0 + tid;
      const int v = i < n_units ? L.len[i] : 0;
      const int incl = wave_inclusive_scan(v);
      const int incl_n = wave_inclusive_scan(v > 0 ? 1 : 0);
      if (i < n_units) {
        L.start[i] = base + incl - v;
        L.nonempty_before[i] = base_n + incl_n - (v > 0 ? 1 : 0);
      }
      base += __shfl(incl, kWave - 1, kWave);
      base_n += __shfl(incl_n, kWave - 1, kWave);
    }
    if (tid == 0) {
      L.start[n_units] = base;
      L.nonempty_before[n_units] = base_n;
    }
  }
  __syncthreads();
  // Cuts, one after the other, in a stream where every unit also takes kGangUnitCost places in
  // front of its tiles (what a workgroup spends on starting and finishing a unit, in tile times):
  // each cut takes an equal share of what lies behind the cut before it (a cut that moved to a
  // unit's end changes what is left).  cost_at = place of the latest cut in that stream.
  const int total = L.start[n_units];
  if (tid == 0) {
    L.cuts[0] = 0;
    L.cuts[p.gangs] = total;
    L.cost_at = 0;
  }
  __syncthreads();
  // units with tiles in front of unit i (their unit costs precede its place in the cost stream)
  auto cost_start = [&](int i) { return L.start[i] + kGangUnitCost * L.nonempty_before[i]; };
  const int cost_total = total + kGangUnitCost * L.nonempty_before[n_units];
  for (int g = 1; g < p.gangs; ++g) {
    const int prev = L.cost_at;
    const int want = prev + (cost_total - prev + (p.gangs - g)) / (p.gangs - g + 1);
    __syncthreads();  // everyone has read cost_at
    for (int i = tid; i < n_units; i += THREADS) {
      const int n = L.len[i];
      const int c0 = cost_start(i);
      if (n > 0 && want >= c0 && want < c0 + kGangUnitCost + n) {  // exactly one unit holds place `want`
        int o = max(want - c0 - kGangUnitCost, 0);                  // tile of the unit the cut falls on
        o = o < p.gang_snap ? 0 : (n - o < p.gang_snap ? n : o);
        L.cuts[g] = L.start[i] + o;
        L.cost_at = o == 0 ? c0 : (o == n ? c0 + kGangUnitCost + n : c0 + kGangUnitCost + o);
      }
    }
    if (tid == 0 && want >= cost_total) {
      L.cuts[g] = total;
      L.cost_at = cost_total;
    }
    __syncthreads();
  }
  GangPlan plan;
  plan.lo = L.cuts[gang];
  plan.hi = L.cuts[gang + 1];
  for (int i = tid; i < n_units; i += THREADS) {
    const int s0 = L.start[i], n = L.len[i];
    if (n > 0 && s0 < plan.hi && s0 + n > plan.lo) {
      atomicMin(&L.first_unit, i);
      atomicMax(&L.last_unit, i);
    }
  }
  __syncthreads();
  plan.first_unit = L.first_unit;
  plan.last_unit = L.last_unit;
  return plan;
}
// Slot (0 or 1) that gang g's part of the unit starting at stream tile `unit_start` uses: 0 if the
// part begins where the gang's range begins, else 1 (then it is the part the range's end cuts).
__device__ __forceinline__ int gang_slot_of(const GangLds& L, int g, int unit_start) {
  return unit_start <= L.cuts[g] ? 0 : 1;
}

// The request whose kv length has rank `want_rank` in decreasing order (ties: lower index first),
// found by the workgroup itself: lengths into LDS once, then each thread ranks one request
// against all of them with broadcast LDS reads.  (Ranking straight from global memory cost every
// workgroup of a 64-request launch 3.4 us.)  Every thread of the workgroup calls it; beyond
// kRankedBatch requests the order is the batch order.
template <int THREADS>
__device__ __forceinline__ int request_of_rank(const int32_t* kv_indptr, int batch, int want_rank, int tid) {
  if (batch > kRankedBatch) return want_rank;  // many requests balance by their number
  __shared__ __attribute__((aligned(16))) int lens[kRankedBatch];
  __shared__ int found;
  const int padded = (batch + 3) & ~3;
  for (int i = tid; i < padded; i += THREADS)
    lens[i] = i < batch ? kv_indptr[i + 1] - kv_indptr[i] : (int)0x80000000;
  __syncthreads();
  for (int i = tid; i < batch; i += THREADS) {
    const int len_i = lens[i];
    int rank = 0;
    for (int j = 0; j < padded; j += 4) {
      const i32x4_t l4 = *reinterpret_cast<const i32x4_t*>(&lens[j]);
#pragma unroll
      for (int e = 0; e < 4; ++e) rank += (l4[e] > len_i) || (l4[e] == len_i && j + e < i);
    }
    if (rank == want_rank) found = i;
  }
  __syncthreads();
  return found;
}

// A block's request where every one has a lane of the wave: all that a block wants to know of it comes in one memory
// round trip, and every wave finds it by itself (a round trip, two barriers and some 0.5 us less at a block's beginning).
struct RequestPlace {
  int b, q_start, q_len, kv_start, kv_len, prefix;  // q_len: not capped
  RaggedUnit unit;                                  // of a launch in ragged shares
  bool ok;
};
// `at`: the wanted unit of ragged shares, or else the wanted rank by length
__device__ __forceinline__ RequestPlace place_in_lanes(const PrefillParams& p, int at) {
  const int lane = lane_id(), i = min(lane, p.batch - 1);
  const int q_start = p.qo_indptr[i], q_end = p.qo_indptr[i + 1], kv_start = p.kv_indptr[i], kv_end = p.kv_indptr[i + 1];
  const int prefix = p.prefix_lens[i], kv_len = max(kv_end - kv_start, 0);
  RequestPlace r{};
  unsigned long long hit;
  int n = 0, first = 0;
  if (p.ragged_tiles > 0) {
    n = lane < p.batch ? ragged_shares(p, min(q_end - q_start, p.max_len_extend), kv_len, prefix) : 0;
    first = wave_inclusive_scan(n) - n;
    hit = __ballot(at >= first && at < first + n);
  } else {
    int rank = 0;
    for (int o = 0; o < p.batch; ++o) {
      const int other = __builtin_amdgcn_readlane(kv_end - kv_start, o);
      rank += (other > kv_end - kv_start) || (other == kv_end - kv_start && o < lane);
    }
    hit = __ballot(lane < p.batch && rank == at);
  }
  if (hit == 0) return r;
  const int src = __builtin_amdgcn_readfirstlane(__ffsll((long long)hit) - 1);
  r.b = src;
  r.q_start = __builtin_amdgcn_readlane(q_start, src);
  r.q_len = __builtin_amdgcn_readlane(q_end, src) - r.q_start;
  r.kv_start = __builtin_amdgcn_readlane(kv_start, src);
  r.kv_len = __builtin_amdgcn_readlane(kv_len, src);
  r.prefix = __builtin_amdgcn_readlane(prefix, src);
  r.unit.request = src;
  r.unit.first = __builtin_amdgcn_readlane(first, src);
  r.unit.share = at - r.unit.first;
  r.unit.count = __builtin_amdgcn_readlane(n, src);
  r.unit.ok = r.ok = true;
  return r;
}
// The same of any number of requests.
template <int THREADS>
__device__ __forceinline__ RequestPlace place_of(const PrefillParams& p, int at, int tid) {
  if (p.batch <= kWave) return place_in_lanes(p, at);
  RequestPlace r{};
  if (p.ragged_tiles > 0) {
    r.unit = ragged_unit<THREADS>(p, at, tid);
    if (!r.unit.ok) return r;
    r.b = r.unit.request;
  } else {
    r.b = request_of_rank<THREADS>(p.kv_indptr, p.batch, at, tid);
  }
  r.b = __builtin_amdgcn_readfirstlane(r.b);
  r.q_start = p.qo_indptr[r.b];
  r.q_len = p.qo_indptr[r.b + 1] - r.q_start;
  r.kv_start = p.kv_indptr[r.b];
  r.kv_len = max(p.kv_indptr[r.b + 1] - r.kv_start, 0);
  r.prefix = p.prefix_lens[r.b];
  r.ok = true;
  return r;
}

// Rows of k and v in front of the first request's and behind the last's are stored by nobody's block: kRestBlocks
// workgroups behind the others take them, all heads of a row at once, and as a rule end after one round trip.  (Spread
// over the launch's own workgroups they cost the tile loop of head_dim 128 12 bytes of spills.)  `n`: what the launch's
// parameters say about its new rows.  False: not one of those workgroups.
template <int THREADS, typename P, typename N>
__device__ __forceinline__ bool store_rows_of_no_request(const P& p, const N& n, int width, int tid) {
  if (blockIdx.x < n.blocks) return false;
  const int front = min(max(p.qo_indptr[0], 0), n.rows), end = min(max(p.qo_indptr[p.batch], front), n.rows);
  for (int i = blockIdx.x - n.blocks; i < front + n.rows - end; i += kRestBlocks) {
    const int64_t row = i < front ? i : i - front + end;
    const uint32_t slot = (uint32_t)n.out_loc[row];
    if (slot > p.max_slot) continue;  // a slot id outside the pool stores nothing
    for (int e = 8 * tid; e < width; e += 8 * THREADS) {
      st_global_b128(n.k_pool + (int64_t)slot * p.k_stride0 + e, ld_global_b128(n.k + row * n.k_stride0 + e));
      st_global_b128(n.v_pool + (int64_t)slot * p.v_stride0 + e, ld_global_b128(n.v + row * n.v_stride0 + e));
    }
  }
  return true;
}

// Whether every request's rows of the launch are its keys, from the first on, and their slots those that it lists: then keys
// and values can be had from the rows.  All threads of the workgroup; 1-2 us for the 12 K rows of six prompts.
template <int THREADS>
__device__ __forceinline__ bool rows_are_the_keys(const PrefillParams& p, int tid) {
  bool same = (uint32_t)p.nt.rows <= p.max_slot + 1u;  // a row's number passes where slot ids are held inside the pool
  for (int b = tid; b < p.batch; b += THREADS) {
    const int start = p.qo_indptr[b], end = p.qo_indptr[b + 1];
    same &= p.kv_indptr[b] == start && p.kv_indptr[b + 1] == end && p.prefix_lens[b] == 0 && start >= 0 && end <= p.nt.rows &&
            end - start <= p.max_len_extend;
  }
  const int end = min(p.qo_indptr[p.batch], p.nt.rows);
  constexpr int U = 8;
  for (int i0 = max(p.qo_indptr[0], 0) + tid; i0 < end; i0 += THREADS * U) {
    int32_t slot[U], id[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      slot[u] = p.nt.out_loc[min(i0 + u * THREADS, end - 1)];
      id[u] = p.kv_indices[min(i0 + u * THREADS, end - 1)];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) same &= slot[u] == id[u] && (uint32_t)slot[u] <= p.max_slot;
  }
  return __syncthreads_and(same) != 0;
}

// A request's new rows of k and v of one kv head into the pool, by the whole workgroup, before it reads the pool: every
// workgroup of a small launch does it for its own request (the same bytes, several times), which is less than the
// launch that it saves.
template <int THREADS, int D>
__device__ __forceinline__ void store_request_rows(const PrefillParams& p, int q_start, int n, int kvh, int tid) {
  constexpr int LANES = D / 8, ROWS = THREADS / LANES;  // of a row, side by side
  const int col = kvh * D + 8 * (tid % LANES);
  auto trips = [&](auto in_flight) {
    constexpr int U = decltype(in_flight)::value;
    for (int r0 = tid / LANES; r0 < n; r0 += ROWS * U) {
      uint32_t slot[U];
      u32x4_t k[U], v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t row = q_start + min(r0 + u * ROWS, n - 1);
        slot[u] = (uint32_t)p.nt.out_loc[row];
        k[u] = ld_global_b128(p.nt.k + row * p.nt.k_stride0 + col);
        v[u] = ld_global_b128(p.nt.v + row * p.nt.v_stride0 + col);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (r0 + u * ROWS >= n || slot[u] > p.max_slot) continue;  // a slot id outside the pool stores nothing
        st_global_b128(p.nt.k_pool + (int64_t)slot[u] * p.k_stride0 + col, k[u]);
        st_global_b128(p.nt.v_pool + (int64_t)slot[u] * p.v_stride0 + col, v[u]);
      }
    }
  };
  if (n <= ROWS) trips(std::integral_constant<int, 1>{});
  else if (n <= 4 * ROWS) trips(std::integral_constant<int, 4>{});
  else trips(std::integral_constant<int, 8>{});
  wait_all_vm();
  __syncthreads();
}

}  // namespace msgl
