// Kernel parameter block and launch geometry shared by the prefill tile kernels.
#pragma once
#include <algorithm>

#include "msgl_internal.h"

namespace msgl {

struct PrefillParams {
  const uint16_t* q;
  const uint16_t* k_cache;
  const uint16_t* v_cache;
  const int32_t* qo_indptr;
  const int32_t* kv_indptr;
  const int32_t* kv_indices;
  const int32_t* prefix_lens;
  uint16_t* out;
  int64_t k_stride0, v_stride0;
  int32_t batch, n_q, n_kv, group;
  int32_t n_qblk, n_pairs;  // q blocks per (request, kv head); batch * n_kv
  int32_t xcds_per_unit;    // see prefill_xcds_per_unit()
  int32_t max_len_extend, is_cross, window;
  float scale_log2e;
  uint32_t max_slot;  // num_slots - 1: slot ids are clamped to it before they become addresses
  // key splits: each workgroup takes one contiguous share of its rows' visible keys
  // and leaves a normalised fp32 partial and a base-2 log-sum-exp per row for the merge kernel
  int32_t n_ksplit;
  int64_t part_rows;  // total_q * n_q: rows of one split's partial
  float* part_o;      // [n_ksplit][part_rows][head_dim]
  float* part_lse;    // [n_ksplit][part_rows]
  // ragged shares (see prefill_ragged_tiles()): a request's keys in shares of `ragged_tiles` tiles,
  // as many as it needs; partials are then [unit][kv head][row of the block], a unit being one
  // (request, share), and req_units[2 b], [2 b + 1] = request b's first unit and unit count
  int32_t ragged_tiles, ragged_units, ragged_rows;
  int32_t* req_units;
  // gang ranges (see prefill_gangs()): `gangs` per XCD, 0 = off; cuts closer than `gang_snap`
  // tiles to either end of a (request, kv head) move to that end; a workgroup that ends up with
  // part of a unit's keys leaves its rows in `gang_slots` and counts itself in `gang_counts`
  int32_t gangs, gang_snap;
  float* gang_slots;
  unsigned long long* gang_counts;
  unsigned long long gang_nonce;
  // query blocks in order of length (see prefill_by_length()): kv heads per XCD, 0 = off, and the
  // logarithm of the number of XCDs that share a kv head's blocks
  int32_t length_heads, length_log2_xcds;
  long long* clock_probe;  // measurement aid, see ClockProbe; nullptr: off
  // head_dim 128: above 0, one workgroup per compute unit stays for the launch and takes one block in each of
  // this many rounds (see kMaxRounds)
  int32_t length_rounds;
  uint32_t group_magic, group_shift;  // row / group of a row below 2^31: see row_to_query()
  // the queries' own rows of k and v, which the launch stores itself (see stores_in_tiles() in api.hip); out_loc nullptr:
  // they are in the pool
  struct {
    const uint16_t *k, *v;
    const int32_t* out_loc;
    uint16_t *k_pool, *v_pool;
    int64_t k_stride0, v_stride0;
    int32_t rows;     // of k and v
    uint32_t blocks;  // workgroups in front of those of store_rows_of_no_request(), which a launch that stores has
  } nt;
};

constexpr int kBN = 64;  // keys per tile
// A stale row max is kept until the new one exceeds it by this much (base-2 exponent):
// P stays below 2^kLazy, far inside bf16 / fp32 range, and O is rescaled rarely.
constexpr float kLazy = 8.0f;
// Requests are processed longest first only up to this batch size: every workgroup ranks the
// requests itself (batch^2 comparisons spread over its threads), which stops paying when there
// are many of them.
constexpr int kRankedBatch = 128;
constexpr int kPrefillBlockRows = 256;      // rows per workgroup, head_dim 128
constexpr int kPrefillBlockRows256 = 128;   // head_dim 256
// Key splits: when (requests x kv heads x query blocks) cannot fill the chip, the keys of every
// query block are shared out over several workgroups.
constexpr int kComputeUnits = 256;
constexpr int kMaxKeySplits = 32;
constexpr int kMinTilesPerSplit = 2;

inline int prefill_block_rows(int64_t head_dim) {
  return head_dim == 256 ? kPrefillBlockRows256 : kPrefillBlockRows;
}

// Workgroup ids go round the 8 XCDs.  A (request, kv head, key split) unit keeps all its query
// blocks on one XCD (they read the same keys: one L2 holds them), so units are dealt to the XCDs
// eight at a time.  The units left over when their number is no multiple of 8 would leave XCDs
// without work (a single request with 2 kv heads: 6 of 8), so up to 4 left-over units spread
// their query blocks over 8 / (their number rounded up to a power of two) XCDs each.
inline int prefill_xcds_per_unit(int64_t n_units) {
  const int64_t left = n_units % 8;
  if (left == 0 || left >= 5) return 1;
  return left == 1 ? 8 : (left == 2 ? 4 : 2);
}
// workgroups on the busiest XCD
inline int64_t prefill_blocks_per_xcd(int64_t n_units, int64_t n_qblk) {
  const int x = prefill_xcds_per_unit(n_units);
  const int64_t last_row = n_units % 8 == 0 ? 0 : (n_qblk + x - 1) / x;
  return n_units / 8 * n_qblk + last_row;
}

// Query blocks with rows, of all requests and one kv head: a request's last block counts half.
inline int64_t prefill_filled_blocks(int64_t batch, int64_t total_q, int64_t group, int block_rows) {
  return (total_q * group + block_rows - 1) / block_rows + batch / 2;
}

// Number of key splits for a launch, from sizes the host knows (the per-request lengths stay on
// the device: the average visible length stands for all of them).  The (request, kv head, split)
// units are dealt round-robin to the 8 XCDs, a unit brings its query blocks, and an XCD runs its
// workgroups in rounds of one per compute unit.  A launch then takes about
//   rounds x (10 us + 1.2 us x tiles / k)  +  for k > 1: 8 us + k partials written and read at 12 TB/s
// (a block's beginning and end; a tile; the merge launch and the wait in front of it).  On 500 launches of 1-10
// requests of 5-2500 tokens on prefixes up to 30 K, of even and uneven lengths, with and without a window or a causal
// mask, at 7 head configurations of both head sizes, each timed with 1-16 splits, the count that this chooses is
// 1.6 % from the best on average (one pass always: 28 %; rounds / k with 3 % a split and 1024 keys or more in one:
// 9.4 %).  The best is mostly the largest that stays in one round, however short the splits (16 / 8 heads, 152 tokens on
// 1000: 32.4 us in one pass, 23.9 in 6 splits; on 4000: 38.4 in 4, 28.9 in 16), unless the partials cost
// more than it saves (32 / 8, 1000 tokens on 1000: 51 us in 1 and in 2), and a second round is rarely worth
// it (24 / 4 heads of 256, 1000 tokens on 6000: 181 us in one pass, 203 in 4 splits).
// Fewer visible keys never mean more splits: both the cost apart from the tiles and the bound grow with k.
// `forced` > 0 overrides (clamped to kMaxKeySplits).
inline int prefill_key_splits(int64_t batch, int64_t total_q, int64_t total_kv, int64_t n_kv, int64_t group,
                              int64_t max_len_extend, int64_t window, int64_t head_dim, int64_t forced) {
  if (forced > 0) return (int)(forced < kMaxKeySplits ? forced : kMaxKeySplits);
  if (batch <= 0 || max_len_extend <= 0) return 1;
  constexpr int64_t kXcds = 8, kUnitsPerXcd = kComputeUnits / kXcds;
  constexpr double kRoundUs = 10.0, kTileUs = 1.2, kMergeUs = 8.0, kPartialBytesPerUs = 12e6;
  const int block_rows = prefill_block_rows(head_dim);
  const int64_t n_qblk = (max_len_extend * group + block_rows - 1) / block_rows;
  // Requests shorter than the longest leave some of the grid's blocks empty, which end at once.  In one pass the
  // others go in order of length (see prefill_by_length()) and fill the rounds; splits of them do not, and the XCD
  // that has the longest requests' counts: a fifth on top of the average.
  const int64_t grid_blocks = batch * n_qblk, filled = prefill_filled_blocks(batch, total_q, group, block_rows);
  auto rounds = [&](int64_t k) {
    const int64_t grid = prefill_blocks_per_xcd(batch * n_kv * k, n_qblk);  // on the busiest XCD
    const int64_t uneven = (6 * grid * filled + 5 * grid_blocks - 1) / (5 * grid_blocks);
    if (k == 1 && filled < grid_blocks) return std::max(1.0, (double)(grid * filled) / (double)(grid_blocks * kUnitsPerXcd));
    return (double)((std::min(grid, uneven) + kUnitsPerXcd - 1) / kUnitsPerXcd);
  };
  if (rounds(1) > 4) return 1;  // what splits could even out is then little
  int64_t keys = total_kv / batch;
  if (window > 0 && keys > window + block_rows / group) keys = window + block_rows / group;  // a block sees that many
  const double tiles = (double)keys / kBN;
  const double partial_us = (double)total_q * (double)(n_kv * group) * (double)head_dim * 2 * sizeof(float) / kPartialBytesPerUs;
  const int64_t most = keys / (kMinTilesPerSplit * kBN) < kMaxKeySplits ? keys / (kMinTilesPerSplit * kBN) : kMaxKeySplits;
  int best = 1;
  double best_us = rounds(1) * (kRoundUs + kTileUs * tiles);
  for (int64_t k = 2; k <= most; ++k) {
    const double us = rounds(k) * (kRoundUs + kTileUs * tiles / (double)k) + kMergeUs + (double)k * partial_us;
    if (us < best_us) {
      best_us = us;
      best = (int)k;
    }
  }
  return best;
}

// Ragged shares, for launches with one query block per (request, kv head) (short query blocks:
// their cost is reading the keys).  Cutting every request's keys the same number of times makes
// the workgroups of a long request long; instead a share is `tiles` key tiles for every request,
// a request gets as many shares as it needs, and the workgroups find their (request, share) by a
// prefix sum over the requests' share counts, so the grid holds no empty workgroups beyond the
// rounding.  tiles = what gives about one workgroup per compute unit, at least kRaggedMinTiles.
// Returns 0 when the launch does not qualify.
// Every workgroup scans the share counts of all requests (LDS): up to 128 requests that is free,
// beyond it costs a workgroup 1.5-5 us, which pays only when the requests are long enough
// (mean of kRaggedLongMean keys or more: 512 requests of 1 K keys +5 %, but -40 % when one of
// them has 60 K; 1000 requests of 100 keys would lose 33 %).
constexpr int kRaggedFreeBatch = 128;
constexpr int kRaggedMaxBatch = 1024;
constexpr int kRaggedLongMean = 1024;
constexpr int kRaggedMinTiles = 8;  // 512 keys: 4-16 % faster than 16 on launches that leave CUs idle, 4 and 2 slower
inline int64_t prefill_tiles_bound(int64_t batch, int64_t total_kv) {
  return (total_kv + kBN - 1) / kBN + 2 * batch;  // sum over requests of their key tiles, at most
}
inline int prefill_ragged_tiles(int64_t batch, int64_t total_kv, int64_t n_kv, int64_t group,
                                int64_t max_len_extend, int block_rows, int64_t forced_splits) {
  if (forced_splits > 0 || batch <= 0 || batch > kRaggedMaxBatch) return 0;
  if (batch > kRaggedFreeBatch && total_kv < (int64_t)kRaggedLongMean * batch) return 0;
  if (max_len_extend * group > block_rows) return 0;
  int64_t t = (prefill_tiles_bound(batch, total_kv) * n_kv + kComputeUnits - 1) / kComputeUnits;
  if (t < kRaggedMinTiles) t = kRaggedMinTiles;
  return (int)(t < (1 << 20) ? t : (1 << 20));
}
// (request, share) units a launch can have at most
inline int64_t prefill_ragged_units(int64_t batch, int64_t total_kv, int tiles) {
  return prefill_tiles_bound(batch, total_kv) / tiles + batch;
}
// no request can need a second share: nothing to merge, no workspace
inline bool prefill_ragged_never_splits(int64_t batch, int64_t total_kv, int tiles) {
  return prefill_tiles_bound(batch, total_kv) <= tiles;
}
inline size_t prefill_ragged_workspace_bytes(int64_t batch, int64_t total_kv, int64_t n_kv, int64_t group,
                                             int64_t max_len_extend, int64_t head_dim, int tiles) {
  if (tiles <= 0 || prefill_ragged_never_splits(batch, total_kv, tiles)) return 0;
  const size_t rows = (size_t)prefill_ragged_units(batch, total_kv, tiles) * (size_t)n_kv *
                      (size_t)(max_len_extend * group);
  return rows * (size_t)(head_dim + 1) * sizeof(float) + (size_t)batch * 2 * sizeof(int32_t);
}

// Query blocks in order of length, for launches in one pass over the keys (no splits, shares or gang
// ranges).  Every XCD takes one kv head in eight of every request (fewer kv heads than XCDs: an equal part
// of one kv head's blocks, taken in turn), so the XCDs have the same work whatever the requests' lengths,
// and issues its blocks longest first, whatever request they belong to: the dispatcher then fills the
// compute units with ever shorter blocks and the last ones end together.  (With whole requests dealt to
// the XCDs one request after the other, an XCD with the two longest of four requests ran 1.5 times as long
// as the average: 4 requests of 512-1972 tokens on prefixes up to 8 K, 24 / 4 heads of 256: 1173 -> 837 us;
// 6 prompts of 771-2710 tokens, 32 / 8 heads of 128: 262 -> 247 us.)  The blocks of a
// request no longer run side by side on one XCD; what its L2 then misses, the memory-side cache has.
//
// `fresh`: see kMinFreshRounds.  The kernel's wave holds one request per lane: at most 64.  The kv heads have to go into the XCDs evenly.
// A launch of fewer blocks than compute units has no order.  Whole prompts of one length in many blocks each are even as
// they are, and at head_dim 256 gain more from a request's blocks side by side (us, side by side and in order, 24 / 4 heads: six of 1000
// tokens 112.0 and 120.1, two of 2000 122.8 and 125.5; 16 / 4: eight of 1024 101.7 and 114.7).  At head_dim 128 the order lets workgroups stay
// (below): 32 / 8 heads, four of 1000 55.4 and 46.5, eight of 1024 96.2 and 81.8, five of 1722 133.9 and 125.1, one of 8000 444 and 437; 16 / 8,
// three of 2000 68.4 and 59.4.  Below two rounds they do not stay, and one or two are better off side by side: 55 launches, in order by side by side:
// those below 0.97-1.036 (two of 3963, 16 / 8 heads, 129.9 and 134.6, two of 1981, 32 / 4, 70.5 and 72.6, one of 4000, 32 / 8, 121.8 and 122.9),
// three and more 0.87-0.98, from two rounds on 0.73-0.99.
inline bool prefill_by_length(const PrefillArgs& a, int64_t n_qblk, bool fresh = false) {
  const bool even_prompts = !a.is_cross && a.total_kv == a.total_q && a.total_q == a.batch * a.max_len_extend;
  const int64_t blocks = a.batch * a.n_kv * n_qblk;
  return a.by_length && a.batch <= 64 && (a.n_kv == 1 || a.n_kv == 2 || a.n_kv == 4 || a.n_kv % 8 == 0) &&
         (fresh || (blocks > kComputeUnits && !(even_prompts && n_qblk >= 16 && (a.head_dim == 256 || (a.batch <= 2 && blocks < 2 * kComputeUnits)))));
}

// Rounds of blocks that a workgroup may stay for.  A workgroup of the head_dim 128 kernel that ends pays for the next
// one's start: some 13 us outside the tile loop (finding the block, three dependent memory round trips, the epilogue)
// with the compute unit idle.  Instead workgroup r of an XCD's 32 takes the blocks 32 i + r of the order above, or
// 32 i + 31 - r in odd rounds i, as one stream of key tiles: the moves of a block's first tiles and its Q rows are
// under way while the block before it is computed, and a block costs 8.4 K cycles (the change, in both wave groups
// in turn, and the masks of its last tiles) beside 2.9 K a tile.  us, 32 / 8 heads unless said: prompts of 771-2710 tokens (11574 in
// all) 249.8 -> 235.3, 30 x 100-300 on up to 500 cached 83.9 -> 74.9, 16 x 50-2000 at 64 / 8 heads 408 -> 370, three
// of 1000-3000 under a window of 1024 166 -> 149.  A wave without rows computes all the same here (a loop of its own
// costs 260 bytes of spills), and of few rounds the last ones are short, so it pays from two rounds of blocks on.  Those
// are blocks with rows: requests shorter than the longest leave most of the grid empty (one extend of 88 tokens beside 63
// of 2, on 8 K keys: 4 rounds of the grid and 1.1 of blocks, 482 us and 601 with workgroups that stay; one of 4096 beside
// fifteen of 16: 32 and 2.4, 153 and 131), so they are counted from all queries, a half for each
// request's last block.  1050 launches of 1-64 even, ragged and very uneven extends, 4 and 8 kv heads, groups of 2-8, on
// up to 8 K keys, staying against not, geometric means by such rounds: up to 1 1.11, 1-1.5 1.04, 1.5-2 0.99, 2-2.5
// 0.96, 2.5-3 0.92, above 0.89; this line is 0.8 % from the better of the two on average, and four rounds of the
// grid were 2.1 %.
// The list of a workgroup's blocks is in LDS, hence the other limit (of the grid's rounds); an XCD's workgroups work on
// one kv head (the bases of the moves stay the same).
constexpr int kMinRounds = 2, kMaxRounds = 64;
// Prompts with nothing cached, whose rows of k and v the launch takes its keys from and stores (prompts_stored() in api.hip), go this
// way from one round of blocks on, those of one length too.  us, the store in front and the launch as it was then against
// this, 32 / 8 heads: 1015, 900 and 800 tokens 45.8 -> 41.8, two of 1000 36.7 -> 35.5, three 49.6 -> 40.4, four 60.0 -> 46.4, five of
// 1722 148 -> 129, 16 of 100-300 33.1 -> 26.5, 237-3333 (11574 in all) 227 -> 217, one of 3000 86.5 -> 84.5; 64 / 8: three of 1000 80.2 ->
// 69.0; 2000 and 1500 under a window of 500 52.3 -> 45.0.  Below one round: one of 1015 31.8 -> 33.0, two of 500 22.7 -> 23.0.
constexpr int kMinFreshRounds = 1;
constexpr int kMaxFreshRows = 1 << 17;  // of k and v, in a launch that takes its keys from them
// The head_dim 256 kernel takes the same list one block after the other (12 K cycles between them; a workgroup that ends
// pays for the dispatch of the next and its search on top), from 1.5 rounds of blocks on.  us: 60 prompts of up to 400 tokens, 16 / 4 heads,
// 124 -> 107, 23 of 129-1833 397 -> 382, three of 1344-2949 under a window of 64, 32 / 4, 105 -> 95, four of 512-1972 on up to 8 K 736 -> 719.
// The blocks are dealt out beforehand, by number and not by length, and those that share a request's keys drift apart: that has to do no harm.
// It does none where lengths follow from the rows' places, causal prompts with nothing cached and windows that most requests exceed (173 launches of
// 1-60 even, ragged and very uneven requests, staying against not, geometric mean, best and worst: 0.938, 0.76 and 1.10), nor where an average
// request's blocks fill their XCDs by themselves (97 on up to 16 K cached: 0.981, 0.91 and 1.02).  Requests of fewer blocks on prefixes of any length
// gain less on average, 0.993 of 359, and lose up to 1.42 where one is much longer than the others (42 requests of 87 tokens, 32 / 2 heads, one on
// 1290 cached, 45.5 and 61.8 us) or small groups' blocks each wait for their own keys (32 of up to 1269 on 4057 each, 8 / 8, 1114 and 1465).  So do
// those whose rows see all keys (80, 0.978 and 1.25), but for prompts with nothing cached and no window that cuts, the longest no longer than
// three on average: 171, 0.950, 0.80 and 1.04, others up to 1.27.
constexpr int kMinHalfRounds256 = 3;
// XCDs that share a kv head's blocks, as a logarithm
inline int prefill_log2_xcds(int64_t n_kv) { return n_kv == 1 ? 3 : n_kv == 2 ? 2 : n_kv == 4 ? 1 : 0; }
inline bool prefill_may_stay_256(const PrefillArgs& a, int64_t group) {
  if (a.is_cross)
    return a.total_kv == a.total_q && (a.window == 0 || a.window >= a.max_len_extend) && 3 * a.total_q >= a.batch * a.max_len_extend;
  if (a.total_kv == a.total_q || (a.window > 0 && a.total_kv >= a.batch * a.window)) return true;
  return a.total_q * group >= a.batch * ((kComputeUnits / 8 * kPrefillBlockRows256) << prefill_log2_xcds(a.n_kv));
}
inline int64_t prefill_length_blocks(int64_t batch, int64_t n_kv, int64_t n_qblk) {
  const int64_t heads = n_kv >= 8 ? n_kv / 8 : 1, xcds = 1 << prefill_log2_xcds(n_kv);
  return 8 * batch * heads * ((n_qblk + xcds - 1) / xcds);
}
// Rounds of a launch in order of length whose workgroups stay; 0: they don't.
inline int prefill_stay_rounds(int64_t batch, int64_t total_q, int64_t n_kv, int64_t group, int64_t n_qblk, int block_rows,
                               int min_half_rounds) {
  const int64_t rounds = (prefill_length_blocks(batch, n_kv, n_qblk) + kComputeUnits - 1) / kComputeUnits;
  const int64_t filled = 8 * prefill_filled_blocks(batch, total_q, group, block_rows);
  return n_kv <= 8 && 2 * filled >= ((int64_t)min_half_rounds * kComputeUnits << prefill_log2_xcds(n_kv)) && rounds <= kMaxRounds ? (int)rounds : 0;
}

// Gang ranges, for launches with several query blocks per (request, kv head) (chunked extends on
// long prefixes: their cost is the MFMA work, and it differs from unit to unit with the prefix).
// One workgroup per compute unit stays for the whole launch.  The 32 workgroups on an XCD form
// 32 / n_qblk gangs; a gang's workgroups take the query blocks of one unit side by side (they read
// the same keys at the same time: one L2 serves them) and the gangs share the XCD's units by
// length: the units' key tiles, laid end to end, are cut into equal ranges, one per gang, so
// every gang has the same MFMA work whatever the prefix lengths are.  A unit that a cut goes
// through is finished by the gang that gets there last: each of its parts leaves unnormalised
// rows, row maxima and row sums in its slot and counts itself; the part that counts last adds the
// others to its registers and writes the result.  Returns gangs per XCD, 0 when the launch does
// not qualify (the host knows sizes, not lengths).
//
// A gang stops at every unit's end and waits there for its longest workgroup, and a unit with fewer blocks than the
// gang has workgroups leaves some idle; blocks in order of length have neither, but pack whole blocks.  Beyond one
// round, then, gangs are for extends of about one length on long prefixes (time of gangs / of the order; 32 / 8,
// 16 / 8 and 64 / 8 heads, 2-6 rounds): on 6000 cached 0.93-1.0, 0-16 K 0.92-1.0, 0-32 K 0.91-0.99, but on 0-12 K
// 1.0-1.04, 1000-6000 1.03-1.17, 0-2000 1.1-1.2; extends of 0.3-1 of the longest 1.06-1.24 whatever the prefixes,
// of 0.8-1 like those of one length.  In one round: 0.76-0.93 on 0-8 K, 0.98-1.08 on prefixes of one length.
constexpr int kGangMaxUnits = 256;   // units per XCD
constexpr int kGangMinTiles = 48;    // key tiles per gang below which one pass per unit is kept
constexpr int kGangLongMean = 6144;  // mean keys of a request from which gangs pay beyond one round
inline int prefill_gangs(int64_t batch, int64_t total_q, int64_t total_kv, int64_t n_kv, int64_t group,
                         int64_t max_len_extend, int64_t window, int block_rows, int key_splits,
                         int64_t forced_splits, bool whatever_the_size = false) {
  if (forced_splits > 0 || key_splits > 1 || window > 0 || batch <= 0 || batch > kRankedBatch) return 0;
  const int64_t n_qblk = (max_len_extend * group + block_rows - 1) / block_rows;
  constexpr int64_t kUnitsPerXcd = kComputeUnits / 8;
  if (n_qblk < 2 || n_qblk > 16 || kUnitsPerXcd % n_qblk != 0) return 0;
  const int64_t n_pairs = batch * n_kv;
  if (n_pairs % 8 != 0 || n_pairs / 8 > kGangMaxUnits) return 0;
  const int64_t gangs = kUnitsPerXcd / n_qblk;
  if (whatever_the_size) return (int)gangs;
  if (n_pairs / 8 < gangs) return 0;  // fewer units than gangs: key splits are the tool
  if (n_pairs / 8 > gangs && (total_kv < kGangLongMean * batch || 4 * total_q < 3 * batch * max_len_extend)) return 0;
  const int64_t tiles_per_xcd = prefill_tiles_bound(batch, total_kv) * n_kv / 8;
  if (tiles_per_xcd < gangs * kGangMinTiles) return 0;
  return (int)gangs;
}
constexpr size_t kGangSlotBytes = (size_t)kPrefillBlockRows * 128 * sizeof(float) + 8 * 64 * 2 * sizeof(float);
inline size_t prefill_gang_workspace_bytes(int64_t batch, int64_t n_kv, int64_t group,
                                           int64_t max_len_extend, int gangs) {
  if (gangs <= 0) return 0;
  const int64_t n_qblk = (max_len_extend * group + kPrefillBlockRows - 1) / kPrefillBlockRows;
  const size_t slots = (size_t)8 * gangs * 2 * n_qblk;
  const size_t counts = (size_t)batch * n_kv * n_qblk;
  return slots * kGangSlotBytes + (counts * sizeof(unsigned long long) + 255) / 256 * 256;
}

inline size_t prefill_split_workspace_bytes(int64_t total_q, int64_t n_q, int64_t head_dim, int n_ksplit) {
  if (n_ksplit <= 1) return 0;
  return (size_t)n_ksplit * (size_t)total_q * (size_t)n_q * (size_t)(head_dim + 1) * sizeof(float);
}

// Combines the partials of a key-split launch into `out` (defined beside the head_dim 128 kernel).
int launch_prefill_merge(const struct PrefillParams& p, int head_dim, hipStream_t stream);

// Fills `p` and the grid size; returns MSGL_OK, or an error, or sets n_blocks = 0 for an
// empty problem.  wide: some pool byte offset needs more than 32 bits.
inline int make_prefill_params(const PrefillArgs& a, PrefillParams& p, int64_t& n_blocks, bool& wide,
                               int block_rows = kPrefillBlockRows) {
  p.q = static_cast<const uint16_t*>(a.q);
  p.k_cache = static_cast<const uint16_t*>(a.k_cache);
  p.v_cache = static_cast<const uint16_t*>(a.v_cache);
  p.qo_indptr = a.qo_indptr;
  p.kv_indptr = a.kv_indptr;
  p.kv_indices = a.kv_indices;
  p.prefix_lens = a.prefix_lens;
  p.out = static_cast<uint16_t*>(a.out);
  p.k_stride0 = a.k_stride0;
  p.v_stride0 = a.v_stride0;
  p.batch = (int32_t)a.batch;
  p.n_q = (int32_t)a.n_q;
  p.n_kv = (int32_t)a.n_kv;
  p.group = (int32_t)(a.n_q / a.n_kv);
  p.max_len_extend = a.max_len_extend;
  p.is_cross = a.is_cross;
  p.window = a.window;
  p.scale_log2e = a.sm_scale * 1.4426950408889634f;
  p.max_slot = (uint32_t)(a.num_slots > 0 ? a.num_slots - 1 : 0);
  p.n_ksplit = a.key_splits > 1 ? a.key_splits : 1;
  p.part_rows = a.total_q * a.n_q;
  p.part_o = static_cast<float*>(a.workspace);
  p.part_lse = p.part_o ? p.part_o + (int64_t)p.n_ksplit * p.part_rows * a.head_dim : nullptr;
  if (p.n_ksplit > 1 && !p.part_o) return MSGL_ERR_WORKSPACE;
  const int64_t rows = (int64_t)a.max_len_extend * p.group;
  const int64_t n_qblk = (rows + block_rows - 1) / block_rows;
  const int64_t n_pairs = a.batch * a.n_kv;
  p.ragged_tiles = 0;
  p.ragged_units = 0;
  p.ragged_rows = 0;
  p.req_units = nullptr;
  p.gangs = 0;
  p.gang_snap = 0;
  p.gang_slots = nullptr;
  p.gang_counts = nullptr;
  p.gang_nonce = 0;
  p.length_heads = 0;
  p.length_log2_xcds = 0;
  p.length_rounds = 0;
  p.group_shift = 0;
  while ((1u << p.group_shift) < (uint32_t)p.group) ++p.group_shift;
  p.group_magic = (uint32_t)(((1ull << (31 + p.group_shift)) + p.group - 1) / p.group);
  p.clock_probe = clock_probe();
  p.nt.k = static_cast<const uint16_t*>(a.new_tokens.k);
  p.nt.v = static_cast<const uint16_t*>(a.new_tokens.v);
  p.nt.out_loc = a.new_tokens.out_loc;
  p.nt.k_pool = const_cast<uint16_t*>(p.k_cache);
  p.nt.v_pool = const_cast<uint16_t*>(p.v_cache);
  p.nt.k_stride0 = a.new_tokens.k_stride0;
  p.nt.v_stride0 = a.new_tokens.v_stride0;
  p.nt.rows = (int32_t)a.new_tokens.rows;
  p.nt.blocks = 0xffffffffu;
  if (a.ragged_tiles > 0 && n_qblk == 1) {
    const int64_t units = prefill_ragged_units(a.batch, a.total_kv, a.ragged_tiles);
    p.n_ksplit = 1;
    p.ragged_tiles = a.ragged_tiles;
    p.ragged_units = (int32_t)units;
    p.ragged_rows = (int32_t)rows;
    if (!prefill_ragged_never_splits(a.batch, a.total_kv, a.ragged_tiles)) {
      if (!a.workspace) return MSGL_ERR_WORKSPACE;
      const int64_t part_rows = units * a.n_kv * rows;
      p.part_rows = part_rows;
      p.part_o = static_cast<float*>(a.workspace);
      p.part_lse = p.part_o + part_rows * a.head_dim;
      p.req_units = reinterpret_cast<int32_t*>(p.part_lse + part_rows);
    }
    n_blocks = units * a.n_kv;
    if (n_blocks > 0x7fffffffLL) return MSGL_ERR_SHAPE;
    p.n_qblk = 1;
    p.n_pairs = (int32_t)n_pairs;
    p.xcds_per_unit = 1;
    wide = (uint64_t)a.num_slots * (uint64_t)a.k_stride0 * 2u >= (1ull << 32) ||
           (uint64_t)a.num_slots * (uint64_t)a.v_stride0 * 2u >= (1ull << 32) ||
           a.num_slots >= (1 << 24) || a.k_stride0 * 2 >= (1 << 24) || a.v_stride0 * 2 >= (1 << 24);
    return MSGL_OK;
  }
  p.xcds_per_unit = prefill_xcds_per_unit(n_pairs * p.n_ksplit);
  n_blocks = 8 * prefill_blocks_per_xcd(n_pairs * p.n_ksplit, n_qblk);
  if (n_qblk <= 0 || n_blocks <= 0) {
    n_blocks = 0;
    return MSGL_OK;
  }
  if (n_blocks > 0x7fffffffLL) return MSGL_ERR_SHAPE;
  p.n_qblk = (int32_t)n_qblk;
  p.n_pairs = (int32_t)n_pairs;
  if (a.gangs > 0 && p.n_ksplit == 1 && block_rows == kPrefillBlockRows) {
    if (!a.workspace) return MSGL_ERR_WORKSPACE;
    p.gangs = a.gangs;
    // the last rows' diagonal lies in the last ceil(extend / 64) tiles of a unit: no cut goes there,
    // so every part of a unit holds keys that every row of every query block sees
    p.gang_snap = (int32_t)((a.max_len_extend + kBN - 1) / kBN + 2);
    const size_t slots = (size_t)8 * a.gangs * 2 * n_qblk;
    p.gang_slots = static_cast<float*>(a.workspace);
    p.gang_counts = reinterpret_cast<unsigned long long*>(static_cast<char*>(a.workspace) + slots * kGangSlotBytes);
    p.gang_nonce = a.gang_nonce;
    n_blocks = kComputeUnits;  // one workgroup per compute unit, 32 per XCD
  }
  if (p.gangs == 0 && p.n_ksplit == 1 && prefill_by_length(a, n_qblk, p.nt.out_loc != nullptr)) {
    p.length_heads = a.n_kv >= 8 ? (int32_t)(a.n_kv / 8) : 1;
    p.length_log2_xcds = prefill_log2_xcds(a.n_kv);
    n_blocks = prefill_length_blocks(a.batch, a.n_kv, n_qblk);
    if (n_blocks > 0x7fffffffLL) return MSGL_ERR_SHAPE;
    const int half_rounds = block_rows != kPrefillBlockRows ? kMinHalfRounds256 : 2 * (p.nt.out_loc != nullptr ? kMinFreshRounds : kMinRounds);
    if (block_rows == kPrefillBlockRows || prefill_may_stay_256(a, p.group))
      p.length_rounds = prefill_stay_rounds(a.batch, a.total_q, a.n_kv, p.group, n_qblk, block_rows, half_rounds);
    if (p.length_rounds > 0) n_blocks = kComputeUnits;
  }
  // narrow offsets: slot * row_bytes fits 32 bits and both factors fit 24 bits (one
  // full-rate 24-bit multiply per row)
  wide = (uint64_t)a.num_slots * (uint64_t)a.k_stride0 * 2u >= (1ull << 32) ||
         (uint64_t)a.num_slots * (uint64_t)a.v_stride0 * 2u >= (1ull << 32) ||
         a.num_slots >= (1 << 24) || a.k_stride0 * 2 >= (1 << 24) || a.v_stride0 * 2 >= (1 << 24);
  if (p.nt.out_loc != nullptr && p.length_rounds > 0) {  // so do the rows of k and v, which the launch reads too
    const NewTokens& n = a.new_tokens;
    wide |= (uint64_t)n.rows * (uint64_t)n.k_stride0 * 2u >= (1ull << 32) || (uint64_t)n.rows * (uint64_t)n.v_stride0 * 2u >= (1ull << 32) ||
            n.rows >= (1 << 24) || n.k_stride0 * 2 >= (1 << 24) || n.v_stride0 * 2 >= (1 << 24);
  }
  return MSGL_OK;
}

}  // namespace msgl
