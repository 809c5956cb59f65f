// Host-side declarations shared by the translation units of libmsgl_paged_attention.so.
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <stddef.h>
#include <stdint.h>

#include "../../include/msgl_paged_attention.h"
#include "../../include/msgl_state_pool.h"

namespace msgl {

// ---- store_kv_cache.hip ------------------------------------------------------------
int launch_store_kv_cache(void* k_cache, void* v_cache, const int32_t* indices, const void* k,
                          const void* v, int64_t length, int64_t num_slots, int64_t row_bytes,
                          int64_t k_cache_stride_bytes, int64_t v_cache_stride_bytes,
                          int64_t k_stride_bytes, int64_t v_stride_bytes, hipStream_t stream);

// The keys that the rows of a launch see, at most.
inline int64_t visible_keys(int64_t batch, int64_t total_kv, int64_t window, int64_t max_len_extend, bool is_cross) {
  if (window <= 0 || is_cross) return total_kv;
  return std::min(total_kv, batch * (window + max_len_extend + 15));  // a window starts at a multiple of 16
}

// ---- paged_splitkv.hip -------------------------------------------------------------
// One description serves decode (qo_indptr == nullptr: one query per request, every key
// visible) and the short-query route of prefill (speculative verify / draft proposal).
struct SplitKvArgs {
  const void* q;
  const void* k_cache;
  const void* v_cache;
  const int32_t* kv_indptr;
  const int32_t* kv_indices;
  const int32_t* qo_indptr;    // nullptr for decode
  const int32_t* prefix_lens;  // nullptr for decode
  void* out;
  void* workspace;
  int64_t batch, total_kv, n_q, n_kv, head_dim, num_slots;
  int64_t k_stride0, v_stride0;  // elements
  float sm_scale;
  int32_t max_len_extend;  // 1 for decode; queries per request handled by this launch
  int32_t q_begin;         // first query of every request handled by this launch
  int32_t q_cap;           // cap on a request's query count (0: max_len_extend)
  int32_t f16;             // 1: q / pools / out are IEEE half (decode only), 0: bf16
  int32_t is_cross, window;
  int32_t n_seg;    // segments the visible token stream is cut into
  int32_t min_seg;  // smallest segment length in tokens, multiple of 64
  int64_t q_stride0;  // elements from one row of q to the next (0: n_q * head_dim)
};
// What a decode step's own tokens bring: request b's new row of k and v, stored at slot out_loc[b] and taken from
// here instead of the pool where the request's last slot is that one.  With norm weights (bf16 only) q and k are
// normalised and rotated first.
struct NewTokens {
  const void* k;  // nullptr: the pool holds every row already
  const void* v;
  const void* q_weight;  // nullptr: q and k as they are
  const void* k_weight;
  const int32_t* positions;
  const int32_t* out_loc;
  int64_t k_stride0, v_stride0;  // elements
  int64_t rows;                  // of k and v
  float eps, rope_base;
};
// Workgroups that a prefill launch which stores its rows has for those of no request.
constexpr int kRestBlocks = 8;
// largest q_len * group the split-K kernel is instantiated for
constexpr int kSplitKvMaxCols = 64;
constexpr int kSplitKvMinSegment = 128;
// one resident round of workgroups for this shape, capped so segments keep min_seg tokens
int splitkv_default_segments(int64_t total_kv, int64_t n_kv, int64_t head_dim, int64_t cols,
                             int32_t min_seg);
// benchmarking switch: stream positions charged per request boundary (0: default, negative: none)
void splitkv_set_boundary(int v);
size_t splitkv_workspace_bytes(int64_t batch, int64_t n_q, int64_t n_kv, int64_t head_dim,
                               int64_t max_len_extend, int32_t n_seg);
int launch_splitkv(const SplitKvArgs& a, const NewTokens& n, hipStream_t stream);  // n without norm weights
// Address (on the current device) and size of the library's built-in split-K scratch, for the
// entry point that takes no workspace.  The first call on a device resolves the address.
int splitkv_scratch(void** ptr, size_t* bytes);
// benchmarking switch: most waves (adjacent kv heads) a split-K workgroup may hold
void splitkv_set_max_waves(int v);

// ---- paged_shares.hip --------------------------------------------------------------
// How a small launch is cut into shares of its requests' keys; share_len == 0: it is not
struct SharePlan {
  int32_t share_len;    // most keys of a share
  int32_t share_waves;  // waves per share and kv head
  int32_t heads_wg;     // adjacent kv heads of a workgroup
  int64_t max_shares;   // most shares these sizes can give
  int32_t col_groups;   // workgroups that a share's columns go to
  int32_t col_tiles;    // most tiles of 16 columns of one
};
// for `keys` visible keys in all; each > 0: about so many in every request
SharePlan share_plan(int64_t batch, int64_t keys, int64_t each, int64_t n_kv, int64_t head_dim, int64_t cols);
// the same plan with as many shares as under any sliding window: for the size of a workspace
SharePlan with_any_window(SharePlan plan, int64_t batch, int64_t n_kv);
// whether the launch is small enough for its shares to beat the segment kernel
bool shares_preferred(const SharePlan& plan, int64_t batch, int64_t keys, int64_t n_kv, int64_t head_dim, int64_t cols);
// whether segments are faster for so few (request, kv head) pairs of `mean` visible keys; windowed: all of them have as many
bool few_pairs_in_segments(int64_t batch, int64_t n_kv, int64_t mean, int64_t head_dim, int64_t cols, bool windowed);
int device_cus();  // paged_splitkv.hip
// Whether a launch that reads so many bytes, each of them once, reads them past the caches (ld_stream_b128): from where its data
// are so much of the 256 MiB of the last level that a later pass does not find them there.  us by MiB, plain and past the caches:
// decode 1253 222 -> 201, 4718 803 -> 723, verify 718 143 -> 126, window shares 129 33.0 -> 27.7.  5600 and 5700 launches of decode and verify at
// head_dim 128 and 256, three sets of keys in turn, past the caches by plain (geometric mean): 16-24 MiB 1.006 and 1.011, 32-64 1.041 and
// 1.020, 64-80 1.034 and 1.018, 80-96 0.999 and 1.003, 96-128 0.939 and 0.967, 128-1024 0.92 and 0.95.  With twelve sets, as the layers of a
// model, they cross at 24 MiB (32-48 0.978, 48-96 0.956), so the line is not higher.
constexpr int64_t kStreamKiB = 80 << 10;
bool streams(int64_t bytes, int64_t from_kib = kStreamKiB);  // paged_splitkv.hip
// benchmarking switch: from how many KiB on (0: default, negative: never)
void set_stream_kib(int64_t v);
size_t share_workspace_bytes(const SharePlan& plan, int64_t batch, int64_t n_kv, int64_t head_dim, int64_t cols);
int launch_shares(const SplitKvArgs& a, const NewTokens& n, const SharePlan& plan, hipStream_t stream);
// benchmarking switch: 0 default, negative never, else share_len | heads_wg << 20
void shares_force(int64_t v);

// ---- paged_prefill.hip -------------------------------------------------------------
struct PrefillArgs {
  const void* q;
  const void* k_cache;
  const void* v_cache;
  const int32_t* qo_indptr;
  const int32_t* kv_indptr;
  const int32_t* kv_indices;
  const int32_t* prefix_lens;
  void* out;
  int64_t batch, total_q, total_kv, n_q, n_kv, head_dim, num_slots;
  int64_t k_stride0, v_stride0;  // elements
  float sm_scale;
  int32_t max_len_extend;
  int32_t is_cross, window;
  // key splits (1: none); above 1, `workspace` holds
  // key_splits * total_q * n_q * (head_dim + 1) floats
  int32_t key_splits;
  void* workspace;
  // ragged shares instead (one query block per (request, kv head) only): key tiles per share,
  // 0 = off; `workspace` then holds prefill_ragged_workspace_bytes()
  int32_t ragged_tiles;
  // gang ranges instead (several query blocks per (request, kv head), head_dim 128 only): gangs
  // per XCD, 0 = off; `workspace` then holds prefill_gang_workspace_bytes(); `gang_nonce` is the
  // launch's number (launch_number.h)
  int32_t gangs;
  unsigned long long gang_nonce;
  int32_t by_length;  // query blocks may go in order of length (the fused kernel does not know that order)
  NewTokens new_tokens;  // k, v, out_loc: rows that the launch stores (neither gangs nor by_length then)
};
int launch_prefill_tile(const PrefillArgs& a, hipStream_t stream);     // head_dim 128
// ---- paged_prefill_d256.hip ----------------------------------------------------------
int launch_prefill_tile256(const PrefillArgs& a, hipStream_t stream);  // head_dim 256
// benchmarking switch: head_dim 128 kernel (0: ping-pong kernel, anything else: the fused kernel
// it replaced, 8 waves x 32 rows)
int tile_variant();
void set_tile_variant(int v);
// measurement aid (MSGL_TUNE_CLOCK_PROBE): two device int64 the attention kernels' workgroup 0
// fills with its shader cycles and 100 MHz wall ticks, or nullptr; one value per host thread
long long* clock_probe();

// ---- build_metadata.hip ------------------------------------------------------------
struct MetadataArgs {
  const int32_t* page_table;
  const int32_t* table_rows;
  const int32_t* kv_lens;
  const int32_t* extend_lens;  // nullptr: decode
  int32_t* kv_indptr;
  int32_t* kv_indices;
  int32_t* qo_indptr;
  int32_t* prefix_lens;
  int32_t* positions;
  int32_t* num_kv_splits;
  int64_t table_stride0, batch, n_table_rows, max_seq_len, kv_capacity, q_capacity;
  int32_t max_kv_splits;
  int32_t lens_on_host;  // table_rows, kv_lens, extend_lens are host pointers
};
// largest batch one launch handles (two scanned offset arrays and the table rows live in LDS)
constexpr int64_t kMetadataMaxBatch = 8000;
int launch_build_metadata(const MetadataArgs& a, hipStream_t stream);

// ---- qk_norm_rope_store.hip ----------------------------------------------------------
struct NormRopeArgs {
  const void* q;
  const void* k;
  const void* v;
  const void* q_weight;
  const void* k_weight;
  const int32_t* positions;
  const int32_t* out_loc;
  void* q_out;
  void* k_cache;
  void* v_cache;
  int64_t q_stride0, k_stride0, v_stride0, kc_stride0, vc_stride0;  // elements
  int64_t n_tokens, n_q, n_kv, head_dim, num_slots;
  float eps, rope_base;
};
int launch_qk_norm_rope_store(const NormRopeArgs& a, hipStream_t stream);

// ---- gdn_state.hip ---------------------------------------------------------------------
struct GdnArgs {
  const void* q;
  const void* k;
  const void* v;
  const void* g;
  const void* beta;
  void* state;
  const int32_t* slot_ids;
  const int32_t* qo_indptr;  // unused in single-token mode
  void* y;
  int64_t tokens, batch, hk, hv;
  int64_t state_stride0, q_stride0, k_stride0, v_stride0;  // elements
  int32_t single_token_mode;
  int64_t longest;  // most tokens of a request, 0: not known (the route is chosen by it, the results do not depend on it)
  void* workspace;  // may be null: requests of many chunks then take the one launch
  size_t workspace_bytes;
};
int launch_gdn_state(const GdnArgs& a, hipStream_t stream);
size_t gdn_state_workspace_bytes(int64_t tokens, int64_t batch, int64_t hv, bool single_token);
// benchmarking switch: state rows per 16-lane group (1, 2, 4; 0 = chosen from the problem size)
void gdn_set_rows(int v);

// ---- state_slots.hip -------------------------------------------------------------------
// src == nullptr: zero fill of the dst slots
int launch_state_slots(void* base, int64_t layer_stride, int64_t slot_stride, int64_t row_bytes,
                       int64_t n_layers, int64_t num_slots, const int32_t* src, const int32_t* dst,
                       int64_t n_pairs, hipStream_t stream);

// A launch without the triple brackets' detour (they put the configuration away and fetch it again, 0.2 us of host time).
template <typename T>
struct AsItIs {
  using type = T;
};
template <typename... P>
int launch_kernel(void (*kernel)(P...), dim3 grid, dim3 block, hipStream_t stream, typename AsItIs<P>::type... parameters) {
  void* at[] = {const_cast<void*>(static_cast<const void*>(&parameters))...};
  if (hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, at, 0, stream) == hipSuccess) return MSGL_OK;
  (void)hipGetLastError();  // reported here, not by a later call
  return MSGL_ERR_LAUNCH;
}

inline int check_launch() { return hipGetLastError() == hipSuccess ? MSGL_OK : MSGL_ERR_LAUNCH; }

}  // namespace msgl
