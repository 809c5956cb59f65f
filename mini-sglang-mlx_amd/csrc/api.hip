// extern "C" entry points of libmsgl_paged_attention.so: argument checks and routing.
// The checks mirror the reference's host functions (paged_decode_attention.cpp:25-62,
// paged_prefill_attention.cpp:31-76, store_kv_cache.cpp:22-63) as far as raw pointers
// and sizes can express them; rank and dtype-equality checks live in the Python shim.
#include <algorithm>

#include "launch_number.h"
#include "msgl_internal.h"
#include "prefill_params.h"

namespace {

// Benchmarking knobs live per host thread: the thread that sets one changes its own later
// calls only, so a *_workspace_bytes() call and the launch that follows it on the same thread
// always agree on the split, whatever other threads (one per stream) do.
thread_local int64_t t_tune[3] = {0, 0, 0};
thread_local int64_t t_key_splits = 0;
thread_local int64_t t_gangs = 0;  // negative: never use gang ranges
thread_local long long* t_clock_probe = nullptr;
constexpr int kTuneKnobs = 12;
thread_local int64_t t_last_set[kTuneKnobs] = {};  // what this thread last passed to msgl_set_tuning

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int check_common(const void* q, const void* k_cache, const void* v_cache, const void* out,
                 int64_t n_q, int64_t n_kv, int64_t d, int64_t k_stride0, int64_t v_stride0,
                 int32_t dtype, bool f16_ok) {
  if (d != 128 && d != 256) return MSGL_ERR_HEAD_DIM;
  if (n_q <= 0 || n_kv <= 0) return MSGL_ERR_SHAPE;
  if (n_q % n_kv != 0) return MSGL_ERR_HEAD_RATIO;
  // IEEE half exists for decode only, as in the reference (paged_decode_attention.metal:596-604
  // against paged_prefill_attention.metal:646-647)
  if (dtype != MSGL_DTYPE_BF16 && !(f16_ok && dtype == MSGL_DTYPE_F16)) return MSGL_ERR_DTYPE;
  if (k_stride0 < n_kv * d || v_stride0 < n_kv * d) return MSGL_ERR_SHAPE;
  if (!q || !k_cache || !v_cache || !out) return MSGL_ERR_NULL_POINTER;
  // 16-byte row segments are the unit of every load and store
  if (!aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(out) ||
      k_stride0 % 8 != 0 || v_stride0 % 8 != 0)
    return MSGL_ERR_ALIGNMENT;
  return MSGL_OK;
}

// Smallest segment: 128 tokens at head_dim 128 (64 changes nothing there), 64 at head_dim 256,
// where a workgroup takes twice as long per token and small launches gain 15-20 % from the
// finer cut.
int32_t min_segment(int64_t head_dim) {
  const int64_t t = t_tune[MSGL_TUNE_MIN_SEGMENT];
  if (t >= 64) return (int32_t)(t / 64 * 64);
  return head_dim == 256 ? 64 : msgl::kSplitKvMinSegment;
}
int32_t segments(int64_t total_kv, int64_t n_kv, int64_t head_dim, int64_t cols) {
  const int64_t t = t_tune[MSGL_TUNE_SEGMENTS];
  if (t >= 1) return (int32_t)(t < (1 << 20) ? t : (1 << 20));
  return msgl::splitkv_default_segments(total_kv, n_kv, head_dim, cols, min_segment(head_dim));
}
// Shares instead of segments (paged_shares.hip); a knob that shapes the segments asks for segments.
msgl::SharePlan shares_for(int64_t batch, int64_t keys, int64_t each, int64_t n_kv, int64_t head_dim, int64_t cols) {
  if (t_tune[MSGL_TUNE_SEGMENTS] != 0 || t_tune[MSGL_TUNE_MIN_SEGMENT] != 0 || t_last_set[MSGL_TUNE_SPLITKV_WAVES] != 0 ||
      t_last_set[MSGL_TUNE_SPLITKV_BOUNDARY] != 0)
    return msgl::SharePlan{};
  const msgl::SharePlan plan = msgl::share_plan(batch, keys, each, n_kv, head_dim, cols);
  return plan.col_groups > 1 && t_tune[MSGL_TUNE_SMALLQ_MAXCOLS] != 0 ? msgl::SharePlan{} : plan;
}
// Under a sliding window that most requests exceed every request shows about `window` keys: one workgroup per
// (request, kv head) is balanced as it is, whatever the requests' lengths, and needs no second launch.  Up to three
// column tiles and windows of some thousand keys the share kernel is that workgroup: 32 requests of 8 tokens,
// 32 / 8 heads, window 1024: 42.8 us in the tile kernel with its merge launch, 38 in shares; 64 of 4 tokens, 64 / 8
// heads: 76 and 61; 64 of 16, 16 / 8 heads: 76 and 63; 16 of 4, 32 / 8: 23.6 both.
// Beyond 32 columns a workgroup of several kv heads has a wave, and most of a window's time, for each (66 requests
// of 6 tokens, 64 / 8 heads: 83 us in the tile kernel, 89 in shares).
// Requests beyond one round of workgroups take whole rounds of a share's time, and a last round that leaves most of
// the chip idle costs more than the tile kernel's second launch.  Windows of 256 and 1024, 32 / 8 heads, tile or
// segment kernel against shares, us: rounds 51 % full (261 requests of 4 tokens) 65 and 78, 222 and 280; 55 % (140 of 8)
// 67 and 52, 148 and 156; 68 % (261 of 8) 126 and 87, 261 and 257; 78 % (400 of 4) 116 and 99, 332 and 308; 91 % (700
// of 4) 202 and 164, 571 and 513.
bool window_shares(const msgl::SharePlan& plan, int64_t batch, int64_t total_kv, int64_t keys, int64_t n_kv,
                   int64_t head_dim, int64_t cols) {
  if (plan.share_len == 0 || plan.col_groups > 1 || keys >= total_kv || keys > 4096 * batch || t_tune[MSGL_TUNE_SMALLQ_MAXCOLS] != 0) return false;
  if (msgl::few_pairs_in_segments(batch, n_kv, keys / batch, head_dim, cols, true)) return false;
  const int64_t blocks = batch * (n_kv / plan.heads_wg), cus = msgl::device_cus();
  if (blocks > cus && 3 * blocks < 2 * cus * ((blocks + cus - 1) / cus)) return false;
  return cols <= 32 || plan.heads_wg == 1;
}
// Largest q_len * group that takes the split-K route whatever the launch: at head_dim 128 48 (up
// to three column tiles in one wave; 49-64 columns would run on two waves per kv head that each
// read every K / V row, and the tile kernel with ragged key shares is as fast or faster on them),
// at head_dim 256 16 (one column tile; more would be a wave per tile, each reading every row,
// and the tile kernel with ragged shares is 10-65 % faster from 17 columns on).  Few keys go in shares beyond that, see
// groups_round() in paged_shares.hip.  Up to 64 columns
// the split-K kernel also takes what the tile kernels cannot give ragged shares to (very many
// or many short requests): its segments are balanced whatever the lengths, and one long request
// among many short ones would otherwise be one long workgroup per kv head.
int64_t smallq_base_cols(int64_t head_dim) { return head_dim == 128 ? 48 : 16; }
// Two column tiles of 256 dims in one wave of the split-K kernel (17 to 32 columns), which reads every row once and balances its segments
// whatever the lengths; beside the tile kernel, by MiB of keys and values (geometric mean, worst, of 150 launches): 64 1.25 (1.5), 128 1.15 (1.3), 181
// 1.0 (1.16), 256 0.92 (1.05), 362 0.81 (1.02), 512 0.79, 1024 0.72, 2048 0.67.  (us: 12 of 531 K keys in all, 6 tokens, 16 / 4 heads, 565 -> 348; six of
// 84 K, 8, 32 / 8, 193 -> 127.)  33 to 64 columns, two such waves a head, 1.0-1.1 up to 2 GiB.
bool two_tiles_in_segments(int64_t keys, int64_t n_kv, int64_t head_dim, int64_t cols) {
  return head_dim == 256 && cols > 16 && cols <= 32 && keys * n_kv * head_dim * 4 >= (int64_t)256 << 20;
}

}  // namespace

namespace msgl {
long long* clock_probe() { return t_clock_probe; }
}  // namespace msgl

extern "C" {

int msgl_version(void) { return 100; }

const char* msgl_strerror(int code) {
  switch (code) {
    case MSGL_OK: return "ok";
    case MSGL_ERR_NULL_POINTER: return "a required pointer is NULL";
    case MSGL_ERR_HEAD_DIM: return "head_dim must be 128 or 256";
    case MSGL_ERR_HEAD_RATIO: return "num_q_heads must be a multiple of num_kv_heads";
    case MSGL_ERR_GROUP_TOO_LARGE: return "only q_heads/kv_heads <= 16 is supported";
    case MSGL_ERR_DTYPE: return "unsupported dtype";
    case MSGL_ERR_BATCH: return "batch must be > 0";
    case MSGL_ERR_WINDOW: return "sliding_window_size must be >= 0";
    case MSGL_ERR_WORKSPACE: return "workspace missing or too small";
    case MSGL_ERR_SHAPE: return "invalid size or stride";
    case MSGL_ERR_ALIGNMENT: return "pointer or stride not aligned to the vector width";
    case MSGL_ERR_LAUNCH: return "HIP kernel launch failed";
    case MSGL_ERR_HEAD_DIM_MULT4: return "head_dim must be a multiple of 4";
    case MSGL_ERR_GDN_DIMS: return "this specialized kernel requires dk=dv=128";
    case MSGL_ERR_SCRATCH_LIMIT:
      return "sizes need more split-K scratch than the library's built-in 12 MiB; use the entry "
             "point that takes a workspace";
    default: return "unknown error code";
  }
}

int msgl_get_tuning(int32_t knob, int64_t* value) {
  if (!value) return MSGL_ERR_NULL_POINTER;
  if (knob < 0 || knob >= kTuneKnobs) return MSGL_ERR_SHAPE;
  *value = t_last_set[knob];
  return MSGL_OK;
}

int msgl_set_tuning(int32_t knob, int64_t value) {
  if (knob >= 0 && knob < kTuneKnobs) t_last_set[knob] = value;
  if (knob == MSGL_TUNE_SPLITKV_WAVES) {
    msgl::splitkv_set_max_waves((int)value);
    return MSGL_OK;
  }
  if (knob == MSGL_TUNE_SPLITKV_BOUNDARY) {
    msgl::splitkv_set_boundary((int)value);
    return MSGL_OK;
  }
  if (knob == MSGL_TUNE_GDN_ROWS) {
    msgl::gdn_set_rows((int)value);
    return MSGL_OK;
  }
  if (knob == MSGL_TUNE_PREFILL_VARIANT) {
    msgl::set_tile_variant((int)value);
    return MSGL_OK;
  }
  if (knob == MSGL_TUNE_PREFILL_KEY_SPLITS) {
    t_key_splits = value < 0 ? 0 : value;
    return MSGL_OK;
  }
  if (knob == MSGL_TUNE_PREFILL_GANGS) {
    t_gangs = value;
    return MSGL_OK;
  }
  if (knob == MSGL_TUNE_CLOCK_PROBE) {
    t_clock_probe = reinterpret_cast<long long*>(static_cast<intptr_t>(value));
    return MSGL_OK;
  }
  if (knob == MSGL_TUNE_SHARES) {
    msgl::shares_force(value);
    return MSGL_OK;
  }
  if (knob == MSGL_TUNE_STREAM) {
    msgl::set_stream_kib(value);
    return MSGL_OK;
  }
  if (knob < 0 || knob > 2) return MSGL_ERR_SHAPE;
  t_tune[knob] = value;
  return MSGL_OK;
}

int msgl_store_kv_cache(void* k_cache, void* v_cache, const int32_t* indices, const void* k,
                        const void* v, int64_t length, int64_t num_kv_heads, int64_t head_dim,
                        int64_t num_slots, int64_t k_cache_stride0, int64_t v_cache_stride0,
                        int64_t k_stride0, int64_t v_stride0, int32_t elem_bytes, void* stream) {
  if (length < 0 || num_kv_heads <= 0 || head_dim <= 0 || num_slots < 0) return MSGL_ERR_SHAPE;
  if (elem_bytes != 2 && elem_bytes != 4) return MSGL_ERR_DTYPE;
  if (head_dim % 4 != 0) return MSGL_ERR_HEAD_DIM_MULT4;  // store_kv_cache.cpp:49-52
  const int64_t row = num_kv_heads * head_dim;
  if (k_cache_stride0 < row || v_cache_stride0 < row || k_stride0 < row || v_stride0 < row)
    return MSGL_ERR_SHAPE;
  if (length == 0) return MSGL_OK;
  if (!k_cache || !v_cache || !indices || !k || !v) return MSGL_ERR_NULL_POINTER;
  return msgl::launch_store_kv_cache(k_cache, v_cache, indices, k, v, length, num_slots, row * elem_bytes,
                                     k_cache_stride0 * elem_bytes, v_cache_stride0 * elem_bytes,
                                     k_stride0 * elem_bytes, v_stride0 * elem_bytes,
                                     static_cast<hipStream_t>(stream));
}

size_t msgl_paged_decode_workspace_bytes(int64_t batch, int64_t total_kv, int64_t num_q_heads,
                                         int64_t num_kv_heads, int64_t head_dim) {
  if (batch <= 0 || total_kv < 0 || num_q_heads <= 0 || num_kv_heads <= 0 ||
      num_q_heads % num_kv_heads != 0)
    return 0;
  const int64_t group = num_q_heads / num_kv_heads;
  const msgl::SharePlan plan = shares_for(batch, total_kv, 0, num_kv_heads, head_dim, group);
  if (msgl::shares_preferred(plan, batch, total_kv, num_kv_heads, head_dim, group))
    return msgl::share_workspace_bytes(plan, batch, num_kv_heads, head_dim, group);
  return msgl::splitkv_workspace_bytes(batch, num_q_heads, num_kv_heads, head_dim, 1,
                                       segments(total_kv, num_kv_heads, head_dim, group));
}

// Both decode entry points: `builtin_scratch` takes the workspace from the library's own
// per-device array instead of the caller.
static int decode_attention(const void* q, const void* k_cache, const void* v_cache,
                            const int32_t* kv_indptr, const int32_t* kv_indices,
                            const int32_t* num_kv_splits, void* out, void* workspace,
                            size_t workspace_bytes, bool builtin_scratch, int64_t batch,
                            int64_t total_kv, int64_t num_q_heads, int64_t num_kv_heads,
                            int64_t head_dim, int64_t num_slots, int64_t k_cache_stride0,
                            int64_t v_cache_stride0, float sm_scale, int32_t max_kv_splits,
                            int32_t dtype, void* stream) {
  const msgl::NewTokens tokens{};  // every row is in the pool
  if (batch < 0 || total_kv < 0 || num_slots < 0) return MSGL_ERR_SHAPE;
  if (batch == 0) return MSGL_OK;
  int rc = check_common(q, k_cache, v_cache, out, num_q_heads, num_kv_heads, head_dim,
                        k_cache_stride0, v_cache_stride0, dtype, /*f16_ok=*/true);
  if (rc != MSGL_OK) return rc;
  const int64_t group = num_q_heads / num_kv_heads;
  if (group > 16) return MSGL_ERR_GROUP_TOO_LARGE;  // paged_decode_attention.cpp:54-57
  if (!kv_indptr || !num_kv_splits || (total_kv > 0 && !kv_indices)) return MSGL_ERR_NULL_POINTER;
  (void)max_kv_splits;  // split hints do not steer the cut (result is split-invariant)
  const int32_t n_seg = segments(total_kv, num_kv_heads, head_dim, group);
  const msgl::SharePlan plan = shares_for(batch, total_kv, 0, num_kv_heads, head_dim, group);
  const bool shares = msgl::shares_preferred(plan, batch, total_kv, num_kv_heads, head_dim, group);
  const size_t need = shares
                          ? msgl::share_workspace_bytes(plan, batch, num_kv_heads, head_dim, group)
                          : msgl::splitkv_workspace_bytes(batch, num_q_heads, num_kv_heads, head_dim, 1, n_seg);
  if (builtin_scratch) {
    rc = msgl::splitkv_scratch(&workspace, &workspace_bytes);
    if (rc != MSGL_OK) return rc;
    if (need > workspace_bytes) return MSGL_ERR_SCRATCH_LIMIT;
  }
  if (!workspace || workspace_bytes < need || !aligned16(workspace)) return MSGL_ERR_WORKSPACE;
  msgl::SplitKvArgs a{};
  a.q = q;
  a.k_cache = k_cache;
  a.v_cache = v_cache;
  a.kv_indptr = kv_indptr;
  a.kv_indices = kv_indices;
  a.qo_indptr = nullptr;
  a.prefix_lens = nullptr;
  a.out = out;
  a.workspace = workspace;
  a.batch = batch;
  a.total_kv = total_kv;
  a.n_q = num_q_heads;
  a.n_kv = num_kv_heads;
  a.head_dim = head_dim;
  a.num_slots = num_slots;
  a.k_stride0 = k_cache_stride0;
  a.v_stride0 = v_cache_stride0;
  a.sm_scale = sm_scale;
  a.max_len_extend = 1;
  a.f16 = (dtype == MSGL_DTYPE_F16) ? 1 : 0;
  a.is_cross = 0;
  a.window = 0;
  a.n_seg = n_seg;
  a.min_seg = min_segment(head_dim);
  if (shares) return msgl::launch_shares(a, tokens, plan, static_cast<hipStream_t>(stream));
  return msgl::launch_splitkv(a, tokens, static_cast<hipStream_t>(stream));
}

int msgl_paged_decode_attention(const void* q, const void* k_cache, const void* v_cache,
                                const int32_t* kv_indptr, const int32_t* kv_indices,
                                const int32_t* num_kv_splits, void* out, void* workspace,
                                size_t workspace_bytes, int64_t batch, int64_t total_kv,
                                int64_t num_q_heads, int64_t num_kv_heads, int64_t head_dim,
                                int64_t num_slots, int64_t k_cache_stride0,
                                int64_t v_cache_stride0, float sm_scale, int32_t max_kv_splits,
                                int32_t dtype, void* stream) {
  return decode_attention(q, k_cache, v_cache, kv_indptr, kv_indices, num_kv_splits, out, workspace,
                          workspace_bytes, false, batch, total_kv, num_q_heads, num_kv_heads,
                          head_dim, num_slots, k_cache_stride0, v_cache_stride0, sm_scale,
                          max_kv_splits, dtype, stream);
}

int msgl_paged_decode_attention_noalloc(const void* q, const void* k_cache, const void* v_cache,
                                        const int32_t* kv_indptr, const int32_t* kv_indices,
                                        const int32_t* num_kv_splits, void* out, int64_t batch,
                                        int64_t total_kv, int64_t num_q_heads,
                                        int64_t num_kv_heads, int64_t head_dim, int64_t num_slots,
                                        int64_t k_cache_stride0, int64_t v_cache_stride0,
                                        float sm_scale, int32_t max_kv_splits, int32_t dtype,
                                        void* stream) {
  return decode_attention(q, k_cache, v_cache, kv_indptr, kv_indices, num_kv_splits, out, nullptr,
                          0, true, batch, total_kv, num_q_heads, num_kv_heads, head_dim, num_slots,
                          k_cache_stride0, v_cache_stride0, sm_scale, max_kv_splits, dtype, stream);
}

// The workspace of a decode step in one launch, 0: it is not the way; `plan`: of its shares, share_len 0 where it goes in segments.
static size_t decode_step_route(int64_t batch, int64_t total_kv, int64_t num_q_heads, int64_t num_kv_heads, int64_t head_dim,
                                bool norm_rope, msgl::SharePlan* plan) {
  if (batch <= 0 || total_kv < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || num_q_heads % num_kv_heads != 0 ||
      num_q_heads / num_kv_heads > 16 || (head_dim != 128 && head_dim != 256))
    return 0;
  const int64_t group = num_q_heads / num_kv_heads;
  *plan = shares_for(batch, total_kv, 0, num_kv_heads, head_dim, group);
  if (!msgl::shares_preferred(*plan, batch, total_kv, num_kv_heads, head_dim, group)) {
    // norm and rotary embedding would be made anew by every segment of a request: 3.5 us of a launch of their own is
    // less on the launches that go in segments.  On large ones the store's launch hides behind the start of the next,
    // and its part of the segments is paid by the slowest of them; us (all read through the caches), store in front against inside, by MiB of keys and
    // values: 22 23.3 and 20.9 (2 requests, 24 / 4 heads of 256), 113 24.2 and 22.4 (1), 183 38.2 and 37.0 (68); 281
    // 53.5 and 53.6 (16 requests), 366 81.2 and 83.4 (128), 625 126.8 and 127.8 (64); at head_dim 256 312 65.3 and 63.5 (16)
    if (norm_rope || (total_kv * num_kv_heads * head_dim * 4 >> 20) > (head_dim == 256 ? 384 : 192)) return 0;
    plan->share_len = 0;
    return msgl::splitkv_workspace_bytes(batch, num_q_heads, num_kv_heads, head_dim, 1, segments(total_kv, num_kv_heads, head_dim, group));
  }
  return msgl::share_workspace_bytes(*plan, batch, num_kv_heads, head_dim, group);
}

size_t msgl_decode_step_workspace_bytes(int64_t batch, int64_t total_kv, int64_t num_q_heads, int64_t num_kv_heads,
                                        int64_t head_dim, int32_t norm_rope) {
  msgl::SharePlan plan{};
  return decode_step_route(batch, total_kv, num_q_heads, num_kv_heads, head_dim, norm_rope != 0, &plan);
}

int msgl_decode_step(const void* q, const void* k, const void* v, int64_t q_stride0, int64_t k_stride0, int64_t v_stride0,
                     const void* q_weight, const void* k_weight, const int32_t* positions, const int32_t* out_loc,
                     void* k_cache, void* v_cache, const int32_t* kv_indptr, const int32_t* kv_indices, void* out,
                     void* workspace, size_t workspace_bytes, int64_t batch, int64_t total_kv, int64_t num_q_heads,
                     int64_t num_kv_heads, int64_t head_dim, int64_t num_slots, int64_t k_cache_stride0,
                     int64_t v_cache_stride0, float sm_scale, float rms_norm_eps, float rope_base, int32_t dtype,
                     void* stream) {
  if (batch < 0 || total_kv < 0 || num_slots <= 0) return MSGL_ERR_SHAPE;
  if (batch == 0) return MSGL_OK;
  const int rc = check_common(q, k_cache, v_cache, out, num_q_heads, num_kv_heads, head_dim, k_cache_stride0,
                              v_cache_stride0, dtype, /*f16_ok=*/q_weight == nullptr);
  if (rc != MSGL_OK) return rc;
  const int64_t group = num_q_heads / num_kv_heads;
  if (group > 16) return MSGL_ERR_GROUP_TOO_LARGE;
  if (!k || !v || !out_loc || !kv_indptr || (total_kv > 0 && !kv_indices)) return MSGL_ERR_NULL_POINTER;
  if ((q_weight == nullptr) != (k_weight == nullptr) || (q_weight && !positions)) return MSGL_ERR_NULL_POINTER;
  if (q_stride0 < num_q_heads * head_dim || k_stride0 < num_kv_heads * head_dim || v_stride0 < num_kv_heads * head_dim)
    return MSGL_ERR_SHAPE;
  if (q_weight && (!(rope_base > 1.0f) || !(rms_norm_eps >= 0.0f))) return MSGL_ERR_SHAPE;
  if (!aligned16(k) || !aligned16(v) || q_stride0 % 8 || k_stride0 % 8 || v_stride0 % 8 || !aligned16(q_weight) ||
      !aligned16(k_weight))
    return MSGL_ERR_ALIGNMENT;
  msgl::SharePlan plan{};
  const size_t need = decode_step_route(batch, total_kv, num_q_heads, num_kv_heads, head_dim, q_weight != nullptr, &plan);
  if (need == 0) return MSGL_ERR_SHAPE;
  if (!workspace || workspace_bytes < need || !aligned16(workspace)) return MSGL_ERR_WORKSPACE;
  msgl::SplitKvArgs a{};
  a.q = q;
  a.k_cache = k_cache;
  a.v_cache = v_cache;
  a.kv_indptr = kv_indptr;
  a.kv_indices = kv_indices;
  a.out = out;
  a.workspace = workspace;
  a.batch = batch;
  a.total_kv = total_kv;
  a.n_q = num_q_heads;
  a.n_kv = num_kv_heads;
  a.head_dim = head_dim;
  a.num_slots = num_slots;
  a.k_stride0 = k_cache_stride0;
  a.v_stride0 = v_cache_stride0;
  a.q_stride0 = q_stride0;
  a.sm_scale = sm_scale;
  a.max_len_extend = 1;
  a.f16 = (dtype == MSGL_DTYPE_F16) ? 1 : 0;
  msgl::NewTokens tokens{};
  tokens.k = k;
  tokens.v = v;
  tokens.q_weight = q_weight;
  tokens.k_weight = k_weight;
  tokens.positions = positions;
  tokens.out_loc = out_loc;
  tokens.k_stride0 = k_stride0;
  tokens.v_stride0 = v_stride0;
  tokens.rows = batch;
  tokens.eps = rms_norm_eps;
  tokens.rope_base = rope_base;
  if (plan.share_len > 0) return msgl::launch_shares(a, tokens, plan, static_cast<hipStream_t>(stream));
  a.n_seg = segments(total_kv, num_kv_heads, head_dim, group);
  a.min_seg = min_segment(head_dim);
  return msgl::launch_splitkv(a, tokens, static_cast<hipStream_t>(stream));
}

// Ragged key shares for the tile kernels (one query block per (request, kv head)): the ping-pong
// kernel and the head_dim 256 kernel know them, the fused head_dim 128 kernels do not.
static int ragged_tiles(int64_t batch, int64_t total_kv, int64_t n_kv, int64_t group,
                        int64_t max_len_extend, int64_t head_dim) {
  if (head_dim == 128 && msgl::tile_variant() != 0) return 0;
  return msgl::prefill_ragged_tiles(batch, total_kv, n_kv, group, max_len_extend,
                                    msgl::prefill_block_rows(head_dim), t_key_splits);
}

// Gang ranges for the head_dim 128 ping-pong kernel (several query blocks per (request, kv head)).
static int gangs_for(int64_t batch, int64_t total_q, int64_t total_kv, int64_t n_kv, int64_t group, int64_t max_len_extend,
                     int64_t head_dim, int64_t window, int key_splits) {
  if (head_dim != 128 || msgl::tile_variant() != 0 || t_gangs < 0) return 0;
  return msgl::prefill_gangs(batch, total_q, total_kv, n_kv, group, max_len_extend, window, msgl::kPrefillBlockRows,
                             t_gangs > 0 ? 1 : key_splits, t_key_splits, /*whatever_the_size=*/t_gangs > 0);
}

static bool use_splitkv_route(int64_t group, int64_t max_len_extend, int64_t head_dim, int64_t batch,
                              int64_t total_kv, int64_t n_kv) {
  const int64_t cols = group * max_len_extend;
  if (max_len_extend < 1 || cols > msgl::kSplitKvMaxCols) return false;
  const int64_t t = t_tune[MSGL_TUNE_SMALLQ_MAXCOLS];
  if (t != 0) return t > 0 && cols <= t;  // set by hand; negative: never
  if (cols <= smallq_base_cols(head_dim) || two_tiles_in_segments(total_kv, n_kv, head_dim, cols)) return true;
  return ragged_tiles(batch, total_kv, n_kv, group, max_len_extend, head_dim) == 0;
}
// Under a sliding window that most requests exceed (mean kv length at least twice the window),
// every request shows about `window` keys, the one case where one workgroup per (request, kv
// head) is balanced: the tile kernel then streams 5-20 % faster than the split-K kernel from
// 17 columns on (shape 5 with a window of 1024: 32 against 36 us).  Only the default routing
// does this; MSGL_TUNE_SMALLQ_MAXCOLS set by hand is obeyed as it stands.
static bool window_prefers_tiles(int64_t batch, int64_t total_kv, int64_t n_kv, int64_t group,
                                 int64_t max_len_extend, int64_t head_dim, int64_t window) {
  if (window <= 0 || t_tune[MSGL_TUNE_SMALLQ_MAXCOLS] != 0) return false;
  if (group * max_len_extend <= 16) return false;
  if (head_dim == 256)  // what two_tiles_in_segments() took for its size is less under the window
    return two_tiles_in_segments(total_kv, n_kv, head_dim, group * max_len_extend) &&
           !two_tiles_in_segments(msgl::visible_keys(batch, total_kv, window, max_len_extend, false), n_kv, head_dim, group * max_len_extend) &&
           ragged_tiles(batch, total_kv, n_kv, group, max_len_extend, head_dim) > 0;
  if (total_kv < 2 * batch * (window + max_len_extend)) return false;
  return ragged_tiles(batch, total_kv, n_kv, group, max_len_extend, head_dim) > 0;
}

// Whether a prefill call goes in shares, given room for their partials: `window_share` for its window's sake, else where
// it is a short query block's call and small.
static bool shares_route(const msgl::SharePlan& plan, bool window_share, int64_t batch, int64_t total_kv, int64_t keys,
                         int64_t n_kv, int64_t group, int64_t max_len_extend, int64_t head_dim, int64_t window) {
  if (plan.share_len == 0) return false;
  if (plan.col_groups > 1) return msgl::shares_preferred(plan, batch, keys, n_kv, head_dim, group * max_len_extend);
  if (window_share) return true;
  if (keys < total_kv && msgl::few_pairs_in_segments(batch, n_kv, keys / batch, head_dim, group * max_len_extend, true)) return false;
  return use_splitkv_route(group, max_len_extend, head_dim, batch, total_kv, n_kv) &&
         !window_prefers_tiles(batch, total_kv, n_kv, group, max_len_extend, head_dim, window) &&
         msgl::shares_preferred(plan, batch, keys, n_kv, head_dim, group * max_len_extend);
}

size_t msgl_paged_prefill_workspace_bytes(int64_t batch, int64_t total_q, int64_t total_kv,
                                          int64_t num_q_heads, int64_t num_kv_heads,
                                          int64_t head_dim, int64_t max_len_extend) {
  if (batch <= 0 || total_q < 0 || total_kv < 0 || num_q_heads <= 0 || num_kv_heads <= 0 ||
      num_q_heads % num_kv_heads != 0)
    return 0;
  const int64_t group = num_q_heads / num_kv_heads;
  const int64_t cols = group * max_len_extend;
  // a window, unknown here, may make the launch one for shares
  size_t share_need = 0;
  if (const msgl::SharePlan plan = shares_for(batch, total_kv, 0, num_kv_heads, head_dim, cols); plan.share_len > 0)
    share_need = msgl::share_workspace_bytes(msgl::with_any_window(plan, batch, num_kv_heads), batch, num_kv_heads, head_dim, cols);
  if (!use_splitkv_route(group, max_len_extend, head_dim, batch, total_kv, num_kv_heads)) {
    // tile kernels: partials of a key split, if this launch would use one (a sliding window,
    // unknown here, can only lower the count)
    const int ragged = ragged_tiles(batch, total_kv, num_kv_heads, group, max_len_extend, head_dim);
    if (ragged > 0)
      return std::max(share_need, msgl::prefill_ragged_workspace_bytes(batch, total_kv, num_kv_heads, group,
                                                                       max_len_extend, head_dim, ragged));
    const int k = msgl::prefill_key_splits(batch, total_q, total_kv, num_kv_heads, group, max_len_extend, 0, head_dim,
                                           t_key_splits);
    // (the slots of gang ranges are the same however many queries there are)
    const int gangs = gangs_for(batch, batch * max_len_extend, total_kv, num_kv_heads, group, max_len_extend, head_dim, 0, k);
    const size_t split_need = std::max(share_need, msgl::prefill_split_workspace_bytes(total_q, num_q_heads, head_dim, k));
    if (gangs > 0)
      return std::max(split_need, msgl::prefill_gang_workspace_bytes(batch, num_kv_heads, group, max_len_extend, gangs));
    return split_need;
  }
  const size_t split_need =
      std::max(share_need, msgl::splitkv_workspace_bytes(batch, num_q_heads, num_kv_heads, head_dim, max_len_extend,
                                                         segments(total_kv, num_kv_heads, head_dim, cols)));
  // a sliding window (unknown here) may send the launch to the tile kernel instead
  const int ragged = ragged_tiles(batch, total_kv, num_kv_heads, group, max_len_extend, head_dim);
  const size_t tile_need = ragged > 0 ? msgl::prefill_ragged_workspace_bytes(batch, total_kv, num_kv_heads, group,
                                                                             max_len_extend, head_dim, ragged)
                                      : 0;
  return std::max(split_need, tile_need);
}

static bool stores_in_tiles(int64_t batch, int64_t total_q, int64_t total_kv, int64_t n_q, int64_t n_kv, int64_t head_dim,
                            int64_t max_len_extend, bool is_cross, int64_t window);

// Whether prompts with nothing cached go through the tile kernel whose workgroups stay, which takes their keys and values from
// the new rows and stores those on the way (see kMinFreshRounds): as many keys as rows, in one pass over them, from one round of blocks on.
// Not those whose only round stores_in_tiles() has (us, there and here: 8 of 126 tokens, 64 / 8 heads, 16.0 and 18.4, 16 of 64 15.0 and 18.6,
// 16 of 127, 32 / 4, 16.3 and 18.1, 16 of 126, 32 / 8, 17.3 and 18.8).
// The rows have to be most of a round themselves: many short requests leave their blocks nearly empty and have little to store.
// 338 launches of causal prompts, this against two launches by the rounds that their rows fill, geometric mean and worst: up
// to 0.6 1.018 and 1.084, 0.6-0.8 0.976 and 1.159, 0.8-1 0.951 and 1.095 (1.027 from 0.875 on), 1-2 0.925 and 1.058, above 0.965 and 1.053.
// Where a row sees all keys, a block's own tokens are not in its last tile and come from memory a second time: groups above
// 4, whose blocks have less than half a tile of them, lose 3 % from two rounds on and gain 2 % (0.84-1.11) below.
static bool prompts_stored(int64_t batch, int64_t total_q, int64_t total_kv, int64_t n_q, int64_t n_kv, int64_t head_dim,
                           int64_t max_len_extend, bool is_cross, int64_t window) {
  if (batch <= 0 || total_q <= 0 || total_kv != total_q || total_q > msgl::kMaxFreshRows || n_q <= 0 || n_kv <= 0 || n_q % n_kv != 0 || max_len_extend <= 0 ||
      window < 0 || head_dim != 128 || msgl::tile_variant() != 0 || t_gangs > 0 ||
      stores_in_tiles(batch, total_q, total_kv, n_q, n_kv, head_dim, max_len_extend, is_cross, window))
    return false;
  const int64_t group = n_q / n_kv;
  if ((is_cross && group > 4) || 8 * total_q * n_q < 7 * (int64_t)msgl::kComputeUnits * msgl::kPrefillBlockRows) return false;
  if (use_splitkv_route(group, max_len_extend, head_dim, batch, total_kv, n_kv) ||
      ragged_tiles(batch, total_kv, n_kv, group, max_len_extend, head_dim) > 0)
    return false;
  const int splits = msgl::prefill_key_splits(batch, total_q, total_kv, n_kv, group, max_len_extend, window, head_dim, t_key_splits);
  if (splits > 1 || gangs_for(batch, total_q, total_kv, n_kv, group, max_len_extend, head_dim, window, splits) > 0) return false;
  msgl::PrefillArgs a{};
  a.batch = batch;
  a.total_q = total_q;
  a.total_kv = total_kv;
  a.n_kv = n_kv;
  a.max_len_extend = (int32_t)max_len_extend;
  a.is_cross = is_cross ? 1 : 0;
  a.by_length = 1;
  const int64_t n_qblk = (max_len_extend * group + msgl::kPrefillBlockRows - 1) / msgl::kPrefillBlockRows;
  return msgl::prefill_by_length(a, n_qblk, true) && msgl::prefill_stay_rounds(batch, total_q, n_kv, group, n_qblk, msgl::kPrefillBlockRows,
                                   2 * msgl::kMinFreshRounds) > 0;
}

// `tokens`: rows that the launch stores itself, where stores_in_tiles() or prompts_stored() holds; out_loc nullptr: none.
static int prefill_attention(const void* q, const void* k_cache, const void* v_cache,
                                 const int32_t* qo_indptr, const int32_t* kv_indptr,
                                 const int32_t* kv_indices, const int32_t* prefix_lens, void* out,
                                 void* workspace, size_t workspace_bytes, int64_t batch,
                                 int64_t total_q, int64_t total_kv, int64_t num_q_heads,
                                 int64_t num_kv_heads, int64_t head_dim, int64_t num_slots,
                                 int64_t k_cache_stride0, int64_t v_cache_stride0, float sm_scale,
                                 int32_t max_len_extend, int32_t is_cross_attention,
                                 int32_t sliding_window_size, int32_t dtype, const msgl::NewTokens& tokens, void* stream) {
  if (head_dim != 128 && head_dim != 256) return MSGL_ERR_HEAD_DIM;
  if (num_q_heads <= 0 || num_kv_heads <= 0) return MSGL_ERR_SHAPE;
  if (num_q_heads % num_kv_heads != 0) return MSGL_ERR_HEAD_RATIO;
  if (sliding_window_size < 0) return MSGL_ERR_WINDOW;  // paged_prefill_attention.cpp:67-70
  if (batch <= 0) return MSGL_ERR_BATCH;                // :74-77
  if (total_q < 0 || total_kv < 0 || num_slots < 0) return MSGL_ERR_SHAPE;
  if (total_q == 0 || max_len_extend <= 0) return MSGL_OK;
  int rc = check_common(q, k_cache, v_cache, out, num_q_heads, num_kv_heads, head_dim,
                        k_cache_stride0, v_cache_stride0, dtype, /*f16_ok=*/false);
  if (rc != MSGL_OK) return rc;
  if (!qo_indptr || !kv_indptr || !prefix_lens || (total_kv > 0 && !kv_indices))
    return MSGL_ERR_NULL_POINTER;
  const int64_t group = num_q_heads / num_kv_heads;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t cols = group * max_len_extend;
  const int64_t keys = msgl::visible_keys(batch, total_kv, sliding_window_size, max_len_extend, is_cross_attention != 0);
  const msgl::SharePlan plan = shares_for(batch, keys, keys < total_kv ? keys / batch : 0, num_kv_heads, head_dim, cols);
  // without room for their partials a launch goes the way it goes without shares
  const bool share_room = plan.share_len > 0 && workspace && aligned16(workspace) &&
                          workspace_bytes >= msgl::share_workspace_bytes(plan, batch, num_kv_heads, head_dim, cols);
  const bool window_share = share_room && window_shares(plan, batch, total_kv, keys, num_kv_heads, head_dim, cols);
  const bool shares = share_room && shares_route(plan, window_share, batch, total_kv, keys, num_kv_heads, group, max_len_extend,
                                                 head_dim, sliding_window_size);
  bool direct = shares || (use_splitkv_route(group, max_len_extend, head_dim, batch, total_kv, num_kv_heads) &&
                           !window_prefers_tiles(batch, total_kv, num_kv_heads, group, max_len_extend, head_dim,
                                                 sliding_window_size));
  const int32_t n_seg = direct ? segments(total_kv, num_kv_heads, head_dim, cols) : 0;
  if (direct && !shares) {
    const size_t need = msgl::splitkv_workspace_bytes(batch, num_q_heads, num_kv_heads, head_dim, max_len_extend, n_seg);
    const bool room = workspace && workspace_bytes >= need && aligned16(workspace);
    // the tile kernel, which does without, where only the size asks for segments
    if (!room && (t_tune[MSGL_TUNE_SMALLQ_MAXCOLS] != 0 || !two_tiles_in_segments(total_kv, num_kv_heads, head_dim, cols) ||
                  ragged_tiles(batch, total_kv, num_kv_heads, group, max_len_extend, head_dim) == 0))
      return MSGL_ERR_WORKSPACE;
    direct = room;
  }
  if (direct) {
    msgl::SplitKvArgs a{};
    a.q = q;
    a.k_cache = k_cache;
    a.v_cache = v_cache;
    a.kv_indptr = kv_indptr;
    a.kv_indices = kv_indices;
    a.qo_indptr = qo_indptr;
    a.prefix_lens = prefix_lens;
    a.out = out;
    a.workspace = workspace;
    a.batch = batch;
    a.total_kv = total_kv;
    a.n_q = num_q_heads;
    a.n_kv = num_kv_heads;
    a.head_dim = head_dim;
    a.num_slots = num_slots;
    a.k_stride0 = k_cache_stride0;
    a.v_stride0 = v_cache_stride0;
    a.sm_scale = sm_scale;
    a.max_len_extend = max_len_extend;
    a.q_cap = max_len_extend;
    a.is_cross = is_cross_attention ? 1 : 0;
    a.window = sliding_window_size;
    a.n_seg = n_seg;
    a.min_seg = min_segment(head_dim);
    a.q_begin = 0;
    if (shares) return msgl::launch_shares(a, msgl::NewTokens{}, plan, s);
    return msgl::launch_splitkv(a, msgl::NewTokens{}, s);
  }
  msgl::PrefillArgs a{};
  a.q = q;
  a.k_cache = k_cache;
  a.v_cache = v_cache;
  a.qo_indptr = qo_indptr;
  a.kv_indptr = kv_indptr;
  a.kv_indices = kv_indices;
  a.prefix_lens = prefix_lens;
  a.out = out;
  a.batch = batch;
  a.total_q = total_q;
  a.total_kv = total_kv;
  a.n_q = num_q_heads;
  a.n_kv = num_kv_heads;
  a.head_dim = head_dim;
  a.num_slots = num_slots;
  a.k_stride0 = k_cache_stride0;
  a.v_stride0 = v_cache_stride0;
  a.sm_scale = sm_scale;
  a.max_len_extend = max_len_extend;
  a.is_cross = is_cross_attention ? 1 : 0;
  a.window = sliding_window_size;
  a.key_splits = 1;
  a.new_tokens = tokens;  // stored by the tile kernels alone (see stores_in_tiles())
  a.by_length = tokens.out_loc == nullptr || prompts_stored(batch, total_q, total_kv, num_q_heads, num_kv_heads, head_dim,
                                                            max_len_extend, is_cross_attention != 0, sliding_window_size);
  a.ragged_tiles = ragged_tiles(batch, total_kv, num_kv_heads, group, max_len_extend, head_dim);
  if (a.ragged_tiles > 0) {
    // ragged shares need room for their partials; without it the keys go in one pass
    const size_t need = msgl::prefill_ragged_workspace_bytes(batch, total_kv, num_kv_heads, group,
                                                             max_len_extend, head_dim, a.ragged_tiles);
    if (need > 0 && (!workspace || workspace_bytes < need || !aligned16(workspace))) a.ragged_tiles = 0;
    else a.workspace = workspace;
  } else {
    a.key_splits = msgl::prefill_key_splits(batch, total_q, total_kv, num_kv_heads, group, max_len_extend,
                                            sliding_window_size, head_dim, t_key_splits);
  }
  if (a.key_splits > 1) {
    // the split is an optimisation: without room for its partials the keys go in one pass
    const size_t need = msgl::prefill_split_workspace_bytes(total_q, num_q_heads, head_dim, a.key_splits);
    if (!workspace || workspace_bytes < need || !aligned16(workspace)) a.key_splits = 1;
    else a.workspace = workspace;
  }
  a.gangs = 0;
  if (t_gangs > 0 && a.ragged_tiles == 0) a.key_splits = 1;  // forced for a test: gang ranges instead
  if (a.ragged_tiles == 0 && a.key_splits == 1 && tokens.out_loc == nullptr) {
    const int gangs = gangs_for(batch, total_q, total_kv, num_kv_heads, group, max_len_extend, head_dim,
                                sliding_window_size, a.key_splits);
    // so are gang ranges: without room for their slots every unit goes to one workgroup per query block
    if (gangs > 0 && workspace && aligned16(workspace) &&
        workspace_bytes >= msgl::prefill_gang_workspace_bytes(batch, num_kv_heads, group, max_len_extend, gangs)) {
      a.gangs = gangs;
      a.workspace = workspace;
      a.gang_nonce = msgl::next_launch_number();
    }
  }
  return head_dim == 256 ? msgl::launch_prefill_tile256(a, s) : msgl::launch_prefill_tile(a, s);
}

int msgl_paged_prefill_attention(const void* q, const void* k_cache, const void* v_cache,
                                 const int32_t* qo_indptr, const int32_t* kv_indptr,
                                 const int32_t* kv_indices, const int32_t* prefix_lens, void* out,
                                 void* workspace, size_t workspace_bytes, int64_t batch,
                                 int64_t total_q, int64_t total_kv, int64_t num_q_heads,
                                 int64_t num_kv_heads, int64_t head_dim, int64_t num_slots,
                                 int64_t k_cache_stride0, int64_t v_cache_stride0, float sm_scale,
                                 int32_t max_len_extend, int32_t is_cross_attention,
                                 int32_t sliding_window_size, int32_t dtype, void* stream) {
  return prefill_attention(q, k_cache, v_cache, qo_indptr, kv_indptr, kv_indices, prefix_lens, out, workspace, workspace_bytes,
                           batch, total_q, total_kv, num_q_heads, num_kv_heads, head_dim, num_slots, k_cache_stride0,
                           v_cache_stride0, sm_scale, max_len_extend, is_cross_attention, sliding_window_size, dtype,
                           msgl::NewTokens{}, stream);
}

// The plan of a prefill call whose store goes into its attention launch; share_len == 0: none
static msgl::SharePlan extend_step_plan(int64_t batch, int64_t total_q, int64_t total_kv, int64_t n_q, int64_t n_kv,
                                        int64_t head_dim, int64_t max_len_extend, bool is_cross, int64_t window) {
  const msgl::SharePlan none{};
  if (batch <= 0 || total_q <= 0 || total_kv <= 0 || n_q <= 0 || n_kv <= 0 || n_q % n_kv != 0 || max_len_extend <= 0 ||
      window < 0 || (head_dim != 128 && head_dim != 256))
    return none;
  const int64_t group = n_q / n_kv, cols = group * max_len_extend;
  const int64_t keys = msgl::visible_keys(batch, total_kv, window, max_len_extend, is_cross);
  const msgl::SharePlan plan = shares_for(batch, keys, keys < total_kv ? keys / batch : 0, n_kv, head_dim, cols);
  const bool window_share = window_shares(plan, batch, total_kv, keys, n_kv, head_dim, cols);
  return shares_route(plan, window_share, batch, total_kv, keys, n_kv, group, max_len_extend, head_dim, window) ? plan : none;
}

// Whether a tile kernel of such a call stores the rows itself, every workgroup those of its request: in launches of one round,
// of up to kRowsStored tokens a request (half as many at head_dim 256). us: one prompt of 30 tokens 11.8 -> 9.3, nine of 25-86
// 16.8 -> 13.8, 20 of 20-40 on 200-300 23.0 -> 20.4, one of 163 14.3 -> 13.1; beyond the lines the stores in front of every
// workgroup outweigh the launch: one of 250 on 2000 33.6 -> 35.0, of 250 on 1000 at 24 / 4 heads of 256 33.3 -> 36.8.
constexpr int64_t kRowsStored = 192, kBytesStored = 16 << 20;
static bool stores_in_tiles(int64_t batch, int64_t total_q, int64_t total_kv, int64_t n_q, int64_t n_kv, int64_t head_dim,
                            int64_t max_len_extend, bool is_cross, int64_t window) {
  if (batch <= 0 || total_q <= 0 || total_kv <= 0 || n_q <= 0 || n_kv <= 0 || n_q % n_kv != 0 || max_len_extend <= 0 ||
      window < 0 || (head_dim != 128 && head_dim != 256) || max_len_extend * head_dim > kRowsStored * 128 || msgl::tile_variant() != 0 || t_gangs > 0)
    return false;
  const int64_t group = n_q / n_kv;
  if (use_splitkv_route(group, max_len_extend, head_dim, batch, total_kv, n_kv) &&
      !window_prefers_tiles(batch, total_kv, n_kv, group, max_len_extend, head_dim, window))
    return false;
  const int ragged = ragged_tiles(batch, total_kv, n_kv, group, max_len_extend, head_dim);
  if (ragged > 0) return msgl::prefill_ragged_units(batch, total_kv, ragged) * n_kv <= 2 * msgl::device_cus();
  const int splits = msgl::prefill_key_splits(batch, total_q, total_kv, n_kv, group, max_len_extend, window, head_dim, t_key_splits);
  const int64_t rows = msgl::prefill_block_rows(head_dim);
  const int64_t blocks = batch * n_kv * splits * ((max_len_extend * group + rows - 1) / rows);
  return blocks <= msgl::device_cus() && blocks * max_len_extend * head_dim * 4 <= kBytesStored;
}

size_t msgl_extend_step_workspace_bytes(int64_t batch, int64_t total_q, int64_t total_kv, int64_t num_q_heads,
                                        int64_t num_kv_heads, int64_t head_dim, int64_t max_len_extend,
                                        int32_t is_cross_attention, int32_t sliding_window_size) {
  const msgl::SharePlan plan = extend_step_plan(batch, total_q, total_kv, num_q_heads, num_kv_heads, head_dim, max_len_extend,
                                                is_cross_attention != 0, sliding_window_size);
  if (plan.share_len > 0)
    return msgl::share_workspace_bytes(plan, batch, num_kv_heads, head_dim, num_q_heads / num_kv_heads * max_len_extend);
  if (!stores_in_tiles(batch, total_q, total_kv, num_q_heads, num_kv_heads, head_dim, max_len_extend, is_cross_attention != 0,
                       sliding_window_size) &&
      !prompts_stored(batch, total_q, total_kv, num_q_heads, num_kv_heads, head_dim, max_len_extend, is_cross_attention != 0,
                      sliding_window_size))
    return 0;
  return std::max<size_t>(16, msgl_paged_prefill_workspace_bytes(batch, total_q, total_kv, num_q_heads, num_kv_heads, head_dim,
                                                                 max_len_extend));
}

int msgl_extend_step(const void* q, const void* k, const void* v, int64_t k_stride0, int64_t v_stride0, const int32_t* out_loc,
                     void* k_cache, void* v_cache, const int32_t* qo_indptr, const int32_t* kv_indptr,
                     const int32_t* kv_indices, const int32_t* prefix_lens, void* out, void* workspace,
                     size_t workspace_bytes, int64_t batch, int64_t total_q, int64_t total_kv, int64_t num_q_heads,
                     int64_t num_kv_heads, int64_t head_dim, int64_t num_slots, int64_t k_cache_stride0,
                     int64_t v_cache_stride0, float sm_scale, int32_t max_len_extend, int32_t is_cross_attention,
                     int32_t sliding_window_size, int32_t dtype, void* stream) {
  if (num_slots <= 0) return MSGL_ERR_SHAPE;
  const int rc = check_common(q, k_cache, v_cache, out, num_q_heads, num_kv_heads, head_dim, k_cache_stride0,
                              v_cache_stride0, dtype, /*f16_ok=*/false);
  if (rc != MSGL_OK) return rc;
  if (!k || !v || !out_loc || !qo_indptr || !kv_indptr || !kv_indices || !prefix_lens) return MSGL_ERR_NULL_POINTER;
  if (k_stride0 < num_kv_heads * head_dim || v_stride0 < num_kv_heads * head_dim) return MSGL_ERR_SHAPE;
  if (!aligned16(k) || !aligned16(v) || k_stride0 % 8 || v_stride0 % 8) return MSGL_ERR_ALIGNMENT;
  const msgl::SharePlan plan = extend_step_plan(batch, total_q, total_kv, num_q_heads, num_kv_heads, head_dim, max_len_extend,
                                                is_cross_attention != 0, sliding_window_size);
  msgl::NewTokens tokens{};
  tokens.k = k;
  tokens.v = v;
  tokens.out_loc = out_loc;
  tokens.k_stride0 = k_stride0;
  tokens.v_stride0 = v_stride0;
  tokens.rows = total_q;
  if (plan.share_len == 0) {
    const size_t need = msgl_extend_step_workspace_bytes(batch, total_q, total_kv, num_q_heads, num_kv_heads, head_dim, max_len_extend,
                                                         is_cross_attention, sliding_window_size);
    if (need == 0) return MSGL_ERR_SHAPE;
    if (!workspace || !aligned16(workspace) || workspace_bytes < need) return MSGL_ERR_WORKSPACE;
    return prefill_attention(q, k_cache, v_cache, qo_indptr, kv_indptr, kv_indices, prefix_lens, out, workspace, workspace_bytes,
                             batch, total_q, total_kv, num_q_heads, num_kv_heads, head_dim, num_slots, k_cache_stride0,
                             v_cache_stride0, sm_scale, max_len_extend, is_cross_attention, sliding_window_size, dtype, tokens, stream);
  }
  const int64_t cols = num_q_heads / num_kv_heads * max_len_extend;
  if (!workspace || !aligned16(workspace) || workspace_bytes < msgl::share_workspace_bytes(plan, batch, num_kv_heads, head_dim, cols))
    return MSGL_ERR_WORKSPACE;
  msgl::SplitKvArgs a{};
  a.q = q;
  a.k_cache = k_cache;
  a.v_cache = v_cache;
  a.kv_indptr = kv_indptr;
  a.kv_indices = kv_indices;
  a.qo_indptr = qo_indptr;
  a.prefix_lens = prefix_lens;
  a.out = out;
  a.workspace = workspace;
  a.batch = batch;
  a.total_kv = total_kv;
  a.n_q = num_q_heads;
  a.n_kv = num_kv_heads;
  a.head_dim = head_dim;
  a.num_slots = num_slots;
  a.k_stride0 = k_cache_stride0;
  a.v_stride0 = v_cache_stride0;
  a.sm_scale = sm_scale;
  a.max_len_extend = max_len_extend;
  a.q_cap = max_len_extend;
  a.is_cross = is_cross_attention ? 1 : 0;
  a.window = sliding_window_size;
  return msgl::launch_shares(a, tokens, plan, static_cast<hipStream_t>(stream));
}

int msgl_copy_state_slots(void* slab, int64_t layer_stride_bytes, int64_t slot_stride_bytes,
                          int64_t row_bytes, int64_t n_layers, int64_t num_slots, const int32_t* src,
                          const int32_t* dst, int64_t n_pairs, void* stream) {
  if (n_layers < 0 || num_slots < 0 || n_pairs < 0 || row_bytes < 0 || slot_stride_bytes < row_bytes ||
      (n_layers > 1 && layer_stride_bytes < num_slots * slot_stride_bytes))
    return MSGL_ERR_SHAPE;
  if (n_layers == 0 || n_pairs == 0 || row_bytes == 0) return MSGL_OK;
  if (!slab || !dst) return MSGL_ERR_NULL_POINTER;
  return msgl::launch_state_slots(slab, layer_stride_bytes, slot_stride_bytes, row_bytes, n_layers,
                                  num_slots, src, dst, n_pairs, static_cast<hipStream_t>(stream));
}

static int build_metadata(bool lens_on_host, const int32_t* page_table, int64_t table_stride0,
                          int64_t n_table_rows, int64_t max_seq_len,
                          const int32_t* table_rows, const int32_t* kv_lens,
                          const int32_t* extend_lens, int64_t batch, int32_t* kv_indptr,
                          int32_t* kv_indices, int64_t kv_capacity, int32_t* qo_indptr,
                          int32_t* prefix_lens, int32_t* positions, int64_t q_capacity,
                          int32_t* num_kv_splits, int32_t max_kv_splits, void* stream) {
  const int64_t max_batch = lens_on_host ? MSGL_METADATA_HOST_BATCH : msgl::kMetadataMaxBatch;
  if (batch < 0 || batch > max_batch || n_table_rows <= 0 || max_seq_len < 0 ||
      table_stride0 < max_seq_len || kv_capacity < 0 || q_capacity < 0 ||
      kv_capacity > 0x7fffffffLL || q_capacity > 0x7fffffffLL || max_seq_len > 0x7fffffffLL ||
      n_table_rows > 0x7fffffffLL)
    return MSGL_ERR_SHAPE;
  if (!kv_indptr) return MSGL_ERR_NULL_POINTER;
  if (batch > 0 && (!page_table || !table_rows || !kv_lens)) return MSGL_ERR_NULL_POINTER;
  if (kv_capacity > 0 && !kv_indices) return MSGL_ERR_NULL_POINTER;
  msgl::MetadataArgs a{};
  a.page_table = page_table;
  a.table_rows = table_rows;
  a.kv_lens = kv_lens;
  a.extend_lens = extend_lens;
  a.kv_indptr = kv_indptr;
  a.kv_indices = kv_indices;
  a.qo_indptr = qo_indptr;
  a.prefix_lens = prefix_lens;
  a.positions = positions;
  a.num_kv_splits = num_kv_splits;
  a.table_stride0 = table_stride0;
  a.batch = batch;
  a.n_table_rows = n_table_rows;
  a.max_seq_len = max_seq_len;
  a.kv_capacity = kv_capacity;
  a.q_capacity = positions ? q_capacity : 0;
  a.max_kv_splits = max_kv_splits;
  a.lens_on_host = lens_on_host ? 1 : 0;
  return msgl::launch_build_metadata(a, static_cast<hipStream_t>(stream));
}

int msgl_build_attention_metadata(const int32_t* page_table, int64_t table_stride0,
                                  int64_t n_table_rows, int64_t max_seq_len, const int32_t* table_rows,
                                  const int32_t* kv_lens, const int32_t* extend_lens, int64_t batch,
                                  int32_t* kv_indptr, int32_t* kv_indices, int64_t kv_capacity, int32_t* qo_indptr,
                                  int32_t* prefix_lens, int32_t* positions, int64_t q_capacity,
                                  int32_t* num_kv_splits, int32_t max_kv_splits, void* stream) {
  return build_metadata(false, page_table, table_stride0, n_table_rows, max_seq_len, table_rows, kv_lens, extend_lens,
                        batch, kv_indptr, kv_indices, kv_capacity, qo_indptr, prefix_lens, positions, q_capacity,
                        num_kv_splits, max_kv_splits, stream);
}

int msgl_build_attention_metadata_host(const int32_t* page_table, int64_t table_stride0,
                                       int64_t n_table_rows, int64_t max_seq_len, const int32_t* table_rows,
                                       const int32_t* kv_lens, const int32_t* extend_lens, int64_t batch,
                                       int32_t* kv_indptr, int32_t* kv_indices, int64_t kv_capacity, int32_t* qo_indptr,
                                       int32_t* prefix_lens, int32_t* positions, int64_t q_capacity,
                                       int32_t* num_kv_splits, int32_t max_kv_splits, void* stream) {
  return build_metadata(true, page_table, table_stride0, n_table_rows, max_seq_len, table_rows, kv_lens, extend_lens,
                        batch, kv_indptr, kv_indices, kv_capacity, qo_indptr, prefix_lens, positions, q_capacity,
                        num_kv_splits, max_kv_splits, stream);
}

int msgl_qk_norm_rope_store(const void* q, const void* k, const void* v, int64_t q_stride0,
                            int64_t k_stride0, int64_t v_stride0, const void* q_weight,
                            const void* k_weight, const int32_t* positions,
                            const int32_t* out_loc, void* q_out, void* k_cache, void* v_cache,
                            int64_t k_cache_stride0, int64_t v_cache_stride0, int64_t num_slots,
                            int64_t n_tokens, int64_t num_q_heads, int64_t num_kv_heads,
                            int64_t head_dim, float rms_norm_eps, float rope_base, int32_t dtype,
                            void* stream) {
  if (head_dim != 128 && head_dim != 256) return MSGL_ERR_HEAD_DIM;
  if (dtype != MSGL_DTYPE_BF16) return MSGL_ERR_DTYPE;
  if (n_tokens < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || num_slots < 0) return MSGL_ERR_SHAPE;
  if (!(rope_base > 1.0f) || !(rms_norm_eps >= 0.0f)) return MSGL_ERR_SHAPE;
  if (q_stride0 < num_q_heads * head_dim || k_stride0 < num_kv_heads * head_dim ||
      v_stride0 < num_kv_heads * head_dim || k_cache_stride0 < num_kv_heads * head_dim ||
      v_cache_stride0 < num_kv_heads * head_dim)
    return MSGL_ERR_SHAPE;
  if (n_tokens == 0) return MSGL_OK;
  if (!q || !k || !v || !q_weight || !k_weight || !positions || !out_loc || !q_out || !k_cache ||
      !v_cache)
    return MSGL_ERR_NULL_POINTER;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(q_weight) ||
      !aligned16(k_weight) || !aligned16(q_out) || !aligned16(k_cache) || !aligned16(v_cache) ||
      q_stride0 % 8 || k_stride0 % 8 || v_stride0 % 8 || k_cache_stride0 % 8 || v_cache_stride0 % 8)
    return MSGL_ERR_ALIGNMENT;
  msgl::NormRopeArgs a{};
  a.q = q;
  a.k = k;
  a.v = v;
  a.q_weight = q_weight;
  a.k_weight = k_weight;
  a.positions = positions;
  a.out_loc = out_loc;
  a.q_out = q_out;
  a.k_cache = k_cache;
  a.v_cache = v_cache;
  a.q_stride0 = q_stride0;
  a.k_stride0 = k_stride0;
  a.v_stride0 = v_stride0;
  a.kc_stride0 = k_cache_stride0;
  a.vc_stride0 = v_cache_stride0;
  a.n_tokens = n_tokens;
  a.num_slots = num_slots;
  a.n_q = num_q_heads;
  a.n_kv = num_kv_heads;
  a.head_dim = head_dim;
  a.eps = rms_norm_eps;
  a.rope_base = rope_base;
  return msgl::launch_qk_norm_rope_store(a, static_cast<hipStream_t>(stream));
}

size_t msgl_gdn_state_workspace_bytes(int64_t tokens, int64_t batch, int64_t hv, int32_t single_token_mode) {
  if (tokens <= 0 || batch <= 0 || hv <= 0) return 0;
  return msgl::gdn_state_workspace_bytes(tokens, batch, hv, single_token_mode != 0);
}

int msgl_gdn_state_inplace_longest(const void* q, const void* k, const void* v, const void* g,
                           const void* beta, void* state, const int32_t* slot_ids,
                           const int32_t* qo_indptr, void* y, int64_t tokens, int64_t batch,
                           int64_t hk, int64_t hv, int64_t dk, int64_t dv, int64_t num_slots,
                           int64_t state_stride0, int64_t q_stride0, int64_t k_stride0,
                           int64_t v_stride0, int32_t single_token_mode, int64_t longest,
                           void* workspace, size_t workspace_bytes, void* stream) {
  if (dk != 128 || dv != 128) return MSGL_ERR_GDN_DIMS;  // gdn_state.cpp:80-83
  if (tokens < 0 || batch < 0 || hk <= 0 || hv <= 0 || num_slots < 0 || longest < 0) return MSGL_ERR_SHAPE;
  if (hv % hk != 0) return MSGL_ERR_HEAD_RATIO;          // gdn_state.cpp:76-79
  if (single_token_mode && tokens != batch) return MSGL_ERR_SHAPE;  // :107-111
  if (state_stride0 < hv * dv * dk || q_stride0 < hk * dk || k_stride0 < hk * dk ||
      v_stride0 < hv * dv)
    return MSGL_ERR_SHAPE;
  if (tokens == 0 || batch == 0) return MSGL_OK;
  if (!q || !k || !v || !g || !beta || !state || !slot_ids || !y) return MSGL_ERR_NULL_POINTER;
  if (!single_token_mode && !qo_indptr) return MSGL_ERR_NULL_POINTER;
  if (!aligned16(q) || !aligned16(k) || !aligned16(state) || q_stride0 % 8 || k_stride0 % 8 ||
      state_stride0 % 4)
    return MSGL_ERR_ALIGNMENT;
  if (workspace && !aligned16(workspace)) return MSGL_ERR_ALIGNMENT;
  msgl::GdnArgs a{};
  a.q = q;
  a.k = k;
  a.v = v;
  a.g = g;
  a.beta = beta;
  a.state = state;
  a.slot_ids = slot_ids;
  a.qo_indptr = qo_indptr;
  a.y = y;
  a.tokens = tokens;
  a.batch = batch;
  a.hk = hk;
  a.hv = hv;
  a.state_stride0 = state_stride0;
  a.q_stride0 = q_stride0;
  a.k_stride0 = k_stride0;
  a.v_stride0 = v_stride0;
  a.single_token_mode = single_token_mode;
  a.longest = longest;
  a.workspace = workspace;
  a.workspace_bytes = workspace_bytes;
  return msgl::launch_gdn_state(a, static_cast<hipStream_t>(stream));
}

int msgl_gdn_state_inplace_in(const void* q, const void* k, const void* v, const void* g,
                           const void* beta, void* state, const int32_t* slot_ids,
                           const int32_t* qo_indptr, void* y, int64_t tokens, int64_t batch,
                           int64_t hk, int64_t hv, int64_t dk, int64_t dv, int64_t num_slots,
                           int64_t state_stride0, int64_t q_stride0, int64_t k_stride0,
                           int64_t v_stride0, int32_t single_token_mode, void* workspace,
                           size_t workspace_bytes, void* stream) {
  return msgl_gdn_state_inplace_longest(q, k, v, g, beta, state, slot_ids, qo_indptr, y, tokens, batch, hk, hv, dk, dv, num_slots,
                                        state_stride0, q_stride0, k_stride0, v_stride0, single_token_mode, 0, workspace,
                                        workspace_bytes, stream);
}

int msgl_gdn_state_inplace(const void* q, const void* k, const void* v, const void* g,
                           const void* beta, void* state, const int32_t* slot_ids,
                           const int32_t* qo_indptr, void* y, int64_t tokens, int64_t batch,
                           int64_t hk, int64_t hv, int64_t dk, int64_t dv, int64_t num_slots,
                           int64_t state_stride0, int64_t q_stride0, int64_t k_stride0,
                           int64_t v_stride0, int32_t single_token_mode, void* stream) {
  return msgl_gdn_state_inplace_in(q, k, v, g, beta, state, slot_ids, qo_indptr, y, tokens, batch, hk, hv, dk, dv, num_slots,
                                   state_stride0, q_stride0, k_stride0, v_stride0, single_token_mode, nullptr, 0, stream);
}

}  // extern "C"
