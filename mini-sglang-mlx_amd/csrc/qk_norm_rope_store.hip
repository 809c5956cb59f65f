// Per-head RMSNorm of q and k, rotary embedding of both, and the KV-store, in one pass.
// Replaces the chain in front of the attention call of the reference's Qwen3 attention layer
// (mini_sglang_mlx/models/qwen3.py:60-68: q_norm, k_norm, rope(q), rope(k), then the store
// inside AttnBackend.forward, attention/backend.py:139), which materialises normalised q and k,
// rotated q and k, and then reads k and v again to scatter them into the pools.
//
//   y   = w * bf16(x * rsqrt(mean(x^2) + eps))                       (per head, fp32 inside)
//   o_i = y_i cos(t_i) - y_{i+d/2} sin(t_i),  o_{i+d/2} = y_i sin(t_i) + y_{i+d/2} cos(t_i)
//   t_i = float(position) * exp2(-(i / (d/2)) * log2(base))          (rotate-half form, rotary_dim = d)
//   q_out[t, h] = o(q[t, h]);  k_cache[out_loc[t], h] = o(k[t, h]);  v_cache[out_loc[t], h] = v[t, h]
//
// HBM-bound: every element of q, k, v is read once and written once
// (2 * (n_q + 2 n_kv) * d * 2 bytes per token, + 8 for position and slot).
// Sixteen lanes own one token's head: lane j holds elements E j .. E j + E - 1 of both halves
// (E = d / 32), so the rotation pairs are lane-local and the mean is a 16-lane xor reduction.
// A group walks a chunk of the token's heads, so sines and cosines (accurate range reduction:
// positions reach 10^5 radians) are computed once per chunk, not once per head.
#include "msgl_device.h"
#include "msgl_internal.h"
#include "norm_rope.h"

namespace msgl {
namespace {

// Heads a group of lanes walks.  Many tokens: 8, so that the sines and cosines are computed once per
// 8 heads (HBM-bound, 21 us for 4096 tokens of 32 + 16 heads, 4.8 TB/s).  Few tokens: 1, because
// then the launch is the chain of one group's loads and not bytes: with 8 heads one after the other
// a decode step of 4 requests (16 + 16 heads) took 11.1 us on a single workgroup.
constexpr int kHeadsPerGroupMany = 8;
constexpr int kGroupLanes = 16;
constexpr int kThreads = 256;

struct NormRopeParams {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const uint16_t* q_weight;
  const uint16_t* k_weight;
  const int32_t* positions;
  const int32_t* out_loc;
  uint16_t* q_out;
  uint16_t* k_cache;
  uint16_t* v_cache;
  int64_t q_stride0, k_stride0, v_stride0, kc_stride0, vc_stride0, num_slots;
  int32_t n_tokens, n_q, n_kv, chunks;  // chunks of heads per token
  float eps, log2_base;
};

template <int D, int kHeadsPerGroup>
__global__ __launch_bounds__(kThreads) void qk_norm_rope_store_kernel(NormRopeParams p) {
  constexpr int E = D / 32;  // elements per lane and half
  using V = typename HalfRow<E>::type;
  const int j = threadIdx.x & (kGroupLanes - 1);
  const int64_t item = (int64_t)blockIdx.x * (kThreads / kGroupLanes) + (threadIdx.x / kGroupLanes);
  if (item >= (int64_t)p.n_tokens * p.chunks) return;  // whole groups leave together
  // few tokens: the item number fits 32 bits (a 64-bit division is 40 instructions of the chain)
  const int t = kHeadsPerGroup == 1 ? (int)((uint32_t)item / (uint32_t)p.chunks) : (int)(item / p.chunks);
  const int chunk = (int)(item - (int64_t)t * p.chunks);
  const int n_heads = p.n_q + 2 * p.n_kv;
  const int h_begin = chunk * kHeadsPerGroup;
  const int h_end = min(h_begin + kHeadsPerGroup, n_heads);

  const int off = j * E;
  // a head's row and, for q and k, its norm weights; asked for one head ahead, the first ones before
  // the sines and cosines
  struct Head {
    V lo, hi, wl, wh;
  };
  auto fetch = [&](int h) {
    Head x{};
    const uint16_t* src = h < p.n_q ? p.q + (int64_t)t * p.q_stride0 + (int64_t)h * D
                          : h < p.n_q + p.n_kv ? p.k + (int64_t)t * p.k_stride0 + (int64_t)(h - p.n_q) * D
                                               : p.v + (int64_t)t * p.v_stride0 + (int64_t)(h - p.n_q - p.n_kv) * D;
    const uint16_t* w = h < p.n_q ? p.q_weight : p.k_weight;  // of no use to a v head
    x.lo = *reinterpret_cast<const V*>(src + off);
    x.hi = *reinterpret_cast<const V*>(src + D / 2 + off);
    x.wl = *reinterpret_cast<const V*>(w + off);
    x.wh = *reinterpret_cast<const V*>(w + D / 2 + off);
    return x;
  };
  const int32_t position = p.positions[t];
  const int64_t slot = p.out_loc[t];
  Head next = fetch(h_begin);

  // sines and cosines of this lane's pairs (only if the chunk holds a q or k head)
  float cs[E], sn[E];
  if (h_begin < p.n_q + p.n_kv) {
    const float pos = (float)position;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      sincosf(rope_angle<D>(pos, j * E + e, p.log2_base), &sn[e], &cs[e]);
    }
  }
  // a slot id outside the pools stores no k / v row (q_out is still produced): a wild store
  // would be a GPU memory fault
  const bool slot_ok = (uint64_t)slot < (uint64_t)p.num_slots;

  for (int h = h_begin; h < h_end; ++h) {
    uint16_t* dst = h < p.n_q ? p.q_out + ((int64_t)t * p.n_q + h) * D
                    : h < p.n_q + p.n_kv ? p.k_cache + slot * p.kc_stride0 + (int64_t)(h - p.n_q) * D
                                         : p.v_cache + slot * p.vc_stride0 + (int64_t)(h - p.n_q - p.n_kv) * D;
    V lo = next.lo, hi = next.hi;
    const V wl = next.wl, wh = next.wh;
    if (h + 1 < h_end) next = fetch(h + 1);
    if (h < p.n_q + p.n_kv) norm_rope_head<D>(lo, hi, wl, wh, cs, sn, p.eps);
    if (h >= p.n_q && !slot_ok) continue;
    *reinterpret_cast<V*>(dst + off) = lo;
    *reinterpret_cast<V*>(dst + D / 2 + off) = hi;
  }
}

}  // namespace

int launch_qk_norm_rope_store(const NormRopeArgs& a, hipStream_t stream) {
  NormRopeParams p;
  p.q = static_cast<const uint16_t*>(a.q);
  p.k = static_cast<const uint16_t*>(a.k);
  p.v = static_cast<const uint16_t*>(a.v);
  p.q_weight = static_cast<const uint16_t*>(a.q_weight);
  p.k_weight = static_cast<const uint16_t*>(a.k_weight);
  p.positions = a.positions;
  p.out_loc = a.out_loc;
  p.q_out = static_cast<uint16_t*>(a.q_out);
  p.k_cache = static_cast<uint16_t*>(a.k_cache);
  p.v_cache = static_cast<uint16_t*>(a.v_cache);
  p.q_stride0 = a.q_stride0;
  p.k_stride0 = a.k_stride0;
  p.v_stride0 = a.v_stride0;
  p.kc_stride0 = a.kc_stride0;
  p.vc_stride0 = a.vc_stride0;
  p.num_slots = a.num_slots;
  p.n_tokens = (int32_t)a.n_tokens;
  p.n_q = (int32_t)a.n_q;
  p.n_kv = (int32_t)a.n_kv;
  const int64_t n_heads = a.n_q + 2 * a.n_kv;
  // one head per group until its workgroups fill the chip twice over
  const bool few = a.n_tokens * n_heads <= 512 * (kThreads / kGroupLanes);
  const int per_group = few ? 1 : kHeadsPerGroupMany;
  p.chunks = (int32_t)((n_heads + per_group - 1) / per_group);
  p.eps = a.eps;
  p.log2_base = log2f(a.rope_base);
  const int64_t items = a.n_tokens * p.chunks;
  const int64_t per_block = kThreads / kGroupLanes;
  const int64_t blocks = (items + per_block - 1) / per_block;
  if (blocks <= 0) return MSGL_OK;
  if (blocks > 0x7fffffffLL) return MSGL_ERR_SHAPE;
  if (a.head_dim != 128 && a.head_dim != 256) return MSGL_ERR_HEAD_DIM;
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kThreads), 0, stream, p); };
  if (a.head_dim == 128) few ? launch(qk_norm_rope_store_kernel<128, 1>) : launch(qk_norm_rope_store_kernel<128, kHeadsPerGroupMany>);
  else few ? launch(qk_norm_rope_store_kernel<256, 1>) : launch(qk_norm_rope_store_kernel<256, kHeadsPerGroupMany>);
  return check_launch();
}

}  // namespace msgl
