// Gated delta-rule recurrence with a slot-indexed fp32 state that is updated in place.
// Replaces gdn_state_inplace (mini-sglang-mlx-kernel/csrc/gdn_state.metal:14-99, host side
// gdn_state.cpp:87-183).  For request b with state rows S[hv][dv][dk] at slot slot_ids[b] and
// every token t of the request, in order:
//     S *= g[t, hv]
//     delta = (v[t, hv, dv] - <S[hv][dv][:], k[t, hk]>) * beta[t, hv]
//     S[hv][dv][:] += k[t, hk] * delta
//     y[t, hv, dv] = <S[hv][dv][:], q[t, hk]>                    hk = hv / (HV / HK)
// q, k, v, g, beta, y are bf16; the state and all arithmetic are fp32.
//
// One state row (dk = 128 floats) lives in the registers of 16 lanes, 8 values each (for one token 4 neighbours of each half, so that a
// load or store of a wave is 256 bytes of 4 rows: two whole lines each), for the whole token loop: the two inner products are 8 lane-local FMAs and a 4-step rotate-and-add
// inside the 16-lane DPP row (no LDS, no cross-row traffic).  A lane group carries R rows, so
// one load of k and q serves R independent recurrences whose latencies overlap; the inputs of
// the next kDepth tokens are always in flight.  Decode (one token) is
// HBM-bound: 2 * dv * dk * 4 bytes of state per (request, hv head) read and written once, past the caches where
// launch_gdn_state() says so: 64 requests of 32 heads 53.2 -> 45.9 us, 5.85 TB/s (a large copy reaches 4.9; 8 neighbours to a lane, 16 bytes
// of every 32 a load: plain 52.8, past the caches 53.7).
// Prefill is a serial chain per row (as in the reference); parallelism is batch * hv * dv rows.  It takes
// requests of very few tokens here; longer ones go in chunks (gdn_short.hip, gdn_chunk.hip; gdn_route.h).
#include <algorithm>
#include <type_traits>

#include "gdn_params.h"
#include "gdn_route.h"

namespace msgl {
namespace {

constexpr int kLanesPerRow = 16;
constexpr int kPerLane = kDK / kLanesPerRow;  // 8 state values per lane and row

template <int N>
__device__ __forceinline__ float row_rotate(float x) {  // lane i of a 16-lane row reads lane (i + N) % 16
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x),
                                                               0x120 + N, 0xf, 0xf, true));
}
__device__ __forceinline__ float row_sum(float x) {  // every lane of the row gets the sum
  x += row_rotate<8>(x);
  x += row_rotate<4>(x);
  x += row_rotate<2>(x);
  x += row_rotate<1>(x);
  return x;
}

__device__ __forceinline__ void unpack8(const u32x4_t raw, float (&f)[kPerLane]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    f[2 * e] = __builtin_bit_cast(float, raw[e] << 16);
    f[2 * e + 1] = __builtin_bit_cast(float, raw[e] & 0xffff0000u);
  }
}

// R = dv rows per 16-lane group.  Workgroup = 256 threads = 16 groups = 16 R consecutive rows
// of one (request, hv head).
template <int R, int kDepth, bool STREAM>
__global__ __launch_bounds__(256) void gdn_state_kernel(GdnParams p) {
  constexpr int kRowsPerBlock = 16 * R;
  constexpr int kBlocksPerHead = kDV / kRowsPerBlock;
  const int lane16 = threadIdx.x & 15;
  const int group = threadIdx.x >> 4;
  const int head_item = blockIdx.x / kBlocksPerHead;      // (request, hv head)
  const int row0 = (blockIdx.x - head_item * kBlocksPerHead) * kRowsPerBlock + group * R;
  const int b = head_item / p.hv;
  const int hv = head_item - b * p.hv;
  const int hk = hv / p.hv_per_hk;
  const int start = p.single_token ? b : p.qo_indptr[b];
  const int end = min(p.single_token ? b + 1 : p.qo_indptr[b + 1], p.tokens);
  if (end <= start) return;  // nothing to do: the state stays as it is

  // One token: 4 neighbours of each half, whole lines of state a load.  Several: 8 neighbours, which take one load of k and of q each
  // instead of two (us: one request of 4 and 8 tokens, 32 heads, 4.67 and 5.78, by halves 4.79 and 5.93).
  constexpr bool kHalves = kDepth == 1;
  constexpr int kSecond = kHalves ? kDK / 2 : 4;
  const int lane_at = lane16 * (kHalves ? 4 : kPerLane);
  float* srow = p.state + (int64_t)p.slot_ids[b] * p.state_stride0 +
                ((int64_t)hv * kDV + row0) * kDK + lane_at;
  auto load_state = [](const float* from) {
    if constexpr (STREAM) return __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(from));
    else return *reinterpret_cast<const f32x4_t*>(from);
  };
  float s[R][kPerLane];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const f32x4_t a = load_state(srow + r * kDK), c = load_state(srow + r * kDK + kSecond);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s[r][e] = a[e];
      s[r][4 + e] = c[e];
    }
  }

  auto lane_dims = [&](const uint16_t* row) {
    if constexpr (!kHalves) return ld_global_b128(row + lane_at);
    const u32x2_t a = *reinterpret_cast<const u32x2_t*>(row + lane_at), c = *reinterpret_cast<const u32x2_t*>(row + kSecond + lane_at);
    return u32x4_t{a[0], a[1], c[0], c[1]};
  };
  auto load_token = [&](int t, u32x4_t& kraw, u32x4_t& qraw, uint32_t& graw, uint32_t& braw,
                        uint32_t (&vraw)[R]) {
    kraw = lane_dims(p.k + (int64_t)t * p.k_stride0 + hk * kDK);
    qraw = lane_dims(p.q + (int64_t)t * p.q_stride0 + hk * kDK);
    graw = p.g[(int64_t)t * p.hv + hv];
    braw = p.beta[(int64_t)t * p.hv + hv];
#pragma unroll
    for (int r = 0; r < R; ++r) vraw[r] = p.v[(int64_t)t * p.v_stride0 + hv * kDV + row0 + r];
  };

  // The inputs of the next kDepth tokens are always in flight: one iteration is far shorter
  // than a memory round trip, so a single token of lookahead would leave every iteration
  // waiting for its loads.  Loads are unconditional (clamped to the request's last token).
  struct TokenIn {
    u32x4_t kraw, qraw;
    uint32_t graw, braw, vraw[R];
  };
  TokenIn ring[kDepth];
#pragma unroll
  for (int j = 0; j < kDepth; ++j)
    load_token(min(start + j, end - 1), ring[j].kraw, ring[j].qraw, ring[j].graw, ring[j].braw, ring[j].vraw);
  for (int t0 = start; t0 < end; t0 += kDepth) {
#pragma unroll
    for (int j = 0; j < kDepth; ++j) {
      const int t = t0 + j;
      const TokenIn in = ring[j];
      load_token(min(t + kDepth, end - 1), ring[j].kraw, ring[j].qraw, ring[j].graw, ring[j].braw, ring[j].vraw);
      if (t >= end) break;  // the same for every lane of the workgroup
      float kf[kPerLane], qf[kPerLane];
      unpack8(in.kraw, kf);
      unpack8(in.qraw, qf);
      const float gs = bf16_bits_to_f32(in.graw), bs = bf16_bits_to_f32(in.braw);
      float out[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        // two partial sums per inner product: half the length of the dependent FMA chain
        float dot0 = 0.f, dot1 = 0.f;
#pragma unroll
        for (int e = 0; e < kPerLane; e += 2) {
          s[r][e] *= gs;
          s[r][e + 1] *= gs;
          dot0 = __builtin_fmaf(s[r][e], kf[e], dot0);
          dot1 = __builtin_fmaf(s[r][e + 1], kf[e + 1], dot1);
        }
        const float delta = (bf16_bits_to_f32(in.vraw[r]) - row_sum(dot0 + dot1)) * bs;
        float o0 = 0.f, o1 = 0.f;
#pragma unroll
        for (int e = 0; e < kPerLane; e += 2) {
          s[r][e] = __builtin_fmaf(kf[e], delta, s[r][e]);
          s[r][e + 1] = __builtin_fmaf(kf[e + 1], delta, s[r][e + 1]);
          o0 = __builtin_fmaf(s[r][e], qf[e], o0);
          o1 = __builtin_fmaf(s[r][e + 1], qf[e + 1], o1);
        }
        out[r] = row_sum(o0 + o1);
      }
      // lane r of the group writes row r
      float mine = out[0];
#pragma unroll
      for (int r = 1; r < R; ++r) mine = (lane16 == r) ? out[r] : mine;
      if (lane16 < R)
        p.y[((int64_t)t * p.hv + hv) * kDV + row0 + lane16] = __builtin_bit_cast(uint16_t, (__bf16)mine);
    }
  }

  auto store_state = [](float* to, f32x4_t x) {
    if constexpr (STREAM) __builtin_nontemporal_store(x, reinterpret_cast<f32x4_t*>(to));
    else *reinterpret_cast<f32x4_t*>(to) = x;
  };
#pragma unroll
  for (int r = 0; r < R; ++r) {
    f32x4_t a, c;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      a[e] = s[r][e];
      c[e] = s[r][4 + e];
    }
    store_state(srow + r * kDK, a);
    store_state(srow + r * kDK + kSecond, c);
  }
}

}  // namespace

static GdnRoute route_of(const GdnArgs& a) {
  if (a.v_stride0 >= (1 << 24) || a.k_stride0 >= (1 << 24) || a.q_stride0 >= (1 << 24) || a.hv >= (1 << 17))
    return GdnRoute::kTokens;  // the others' offsets inside a chunk are 32 bits wide
  if ((uintptr_t)a.v % 16 || a.v_stride0 % 8 || (uintptr_t)a.y % 8) return GdnRoute::kTokens;  // loads of 16 bytes, stores of 8
  return gdn_route(a.tokens, a.batch, a.hv, a.longest, device_cus());
}
static thread_local int t_force_rows = 0;  // benchmarking switch, one value per host thread
// Room for the systems of all chunks where making those in a launch of their own pays (gdn_long.hip), 0 elsewhere.  The second
// launch costs 3 to 5 us and saves a tenth to a quarter of a long request's chain; where the requests' heads fill the chip it
// also deals them out by their lengths, which the one launch does not.  680 launches at 32 heads, even, ragged and of one long request
// beside short ones, time in two launches by that in one: one request of 256-320 tokens 1.00, 352-384 0.96; two and three, by
// their mean, 320-384 even 1.01, ragged 0.97, 384-448 0.985 and 0.93; four, whose pairs of workgroups fill the chip in one round, even
// 320-384 1.06, 384-448 1.01, 512-640 0.975, ragged 0.85-1.00; five to eight even 128-192 0.94-1.10, 192-256 0.91-1.05, 256-320 0.93, ragged
// 0.96 and one long 0.68 in all of these; more 96-128 0.99 (up to 1.03), 128-192 0.97, 0.96 and 0.74.  The lines lie where even ones do not
// lose either.  Few heads a request bring more requests to as many workgroups, and even ones then lose (us, in one launch and in two: 32 of
// 452 tokens, 4 heads, 43.6 and 49.6, 64 of 319 69 and 75, 10 of 445 29.6 and 33.6), so the lines go up with the requests' number.  750 launches at
// 2-128 heads, two launches by one: those beyond the lines 0.903 (geometric mean of 583, worst 1.01), those that this leaves behind 0.991 of 167.
// us: one of 4000 208 -> 156, eight of 200-1600 148 -> 139, 2060 among five of 100-260 150 -> 91.  A request and 32 heads
// have 640 KiB for every 64 tokens; a launch that would need more than 2 GiB goes without.
size_t gdn_state_workspace_bytes(int64_t tokens, int64_t batch, int64_t hv, bool single_token) {
  if (single_token || batch <= 0 || hv <= 0 || t_force_rows > 0) return 0;
  const int64_t heads = batch * hv, cus = device_cus();
  auto line = [batch](int64_t least, int64_t most, int64_t step, int64_t from) {
    return std::min(most, least + step * std::max<int64_t>(batch - from, 0));
  };
  const int64_t mean = 8 * heads <= cus && batch <= 3 ? 352
                       : 8 * heads <= 3 * cus         ? line(384, 704, 48, 3)
                       : 2 * heads <= cus             ? line(448, 768, 48, 4)
                       : heads <= cus                 ? line(256, 512, 8, 16)
                       : heads <= 2 * cus && batch >= 48 && batch <= kWave ? 256
                                                                          : 128;
  if (tokens < mean * batch) return 0;
  const size_t bytes = gdn_long_workspace_bytes(tokens, batch, hv);
  return bytes <= ((size_t)2 << 30) ? bytes : 0;
}
void gdn_set_rows(int v) { t_force_rows = (v == 1 || v == 2 || v == 4) ? v : 0; }

int launch_gdn_state(const GdnArgs& a, hipStream_t stream) {
  GdnParams p;
  p.state = static_cast<float*>(a.state);
  p.y = static_cast<uint16_t*>(a.y);
  p.q = static_cast<const uint16_t*>(a.q);
  p.k = static_cast<const uint16_t*>(a.k);
  p.v = static_cast<const uint16_t*>(a.v);
  p.g = static_cast<const uint16_t*>(a.g);
  p.beta = static_cast<const uint16_t*>(a.beta);
  p.slot_ids = a.slot_ids;
  p.qo_indptr = a.qo_indptr;
  p.state_stride0 = a.state_stride0;
  p.q_stride0 = a.q_stride0;
  p.k_stride0 = a.k_stride0;
  p.v_stride0 = a.v_stride0;
  p.batch = (int32_t)a.batch;
  p.hv = (int32_t)a.hv;
  p.hv_per_hk = (int32_t)(a.hv / a.hk);
  p.tokens = (int32_t)a.tokens;
  p.single_token = a.single_token_mode ? 1 : 0;
  const int64_t heads = a.batch * a.hv;
  if (heads <= 0) return MSGL_OK;
  if (!p.single_token && t_force_rows == 0) {
    const GdnRoute route = route_of(a);
    if (route == GdnRoute::kShort) return launch_gdn_short(p, stream);
    if (route == GdnRoute::kChunks) {
      const size_t bytes = gdn_state_workspace_bytes(a.tokens, a.batch, a.hv, false);
      if (bytes > 0 && a.workspace != nullptr && a.workspace_bytes >= bytes) return launch_gdn_long(p, a.workspace, stream);
      return launch_gdn_chunks(p, stream);
    }
  }
  // more rows per lane group (more overlap inside a wave) once there are enough workgroups
  // to fill the chip without it
  const int64_t blocks_r1 = heads * (kDV / 16);
  int r = 1;
  if (blocks_r1 >= 8 * 1024) r = 4;
  else if (blocks_r1 >= 4 * 1024) r = 2;
  // Decode: the state once in and once out, past the caches from 96 MiB on, and up to 24 MiB, what the L2 caches have room for beside
  // the next pass's.  us, rows 1, 2, 4, plain / past the caches, three sets of states in turn: 14 MiB 7.6, 7.5, 7.4 / 8.0, 7.1, 6.3, 24 MiB 10.3, 9.5, 9.6 /
  // 12.8, 10.5, 9.2, 28 MiB 11.6, 10.9, 10.8 / 14.6, 12.0, 12.0, 64 MiB 22.0, 21.4, 20.6 / 28.4, 24.4, 24.7 (in the last level from the pass before), 92 MiB 38.9, 32.2, 32.8 / 41.1, 33.7, 34.7, 104 MiB
  // 43.9, 38.5, 39.2 / 46.2, 38.1, 38.9, 128 MiB 52.6, 48.9, 52.1 / 51.2, 45.9, 47.2, 512 MiB 210, 200, 210 / 206, 178, 190; up to 12 MiB 5.4 to 6.5 all.
  // (With twelve sets 28 MiB 14.5, 13.6, 14.5 / 14.7, 12.4, 12.8, 64 MiB 28.9, 27.9, 29.0 / 28.5, 24.9, 25.3.)
  const int64_t state_bytes = heads * kDV * kDK * (int64_t)sizeof(float);
  const bool large = streams(state_bytes, 96 << 10);
  const bool stream_state = p.single_token && (large || (state_bytes <= (24 << 20) && streams(state_bytes, 0)));
  if (p.single_token) r = large || heads <= 192 ? 2 : 4;
  if (t_force_rows > 0) r = t_force_rows;
  const int64_t blocks = heads * (kDV / (16 * r));
  if (blocks > 0x7fffffffLL) return MSGL_ERR_SHAPE;
  const dim3 grid((unsigned)blocks), block(256);
  // decode has one token per request: nothing to look ahead to
  auto launch = [&](auto depth, auto past) {
    constexpr int N = decltype(depth)::value;
    constexpr bool STREAM = decltype(past)::value;
    return launch_kernel(r == 4 ? gdn_state_kernel<4, N, STREAM> : r == 2 ? gdn_state_kernel<2, N, STREAM> : gdn_state_kernel<1, N, STREAM>, grid,
                         block, stream, p);
  };
  if (!p.single_token) return launch(std::integral_constant<int, 8>{}, std::false_type{});
  if (stream_state) return launch(std::integral_constant<int, 1>{}, std::true_type{});
  return launch(std::integral_constant<int, 1>{}, std::false_type{});
}

}  // namespace msgl
