// Gated delta rule in chunks of 16 tokens: requests of a few dozen tokens, and of up to 127 where there are many.  Notation, and why
// the chunkwise form is right: gdn_chunk.hip.
//
// Token after token (gdn_state.hip) a wave has four state rows and spends 90 instructions on each token of each; its inputs in
// flight take 130 registers, so three waves share a SIMD and five requests go in two rounds: 0.3 us a token for one request, 0.8 us for
// five, 1.5 us for sixteen.  A chunk of 64 (gdn_chunk.hip) takes all of a compute unit's LDS, 12.8 us a round of workgroups whatever
// the chunk holds.  A chunk of 16 is one tile of the matrix instructions: its triangular system is one block whose inverse is made in
// registers (eliminate()), and all products of 16 state rows fit one wave, state included, so waves meet only where one makes the
// system that the others use too:
//     X = K S^T, Z = S Q^T          12 products each, S in three bf16 parts (16 products take them off)
//     R = beta (V - G X), U = T R   4 fp32 products
//     Y = G Z + P U                 4 fp32 products, transposed: a lane stores four rows of a token
//     S = G S + K^T (tail U)        16 products: two parts of U side by side in the 32 columns of one, the third beside zeros
// A workgroup takes a head, or half of one where that fills the chip better (launch_gdn_short()).  Chunks go in groups of four: each
// of four waves fetches the rows of one and makes its system; the next group's rows are asked for in a group's first chunk.  K and Q come by
// LDS, four whole rows a load, once for all waves: as operands straight from memory, 16 rows a load, the address unit was the limit
// (16 requests of 64 tokens 38 us, now 26).  74 KB of LDS and 128 registers let two workgroups of eight waves share a compute unit
// (lane_here() keeps what only a group's start needs out of the registers: in it they were 16 too many, 5-15 % of the time).
//
// What bounds it: up to 16 tokens the state, read and written (16 requests of 32 heads of 8 tokens 13.5 us, 5.0 TB/s); beyond, the
// chain of a chunk, 1.25 us for one request, 1.45 for four, and from eight on the issue of the waves of a SIMD, 0.2-0.3 us a chunk and request, the
// matrix pipe busy for a quarter to 38 % of the cycles.  A chunk ends in a wait for all memory operations of its wave (behind V's loads, which
// are under a condition, and the masked rows of Y the compiler does not know how many are under way): V's round trip is in every chunk,
// that of the next group's K and Q in a group's first.  us, by requests of 32 heads and tokens, before and now: 1 x 16 8.3 and 6.0, 32 9.3
// and 6.7; 4 x 16 12.1 and 7.2; 8 x 16 24.9 and 9.1, 40 24.9 and 12.5; 16 x 40 50.7 and 21.5; 24 x 80 105 and 44; 48 x 8 57 and 42.7.  Four more
// waves that fetch and make the systems ahead: 1.1 us a chunk for one request, no change for four.
//
// Precision: fp32 throughout, the parts are exact (see upper()).  The state's error against 64 bits, rms: 1.0-1.7e-8 at states of 0.1
// (the token kernel 1.2-2.5e-8, chunks of 64 1.2-1.8e-8); the chunk's addition to S in a sum of its own, joined by one multiply-add, is 7-10 %
// of that.  Infinities and NaN as in gdn_chunk.hip: a wave whose U or P is not finite goes through its request again.
#include "gdn_chunk_tiles.h"

namespace msgl {
namespace {

constexpr int kShortChunk = 16, kGroup = 4;  // tokens of a chunk, chunks whose systems are made side by side

// The values of the four rows of 16 lanes, each in all of them.
__device__ __forceinline__ void spread(float x, float (&of)[4]) {
  const uint32_t bits = __builtin_bit_cast(uint32_t, x);
  const auto halves = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
  const auto low = __builtin_amdgcn_permlane16_swap(halves[0], halves[0], false, false);
  const auto high = __builtin_amdgcn_permlane16_swap(halves[1], halves[1], false, false);
  of[0] = __builtin_bit_cast(float, (uint32_t)low[0]);
  of[1] = __builtin_bit_cast(float, (uint32_t)low[1]);
  of[2] = __builtin_bit_cast(float, (uint32_t)high[0]);
  of[3] = __builtin_bit_cast(float, (uint32_t)high[1]);
}

// A chunk's part that depends on no state, lane % 16 the token, 4 g .. the ones before it: the inverse, the products of q and k.
struct ShortSystem {
  f32x4_t t[64], p[64];
  float beta[kShortChunk], gamma[kShortChunk], tail[kShortChunk], g[2][kShortChunk];
};
struct ShortLds {
  uint16_t k[2][kGroup][kShortChunk][kDK], q[2][kGroup][kShortChunk][kDK];
  ShortSystem systems[kGroup];
};

// The lane, where what follows from it is not worth a register for the whole kernel.
__device__ __forceinline__ int lane_here() {
  uint32_t lane = lane_id();
  pin(lane);
  return (int)lane;
}
__device__ __forceinline__ void load_rows(const uint16_t* m, uint32_t place, bf16x8_t (&x)[4]) {
#pragma unroll
  for (int c = 0; c < 4; ++c) x[c] = operand(m + (place ^ 32 * c));
}

// Decays of a chunk, a token per lane % 16 (1 past the end).
struct ShortDecays {
  float pre, suf, quad_pre;  // products up to the token, behind it, up to it within its quad
  __device__ __forceinline__ ShortDecays(float gv, int x16) {
    const float before1 = row_shift<0x111>(gv);
    pre = gv * before1;
    suf = gv * row_shift<0x101>(gv);
    quad_pre = gv * ((x16 & 3) >= 1 ? before1 : 1.f);
    const float quad2 = row_shift<0x112>(quad_pre);
    quad_pre *= (x16 & 3) >= 2 ? quad2 : 1.f;
    pre *= row_shift<0x112>(pre);
    suf *= row_shift<0x102>(suf);
    pre *= row_shift<0x114>(pre);
    suf *= row_shift<0x104>(suf);
    pre *= row_shift<0x118>(pre);
    suf *= row_shift<0x108>(suf);
    suf = row_shift<0x101>(suf);
  }
  // token t = lane % 16 against the tokens i = 4 g + n before it; `decays` is room for the 16 of them
  __device__ __forceinline__ f32x4_t ratios(float gv, float* decays, int x16, int g) const {
    decays[x16] = gv;
    __builtin_amdgcn_wave_barrier();
    const f32x4_t decay = *reinterpret_cast<const f32x4_t*>(&decays[4 * g]);
    auto lane_value = [](float f, int l) {
      return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f), l));
    };
    const float quad_1 = lane_value(quad_pre, 7), quad_2 = lane_value(quad_pre, 11);
    const float far = quad_pre * (g < 1 && x16 >= 8 ? quad_1 : 1.f) * (g < 2 && x16 >= 12 ? quad_2 : 1.f);
    f32x4_t ratio;
    ratio[3] = (x16 >> 2) > g ? far : 1.f;
#pragma unroll
    for (int n = 2; n >= 0; --n) ratio[n] = ratio[n + 1] * (4 * g + n + 1 <= x16 ? decay[n + 1] : 1.f);
    return ratio;
  }
};
__device__ __forceinline__ void make_inverse(ShortSystem& to, const uint16_t* k, uint32_t place, float gv, float bv) {
  const int lane = lane_here(), x16 = lane & 15, g = lane >> 4;
  bf16x8_t rows[4];
  load_rows(k, place, rows);
  const ShortDecays decays(gv, x16);
  to.beta[x16] = bv;
  to.gamma[x16] = decays.pre;
  to.tail[x16] = decays.suf;
  const f32x4_t ratio = decays.ratios(gv, to.g[0], x16, g);
  const f32x4_t kk = block_dots(rows, rows);
  f32x4_t inv;
  float minus_a[16];
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    float of[4];
    spread(4 * g + n < x16 ? -bv * ratio[n] * kk[n] : 0.f, of);
#pragma unroll
    for (int i = 0; i < 4; ++i) minus_a[4 * i + n] = of[i];
    inv[n] = 4 * g + n == x16 ? 1.f : 0.f;
  }
  eliminate<0>(minus_a, inv);
  to.t[lane] = inv;
}
__device__ __forceinline__ void make_products(ShortSystem& to, const uint16_t* k, const uint16_t* q, uint32_t place, float gv) {
  const int lane = lane_here(), x16 = lane & 15, g = lane >> 4;
  bf16x8_t k_rows[4], q_rows[4];
  load_rows(k, place, k_rows);
  load_rows(q, place, q_rows);
  const f32x4_t ratio = ShortDecays(gv, x16).ratios(gv, to.g[1], x16, g);
  f32x4_t pt = block_dots(k_rows, q_rows);
#pragma unroll
  for (int n = 0; n < 4; ++n) pt[n] = 4 * g + n <= x16 ? ratio[n] * pt[n] : 0.f;
  to.p[lane] = pt;
}

// The upper halves of four values, and of eight.  Parts as in split(), but cut instead of rounded: three of 8 significant bits and one
// sign, exact as well (a permutation takes 5 cycles where a conversion takes 8).
__device__ __forceinline__ u32x2_t upper(f32x4_t f) {
  const u32x4_t bits = __builtin_bit_cast(u32x4_t, f);
  return u32x2_t{__builtin_amdgcn_perm(bits[1], bits[0], 0x07060302u), __builtin_amdgcn_perm(bits[3], bits[2], 0x07060302u)};
}
__device__ __forceinline__ bf16x8_t upper(f32x4_t a, f32x4_t b) {
  const u32x2_t x = upper(a), y = upper(b);
  return as_bf16x8(u32x4_t{x[0], x[1], y[0], y[1]});
}
// A wave's 16 state rows by whole lines, which can go past the caches: a load takes 128 bytes of 8 rows, s[2 c] of rows lane % 8, s[2 c + 1]
// of the others, and of the line's pieces of 16 bytes the lanes below 8 of 16 the even ones.  Lanes 8 apart then give each other
// what is of the other's row, and the same brings them back.
__device__ __forceinline__ float* state_lines(int slot, int hv, int row) {
  uint32_t lane = lane_id();
  pin(lane);
  return parameter(&GdnParams::state) + (int64_t)slot * parameter(&GdnParams::state_stride0) +
         ((int64_t)hv * kDV + row + (lane & 7)) * kDK + 8 * (lane >> 4) + 4 * ((lane >> 3) & 1);
}
__device__ constexpr int line_at(int c) { return 32 * (c >> 1) + 8 * kDK * (c & 1); }
__device__ __forceinline__ void exchange_lines(f32x4_t (&s)[8]) {
  constexpr int kRor8 = 0x128;  // DPP: from the lane 8 away in a row of 16
#pragma unroll
  for (int c = 0; c < 8; c += 2)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float even = s[c][i], odd = s[c + 1][i];  // (a bit cast of an element itself takes the first one)
      const int a = __builtin_bit_cast(int, even), b = __builtin_bit_cast(int, odd);
      s[c][i] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(a, b, kRor8, 0xf, 0xc, false));
      s[c + 1][i] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(b, a, kRor8, 0xf, 0x3, false));
    }
}
// WAVES: 8, a head's rows in one workgroup, or 4, half of them; LINES: the state by whole lines, past the caches
template <int WAVES, bool LINES>
__global__ __launch_bounds__(64 * WAVES, WAVES / 2) void gdn_short_kernel(GdnParams p) {
  __shared__ __attribute__((aligned(16))) ShortLds lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int kParts = kDV / (16 * WAVES);
  const int item = blockIdx.x / kParts, b = item / p.hv, hv = item - b * p.hv, hk = hv / p.hv_per_hk;
  const int start = p.qo_indptr[b], end = min(p.qo_indptr[b + 1], p.tokens), slot = p.slot_ids[b];
  if (end <= start) return;  // the whole workgroup: the state stays as it is
  const int row = 16 * (WAVES * (blockIdx.x - item * kParts) + wave);
  const int lane = lane_id(), x16 = lane & 15, g = lane >> 4;

  // rows past the request's end: its last row (beta is zero there, and their rows of Y are not stored)
  const int of_group = wave & (kGroup - 1);  // the chunk of a group that this wave fetches, and makes the system of
  const uint32_t k_step = (uint32_t)p.k_stride0 * 2u, q_step = (uint32_t)p.q_stride0 * 2u, v_step = (uint32_t)p.v_stride0 * 2u;
  auto fetch = [&](const uint16_t* m, uint32_t step, const uint16_t (*to)[kDK], int first) {
    const char* const base = reinterpret_cast<const char*>(m) + (int64_t)first * step;
    const uint32_t at = __builtin_amdgcn_readfirstlane((uint32_t)reinterpret_cast<uintptr_t>(to)), last = end - 1 - first;
    const int lane = lane_here();
#pragma unroll
    for (int n = 0; n < 4; ++n) {  // four rows a load
      const uint32_t t = 4 * n + (lane >> 4);
      lds_direct_b128(at + 1024 * n, base, min(t, last) * step + 16 * piece(t, lane & 15));
    }
  };
  uint32_t graw = 0, braw = 0;
  auto fetch_group = [&](int j) {  // a wave's part of chunks j to j + 3
    const int first = start + kShortChunk * (j + of_group);
    if (first >= end) return;
    const int64_t token = (int64_t)min(first + (lane_here() & 15), end - 1) * p.hv + hv;
    graw = p.g[token];
    braw = p.beta[token];
    const int par = (j / kGroup) & 1;
    if (WAVES == 4 || wave < kGroup) fetch(p.k + hk * kDK, k_step, lds.k[par][of_group], first);
    if (WAVES == 4 || wave >= kGroup) fetch(p.q + hk * kDK, q_step, lds.q[par][of_group], first);
  };
  uint32_t v[4];  // tokens 4 g .., row lane % 16
  const char* v_chunk = reinterpret_cast<const char*>(p.v + (int64_t)start * p.v_stride0 + hv * kDV + row);
  auto load_v = [&](int first) {
    const int last = end - 1 - first;
#pragma unroll
    for (int n = 0; n < 4; ++n) v[n] = *reinterpret_cast<const uint16_t*>(v_chunk + ((uint32_t)min(4 * g + n, last) * v_step + 2 * x16));
    v_chunk += kShortChunk * (int64_t)v_step;
  };
  fetch_group(0);
  float* srow = nullptr;  // (by whole lines it is found anew behind the chunks: kept it is two more spilled registers, and 3-8 % of the time)
  f32x4_t s[8];  // s[2 c + h][i]: dim 32 c + 8 g + 4 h + i of row lane % 16
  if constexpr (LINES) {
    const float* const from = state_lines(slot, hv, row);
#pragma unroll
    for (int c = 0; c < 8; ++c) s[c] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(from + line_at(c)));
    exchange_lines(s);
  } else {
    srow = state_row(slot, hv, row);
#pragma unroll
    for (int c = 0; c < 8; ++c) s[c] = *reinterpret_cast<const f32x4_t*>(srow + 32 * (c >> 1) + 4 * (c & 1));
  }
  load_v(start);
  const Picker pick;
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  const uint32_t y_step = (uint32_t)p.hv * kDV * 2u, y_at = x16 * y_step + 8 * g;
  char* y_chunk = reinterpret_cast<char*>(p.y + ((int64_t)start * p.hv + hv) * kDV + row);
  // places of the rows' pieces as operands (row lane % 16), and transposed (row 4 g + lane % 16 / 4)
  const int trow = 4 * g + (x16 >> 2);
  const uint32_t place = x16 * kDK + 8 * piece(x16, g), transposed = trow * kDK + 8 * piece(trow, x16 & 3);
  float most = 0.f;

  for (int first = start, j = 0; first < end; first += kShortChunk, ++j) {
    const int of = j & (kGroup - 1), par = (j / kGroup) & 1;
    if (of == 0) {
      // the group's rows: what this wave asked for last are the state and V, or V and rows of Y of three chunks
      wait_vm_at_most<12>();
      slot_barrier();
      const int mine = first + kShortChunk * of_group;
      if (mine < end) {
        const bool there = mine + x16 < end;
        const float gv = there ? bf16_bits_to_f32(graw) : 1.f, bv = there ? bf16_bits_to_f32(braw) : 0.f;
        ShortSystem& to = lds.systems[of_group];
        if (WAVES == 4 || wave < kGroup) make_inverse(to, &lds.k[par][of_group][0][0], place, gv, bv);
        if (WAVES == 4 || wave >= kGroup) make_products(to, &lds.k[par][of_group][0][0], &lds.q[par][of_group][0][0], place, gv);
      }
    }
    // X = K S^T, tokens on the rows, and Z = S Q^T, tokens on the columns
    const uint16_t *const k = &lds.k[par][of][0][0], *const q = &lds.q[par][of][0][0];
    // The parts of S come off for 64 dims at a time, the products with the first ones in a sum of their own, so that the matrix
    // pipe has work while the next is taken off (32 dims at a time 2-6 % slower, 128 twice as slow for want of registers).
    constexpr int kSide = 2;
    f32x4_t x = zero, z = zero, x_rest = zero, z_rest = zero;
#pragma unroll
    for (int h = 0; h < 4; h += kSide) {
      bf16x8_t kc[kSide], qc[kSide], part[kSide];
      f32x4_t a[kSide], b[kSide];
      auto take_off = [&] {
#pragma unroll
        for (int c = 0; c < kSide; ++c) {
          a[c] = mfma_16x16x32(pick.first, part[c], a[c]);
          b[c] = mfma_16x16x32(pick.second, part[c], b[c]);
        }
      };
      auto products = [&](f32x4_t& to_x, f32x4_t& to_z) {
#pragma unroll
        for (int c = 0; c < kSide; ++c) {
          to_x = mfma_16x16x32(kc[c], part[c], to_x);
          to_z = mfma_16x16x32(part[c], qc[c], to_z);
        }
      };
      auto next_part = [&] {
#pragma unroll
        for (int c = 0; c < kSide; ++c) part[c] = upper(a[c], b[c]);
      };
#pragma unroll
      for (int c = 0; c < kSide; ++c) {
        kc[c] = operand(k + (place ^ 32 * (h + c)));
        qc[c] = operand(q + (place ^ 32 * (h + c)));
        a[c] = s[2 * (h + c)];
        b[c] = s[2 * (h + c) + 1];
      }
      next_part();
      take_off();
      fence(); products(x, z);
      next_part();
      take_off();
      fence(); products(x_rest, z_rest);
      next_part();
      fence(); products(x_rest, z_rest);
    }
    x += x_rest;
    z += z_rest;
    if (of == 0) slot_barrier();
    const ShortSystem& sys = lds.systems[of];
    auto of_rows = [&](const float (&m)[kShortChunk]) { return *reinterpret_cast<const f32x4_t*>(&m[4 * g]); };
    const f32x4_t beta = of_rows(sys.beta), gamma = of_rows(sys.gamma), tail = of_rows(sys.tail), inv = sys.t[lane], pt = sys.p[lane];
    const float to_here = sys.gamma[x16], total = sys.gamma[kShortChunk - 1];
    f32x4_t r;
#pragma unroll
    for (int n = 0; n < 4; ++n) r[n] = beta[n] * __builtin_fmaf(-gamma[n], x[n], bf16_bits_to_f32(v[n]));
    if (of == 0 && first + kGroup * kShortChunk < end) fetch_group(j + kGroup);
    if (first + kShortChunk < end) load_v(first + kShortChunk);
    const f32x4_t u = mfma_f32_block(inv, r, zero);
    most = largest(u, largest(pt, most));
    // S = G S + K^T (tail U): U's bf16 parts, the first two side by side in one contraction
    auto rest = [](f32x4_t f) { return f - __builtin_bit_cast(f32x4_t, __builtin_bit_cast(u32x4_t, f) & 0xffff0000u); };
    const f32x4_t w = u * tail, w1 = rest(w), w2 = rest(w1);
    const u32x2_t hi = upper(w), mid = upper(w1), lo = upper(w2);
    const bf16x8_t small = as_bf16x8(u32x4_t{lo[0], lo[1], 0u, 0u}), large = as_bf16x8(u32x4_t{hi[0], hi[1], mid[0], mid[1]});
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const u32x2_t kt = lds_read_tr16(reinterpret_cast<const unsigned char*>(k + (transposed ^ 32 * (c >> 1)) + 4 * (c & 1)));
      const bf16x8_t both = as_bf16x8(u32x4_t{kt[0], kt[1], kt[0], kt[1]});
      const f32x4_t added = mfma_16x16x32(both, large, mfma_16x16x32(both, small, zero));
#pragma unroll
      for (int i = 0; i < 4; ++i) s[c][i] = __builtin_fmaf(s[c][i], total, added[i]);
    }
    const f32x4_t y = mfma_f32_block(u, pt, z * to_here);
    if (first + x16 < end)
      *reinterpret_cast<u32x2_t*>(y_chunk + y_at) = u32x2_t{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
    y_chunk += kShortChunk * (int64_t)y_step;
  }
  if (__builtin_expect(!__all(splits(most)), 0)) {
    token_by_token(start, end, slot, hv, row);
    return;
  }
  if constexpr (LINES) {
    float* const to = state_lines(slot, hv, row);
    exchange_lines(s);
#pragma unroll
    for (int c = 0; c < 8; ++c) __builtin_nontemporal_store(s[c], reinterpret_cast<f32x4_t*>(to + line_at(c)));
  } else {
#pragma unroll
    for (int c = 0; c < 8; ++c) *reinterpret_cast<f32x4_t*>(srow + 32 * (c >> 1) + 4 * (c & 1)) = s[c];
  }
}

}  // namespace

int launch_gdn_short(const GdnParams& p, hipStream_t stream) {
  const int64_t heads = (int64_t)p.batch * p.hv;
  if (2 * heads > 0x7fffffffLL) return MSGL_ERR_SHAPE;
  // Half a head to a workgroup while that leaves one to a compute unit, or two and there is one chunk (8 requests of 32 heads: 16 tokens
  // 10.4 us and 10.8 by whole heads, 32 tokens 12.9 and 11.7).
  const bool halves = 2 * heads <= device_cus() || (heads <= device_cus() && p.tokens <= kShortChunk * (int64_t)p.batch);
  // Whole lines past the caches from four requests of 32 heads on in one chunk, from eight beyond, but for 20 to 39 requests of more than 32
  // tokens: what the states of that many leave in the last level the next pass finds there, and the chunks' chain hides the rest.  That by
  // plain, three sets of states in turn (twelve, as the layers of a model), by requests, of up to 16 tokens, 17-32 and 33-48: 4 0.98-1.01 (0.97),
  // 1.04 (1.02), 1.06 (1.07); 6 0.94-0.97 (0.95), 0.99 (1.01), 1.01 (1.02); 8 0.88 (0.90), 0.95 (0.95), 0.97 (0.97); 16 0.87 (0.72), 0.95 (0.87),
  // 0.97 (0.92); 24 0.93 (0.83), 1.01 (0.90), 1.06 (0.98); 32 0.93 (0.82), 1.00 (0.87), 1.08 (0.98); 40 0.97 (0.89), 0.98 (0.89), 1.00 (0.99);
  // 64 0.96 (0.96), 0.93 (0.91), 0.97 (0.97); 100 0.95 (0.95), 0.93 (0.93), 0.93 (0.95).  One to three find their state in the caches.
  const bool one_chunk = p.tokens <= kShortChunk * (int64_t)p.batch, long_chain = p.tokens > 32 * (int64_t)p.batch;
  const bool lines = heads >= (one_chunk ? 128 : 256) && !(long_chain && heads >= 640 && heads < 1280);
  if (halves)
    return launch_kernel(lines ? gdn_short_kernel<4, true> : gdn_short_kernel<4, false>, dim3((unsigned)(2 * heads)), dim3(256), stream, p);
  return launch_kernel(lines ? gdn_short_kernel<8, true> : gdn_short_kernel<8, false>, dim3((unsigned)heads), dim3(512), stream, p);
}

}  // namespace msgl
