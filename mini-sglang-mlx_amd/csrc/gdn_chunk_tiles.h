// Pieces of the chunked gated delta rule that its kernels share (gdn_chunk.hip, gdn_long.hip): operands in three bf16
// parts, decay ratios, the inverse of a chunk's triangular system, the way through a request token after token.
#pragma once
#include <algorithm>

#include "gdn_params.h"
#include "prefill_tile_common.h"

namespace msgl {
namespace {

constexpr int kChunk = 64;        // tokens per chunk
constexpr int kRanked = 512;      // requests ranked by length (one per thread)

// T and P as operands: fragment f of row block m and contraction step c (32 columns), those that are not
// zero; lane x16 + 16 g of a fragment holds row x16, columns 32 c + 4 g .. and 32 c + 16 + 4 g ..
constexpr int kFragments = 6;
__device__ constexpr int fragment(int m, int c) { return c == 0 ? m : m + 2; }

// Piece `c` of 16 bytes of row `row` lies at this place.  LDS serves 8 lanes of a 16-byte read and 16 of an
// 8-byte one at a time: the rows 0-7 and 8-15 of an operand at one column go to 8 different places modulo 8,
// the 4 rows x 4 columns of a transposing read to 16 different ones.
__device__ __forceinline__ int swizzle(int row) {
  const int r0 = row & 1, r1 = (row >> 1) & 1, r2 = (row >> 2) & 1, r3 = (row >> 3) & 1;
  return (r1 ^ r3) << 3 | r0 << 2 | r1 << 1 | r2;
}
__device__ __forceinline__ int piece(int row, int c) { return c ^ swizzle(row); }

// Eight fp32 values as three operands of bf16 parts: x = hi + mid + lo, each the nearest to what is left, so
// exact.  The matrix pipe takes the parts off: x - hi is x plus the product of a matrix that picks, negated,
// the result tile's rows out of the 32 contraction rows, and hi as it stands (12 conversions and 4 matrix
// instructions; by vector instructions 44, and their issue is what a wave waits for).
struct Split {
  bf16x8_t hi, mid, lo;
};
struct Picker {
  bf16x8_t first, second;
  __device__ __forceinline__ Picker() {  // row 4 a + i of the first tile: contraction row 8 a + i; second: 8 a + 4 + i
    const int x16 = lane_id() & 15, g = lane_id() >> 4;
    u32x4_t f = {0u, 0u, 0u, 0u};
    const uint32_t minus_one = g == (x16 >> 2) ? 0xbf80u << (16 * (x16 & 1)) : 0u;
    const uint32_t even = (x16 & 2) ? 0u : minus_one, odd = (x16 & 2) ? minus_one : 0u;
    f[0] = even;
    f[1] = odd;
    first = as_bf16x8(f);
    second = as_bf16x8(u32x4_t{0u, 0u, even, odd});
  }
};
__device__ __forceinline__ bf16x8_t nearest(f32x4_t a, f32x4_t b) {
  return bf16x8_t{(__bf16)a[0], (__bf16)a[1], (__bf16)a[2], (__bf16)a[3], (__bf16)b[0], (__bf16)b[1], (__bf16)b[2], (__bf16)b[3]};
}
__device__ __forceinline__ Split split(const Picker& pick, f32x4_t a, f32x4_t b) {
  Split s;
  s.hi = nearest(a, b);
  a = mfma_16x16x32(pick.first, s.hi, a);
  b = mfma_16x16x32(pick.second, s.hi, b);
  s.mid = nearest(a, b);
  a = mfma_16x16x32(pick.first, s.mid, a);
  b = mfma_16x16x32(pick.second, s.mid, b);
  s.lo = nearest(a, b);
  return s;
}

// Four neighbouring values of a row of T or P, a lane's part of block (r, c), to LDS.
__device__ __forceinline__ void split_store(const Picker& pick, f32x4_t x, u32x4_t (*m)[kFragments][64], int r, int c) {
  auto half = [&](f32x4_t f) { return u32x2_t{pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3])}; };
  auto rest = [&](f32x4_t f, u32x2_t part) {
    return mfma_16x16x32(pick.first, as_bf16x8(u32x4_t{part[0], part[1], 0u, 0u}), f);
  };
  const u32x2_t hi = half(x);
  const f32x4_t y = rest(x, hi);
  const u32x2_t mid = half(y);
  const u32x2_t lo = half(rest(y, mid));
  u32x2_t* to = reinterpret_cast<u32x2_t*>(&m[0][fragment(r, c >> 1)][lane_id()]) + (c & 1);
  constexpr int kPart = kFragments * 64 * 2;
  to[0] = hi;
  to[kPart] = mid;
  to[2 * kPart] = lo;
}

// LDS traffic of every wave done, then the workgroup barrier; loads from memory stay in flight.
__device__ __forceinline__ void slot_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ bf16x8_t operand(const uint16_t* p) {
  return as_bf16x8(*reinterpret_cast<const u32x4_t*>(p));
}

struct Triangle {
  bf16x8_t hi[kFragments], mid[kFragments], lo[kFragments];
};
template <int FROM, int TO>
__device__ __forceinline__ void load_triangle(const u32x4_t (*m)[kFragments][64], Triangle& t) {
  const int lane = lane_id();
#pragma unroll
  for (int f = FROM; f < TO; ++f) {
    t.lo[f] = as_bf16x8(m[2][f][lane]);
    t.mid[f] = as_bf16x8(m[1][f][lane]);
    t.hi[f] = as_bf16x8(m[0][f][lane]);
  }
}
// a b, or its transpose: operands of both kinds have the same layout
template <bool TRANSPOSED>
__device__ __forceinline__ f32x4_t product(bf16x8_t a, bf16x8_t b, f32x4_t acc) {
  return TRANSPOSED ? mfma_16x16x32(b, a, acc) : mfma_16x16x32(a, b, acc);
}
// acc += M B for contraction step 0 of M, B split: the six products above 2^-24, smallest first, four rows
// of blocks side by side.
template <bool TRANSPOSED>
__device__ __forceinline__ void triangle_first(const Triangle& t, const Split& b, f32x4_t (&acc)[4]) {
  auto step = [&](const bf16x8_t (&part)[kFragments], const bf16x8_t& b0) {
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[m] = product<TRANSPOSED>(part[fragment(m, 0)], b0, acc[m]);
  };
  step(t.lo, b.hi);
  step(t.mid, b.mid);
  step(t.hi, b.lo);
  step(t.mid, b.hi);
  step(t.hi, b.mid);
  step(t.hi, b.hi);
}
// The same for step 1, which two rows of blocks reach: three products of each in a sum of their own.
template <bool TRANSPOSED>
__device__ __forceinline__ void triangle_second(const Triangle& t, const Split& b, f32x4_t (&acc)[4]) {
  f32x4_t x2 = {0.f, 0.f, 0.f, 0.f}, x3 = x2;
  auto step = [&](const bf16x8_t (&pa)[kFragments], const bf16x8_t& ba, const bf16x8_t (&pb)[kFragments], const bf16x8_t& bb) {
    x2 = product<TRANSPOSED>(pa[fragment(2, 1)], ba, x2);
    x3 = product<TRANSPOSED>(pa[fragment(3, 1)], ba, x3);
    acc[2] = product<TRANSPOSED>(pb[fragment(2, 1)], bb, acc[2]);
    acc[3] = product<TRANSPOSED>(pb[fragment(3, 1)], bb, acc[3]);
  };
  step(t.lo, b.hi, t.mid, b.hi);
  step(t.mid, b.mid, t.hi, b.mid);
  step(t.hi, b.lo, t.hi, b.hi);
  acc[2] += x2;
  acc[3] += x3;
}

__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }

// The larger of m and the magnitudes of x, NaN if there is one (two instructions).
__device__ __forceinline__ float largest(f32x4_t x, float m) {
  auto larger = [](float a, float b) { return __builtin_elementwise_maximum(a, b); };
  m = larger(larger(__builtin_fabsf(x[0]), __builtin_fabsf(x[1])), m);
  return larger(larger(__builtin_fabsf(x[2]), __builtin_fabsf(x[3])), m);
}
// Finite, and so is the nearest bf16.
__device__ __forceinline__ bool splits(float largest) { return largest < 0x1p127f; }

// A parameter of the launch (they are the kernel's first argument), read where it stands: what is only needed behind
// the chunks would push others out of the scalar registers meanwhile (2 % of a launch's time).
template <typename T>
__device__ __forceinline__ T parameter(T GdnParams::* member) {
  auto args = __builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(args));
  return ((const GdnParams*)args)->*member;
}
// Address of a lane's part of state row `row + lane % 16`: its four pieces of 8 dims lie 32 apart.
__device__ __forceinline__ float* state_row(int slot, int hv, int row) {
  uint32_t lane = lane_id();
  pin(lane);
  return parameter(&GdnParams::state) + (int64_t)slot * parameter(&GdnParams::state_stride0) +
         ((int64_t)hv * kDV + row + (lane & 15)) * kDK + 8 * (lane >> 4);
}

// A request token after token, as in gdn_state.hip, for a wave's 16 rows from `row` on.
__device__ __forceinline__ void token_by_token(int start, int end, int slot, int hv, int row) {
  GdnParams p;
  p.y = parameter(&GdnParams::y);
  p.q = parameter(&GdnParams::q);
  p.k = parameter(&GdnParams::k);
  p.v = parameter(&GdnParams::v);
  p.g = parameter(&GdnParams::g);
  p.beta = parameter(&GdnParams::beta);
  p.q_stride0 = parameter(&GdnParams::q_stride0);
  p.k_stride0 = parameter(&GdnParams::k_stride0);
  p.v_stride0 = parameter(&GdnParams::v_stride0);
  p.hv = parameter(&GdnParams::hv);
  p.hv_per_hk = parameter(&GdnParams::hv_per_hk);
  uint32_t lane = lane_id();
  pin(lane);
  const int g = lane >> 4, hk = hv / p.hv_per_hk;
  float* const srow = state_row(slot, hv, row);
  row += lane & 15;
  f32x4_t s[8];  // s[2 c + h][i]: dim 32 c + 8 g + 4 h + i
#pragma unroll
  for (int c = 0; c < 8; ++c) s[c] = *reinterpret_cast<const f32x4_t*>(srow + 32 * (c >> 1) + 4 * (c & 1));
  struct TokenIn {
    u32x4_t k[4], q[4];
    uint32_t g, beta, v;
  };
  auto load = [&](int64_t t, TokenIn& in) {
    const uint16_t* k = p.k + t * p.k_stride0 + hk * kDK + 8 * g;
    const uint16_t* q = p.q + t * p.q_stride0 + hk * kDK + 8 * g;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      in.k[c] = ld_global_b128(k + 32 * c);
      in.q[c] = ld_global_b128(q + 32 * c);
    }
    in.g = p.g[t * p.hv + hv];
    in.beta = p.beta[t * p.hv + hv];
    in.v = p.v[t * p.v_stride0 + hv * kDV + row];
  };
  auto four = [](u32x4_t raw, int h) {
    return f32x4_t{bf16_bits_to_f32(raw[2 * h] & 0xffffu), bf16_bits_to_f32(raw[2 * h] >> 16),
                   bf16_bits_to_f32(raw[2 * h + 1] & 0xffffu), bf16_bits_to_f32(raw[2 * h + 1] >> 16)};
  };
  TokenIn next;
  load(start, next);
  for (int t = start; t < end; ++t) {
    const TokenIn in = next;
    load(min(t + 1, end - 1), next);
    const float decay = bf16_bits_to_f32(in.g);
    float dot = 0.f, y = 0.f;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const f32x4_t k = four(in.k[c >> 1], c & 1);
      s[c] *= decay;
#pragma unroll
      for (int i = 0; i < 4; ++i) dot = __builtin_fmaf(s[c][i], k[i], dot);
    }
    const float delta = (bf16_bits_to_f32(in.v) - sum_across<32>(sum_across<16>(dot))) * bf16_bits_to_f32(in.beta);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const f32x4_t k = four(in.k[c >> 1], c & 1), q = four(in.q[c >> 1], c & 1);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[c][i] = __builtin_fmaf(k[i], delta, s[c][i]);
        y = __builtin_fmaf(s[c][i], q[i], y);
      }
    }
    y = sum_across<32>(sum_across<16>(y));
    if (g == 0) p.y[((int64_t)t * p.hv + hv) * kDV + row] = __builtin_bit_cast(uint16_t, (__bf16)y);
  }
#pragma unroll
  for (int c = 0; c < 8; ++c) *reinterpret_cast<f32x4_t*>(srow + 32 * (c >> 1) + 4 * (c & 1)) = s[c];
}

// Decay ratios G_t / G_i of block (r, c), transposed (lane: token t = 16 r + x16, tokens i = 16 c + 4 g + n).  Below the
// diagonal: token t's block up to it, whole blocks, token i's block behind it; on the diagonal: token t's quad up to
// it and the quads between, then token by token down the columns (1 above the diagonal).
struct Decays {
  f32x4_t col;
  float row;
  template <typename Lds>
  __device__ __forceinline__ void load(const Lds& lds, int r, int c) {
    const int x16 = lane_id() & 15, g = lane_id() >> 4;
    row = r == c ? lds.quad_pre[16 * r + x16] : lds.pre[16 * r + x16];
    col = *reinterpret_cast<const f32x4_t*>(r == c ? &lds.g[16 * r + 4 * g] : &lds.suf[16 * c + 4 * g]);
  }
  template <typename Lds>
  __device__ __forceinline__ f32x4_t below(const Lds& lds, int r, int c) const {
    const float b1 = lds.block[1], b2 = lds.block[2];
    return row * (c < 1 && r > 1 ? b1 : 1.0f) * (c < 2 && r > 2 ? b2 : 1.0f) * col;
  }
  template <typename Lds>
  __device__ __forceinline__ f32x4_t diagonal(const Lds& lds, int r) const {
    const int x16 = lane_id() & 15, g = lane_id() >> 4;
    const float q1 = lds.quad[4 * r + 1], q2 = lds.quad[4 * r + 2];
    const float far = row * (g < 1 && x16 >= 8 ? q1 : 1.0f) * (g < 2 && x16 >= 12 ? q2 : 1.0f);
    f32x4_t ratio;
    ratio[3] = (x16 >> 2) > g ? far : 1.0f;
#pragma unroll
    for (int i = 2; i >= 0; --i) ratio[i] = ratio[i + 1] * (4 * g + i + 1 <= x16 ? col[i + 1] : 1.0f);
    return ratio;
  }
};
// <k, q> or <k, k> of a block, transposed likewise
__device__ __forceinline__ f32x4_t block_dots(const bf16x8_t (&columns)[4], const bf16x8_t (&rows)[4]) {
  f32x4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int n = 0; n < 4; ++n) d = mfma_16x16x32(columns[n], rows[n], d);
  return d;
}
__device__ __forceinline__ void load_block_rows(const uint16_t (*m)[kDK], int r, bf16x8_t (&x)[4]) {
  const int x16 = lane_id() & 15, g = lane_id() >> 4;
#pragma unroll
  for (int d = 0; d < 4; ++d) x[d] = operand(&m[16 * r + x16][8 * piece(x16, 4 * d + g)]);
}

// Block (r, c) of A below the diagonal, to LDS; returns its ratios.
struct BelowBlock {
  bf16x8_t kc[4], kr[4];
  Decays decays;
  float beta;
  template <typename Lds>
  __device__ __forceinline__ void load(const Lds& lds, const uint16_t (*k)[kDK], const float* betas, int r, int c) {
    load_block_rows(k, c, kc);
    load_block_rows(k, r, kr);
    beta = betas[16 * r + (lane_id() & 15)];
    decays.load(lds, r, c);
  }
  template <typename Lds>
  __device__ __forceinline__ f32x4_t store(Lds& lds, int r, int c, f32x4_t dots) const {
    const f32x4_t ratio = decays.below(lds, r, c);
    *reinterpret_cast<f32x4_t*>(&lds.a[16 * r + (lane_id() & 15)][16 * c + 4 * (lane_id() >> 4)]) = beta * ratio * dots;
    return ratio;
  }
};

// Rows of Y from its transpose: a lane has of token 16 m + x16 the state rows 4 g ..
struct Outputs {
  uint32_t step, lane_at;
  int tokens;
  char* base;
  __device__ __forceinline__ Outputs(const GdnParams& p, int start, int end, int hv, int row)
      : step((uint32_t)p.hv * kDV * 2u), lane_at((lane_id() & 15) * step + 8 * (lane_id() >> 4)), tokens(end - start),
        base(reinterpret_cast<char*>(p.y + ((int64_t)start * p.hv + hv) * kDV + row)) {}
  __device__ __forceinline__ void store(int chunk, const f32x4_t (&z)[4]) const {
    char* to = base + (int64_t)chunk * kChunk * step;
    const int left = tokens - chunk * kChunk;
    auto one = [&](int m) {
      *reinterpret_cast<u32x2_t*>(to + (lane_at + 16 * m * step)) = u32x2_t{pack_bf16x2(z[m][0], z[m][1]), pack_bf16x2(z[m][2], z[m][3])};
    };
    if (left >= kChunk) {
#pragma unroll
      for (int m = 0; m < 4; ++m) one(m);
    } else {
#pragma unroll
      for (int m = 0; m < 4; ++m)
        if (16 * m + (lane_id() & 15) < left) one(m);
    }
  }
};

// A value from another lane of the row of 16, 1 where there is none.  DPP control C: 0x110 + n the lane n below,
// 0x100 + n the lane n above.
template <int C>
__device__ __forceinline__ float row_shift(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0x3f800000, __builtin_bit_cast(int, x), C, 0xf, 0xf, false));
}
// Inverse of I + A for a 16 x 16 block: lane x16 holds row x16 of the strictly lower -A and, of the inverse,
// columns 4 g .. 4 g + 3 of that row.  Row T is final when its turn comes and is taken off the rows below it.
template <int T>
__device__ __forceinline__ void eliminate(const float (&minus_a)[16], f32x4_t& inv) {
  // the row and its multiplication in one instruction each (left to the compiler two, one behind the other); a value is read by
  // DPP two instructions after it is written at the earliest
  float a = inv[0], b = inv[1], c = inv[2], d = inv[3];
  asm("s_nop 1\n\t"
      "v_fmac_f32_dpp %0, %0, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %1, %1, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %2, %2, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %3, %3, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
      : "+v"(a), "+v"(b), "+v"(c), "+v"(d)
      : "v"(minus_a[T]), "n"(T));
  inv = f32x4_t{a, b, c, d};
  if constexpr (T < 14) eliminate<T + 1>(minus_a, inv);
}

__device__ __forceinline__ f32x4_t mfma_f32_block(f32x4_t a, f32x4_t b, f32x4_t c) {
  // 16x16x16 in four steps: step i contracts over 4 g + i, which a lane's four values of a row
  // (A operand) and four result rows of a column (B operand) are
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
  return c;
}

// Blocks (R, C) of T below the diagonal from those of A and the inverses on the diagonal:
// T_RC = -T_RR X_R, X_R = sum over C <= k < R of A_Rk T_kC.  A block is made as the operand of the rows below it
// and transposed, four neighbours of a row to a lane, for LDS (T_RC^T = -X_R^T T_RR^T).  Operands of that:
template <typename Lds>
struct Inverse {
  const Lds& lds;
  int x16, g;
  __device__ __forceinline__ explicit Inverse(const Lds& l) : lds(l), x16(lane_id() & 15), g(lane_id() >> 4) {}
  __device__ __forceinline__ f32x4_t a(int r, int k) const { return *reinterpret_cast<const f32x4_t*>(lds.a_row(r, k, x16) + 4 * g); }
  __device__ __forceinline__ f32x4_t minus_diag(int r) const { return -*reinterpret_cast<const f32x4_t*>(lds.diagonal_row(r, x16) + 4 * g); }
  __device__ __forceinline__ f32x4_t diag_plain(int r) const {
    f32x4_t d;
#pragma unroll
    for (int n = 0; n < 4; ++n) d[n] = lds.diagonal_row(r, 4 * g + n)[x16];
    return d;
  }
};

// Decay products of a chunk, a token per lane (1 and beta 0 past the request's end).
template <typename Lds>
__device__ __forceinline__ void decay_products(Lds& lds, float gv, float bv, float* beta, float* gamma, float* tail, float& total) {
  const int lane = lane_id(), x16 = lane & 15, g = lane >> 4;
  // products over a row of 16 lanes, or over quads (every lane shifts, then takes what is in its quad)
  const float before1 = row_shift<0x111>(gv);
  float pre = gv * before1, suf = gv * row_shift<0x101>(gv), quad_pre = gv * ((x16 & 3) >= 1 ? before1 : 1.0f);
  const float quad2 = row_shift<0x112>(quad_pre);
  quad_pre *= (x16 & 3) >= 2 ? quad2 : 1.0f;
  pre *= row_shift<0x112>(pre);
  suf *= row_shift<0x102>(suf);
  pre *= row_shift<0x114>(pre);
  suf *= row_shift<0x104>(suf);
  pre *= row_shift<0x118>(pre);
  suf *= row_shift<0x108>(suf);
  suf = row_shift<0x101>(suf);  // behind the token
  auto lane_value = [](float f, int l) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f), l));
  };
  const float b0 = lane_value(pre, 15), b1 = lane_value(pre, 31), b2 = lane_value(pre, 47), b3 = lane_value(pre, 63);
  const float before = g == 0 ? 1.0f : g == 1 ? b0 : g == 2 ? b0 * b1 : b0 * b1 * b2;
  const float behind = g == 3 ? 1.0f : g == 2 ? b3 : g == 1 ? b2 * b3 : b1 * b2 * b3;
  beta[lane] = bv;
  gamma[lane] = before * pre;
  tail[lane] = suf * behind;
  lds.g[lane] = gv;
  lds.pre[lane] = pre;
  lds.suf[lane] = suf;
  lds.quad_pre[lane] = quad_pre;
  if (x16 == 15) lds.block[g] = pre;
  if ((lane & 3) == 3) lds.quad[lane >> 2] = quad_pre;
  if (lane == 0) total = b0 * b1 * b2 * b3;
}

// Blocks of T below the diagonal, two waves with the first column: (1, 0) and (2, 0); (2, 1) and (3, 1); (3, 2);
// (3, 0).  Everything a chain needs from LDS is asked for before it starts.
struct Below {
  f32x4_t first, second;
};
template <bool LAST_LATER, typename Lds>
__device__ __forceinline__ Below blocks_below(const Lds& lds, int w) {
  const Inverse<Lds> of(lds);
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  if (w == 2) {
    const f32x4_t a32 = of.a(3, 2), t2 = of.diag_plain(2), d3 = of.minus_diag(3);
    return {mfma_f32_block(mfma_f32_block(a32, t2, zero), d3, zero), zero};
  }
  if (w == 1) {
    const f32x4_t a21 = of.a(2, 1), a31 = of.a(3, 1), a32 = of.a(3, 2), t1 = of.diag_plain(1), d2 = of.minus_diag(2), d3 = of.minus_diag(3);
    const f32x4_t x2 = mfma_f32_block(a21, t1, zero);
    f32x4_t x3 = mfma_f32_block(a31, t1, zero);
    const f32x4_t t21 = mfma_f32_block(d2, x2, zero);
    const f32x4_t first = mfma_f32_block(x2, d2, zero);
    x3 = mfma_f32_block(a32, t21, x3);
    return {first, mfma_f32_block(x3, d3, zero)};
  }
  const f32x4_t a10 = of.a(1, 0), a20 = of.a(2, 0), a21 = of.a(2, 1), t0 = of.diag_plain(0), d1 = of.minus_diag(1), d2 = of.minus_diag(2);
  if (w == 0) {
    const f32x4_t x1 = mfma_f32_block(a10, t0, zero);
    f32x4_t x2 = mfma_f32_block(a20, t0, zero);
    const f32x4_t t10 = mfma_f32_block(d1, x1, zero);
    const f32x4_t first = mfma_f32_block(x1, d1, zero);
    x2 = mfma_f32_block(a21, t10, x2);
    return {first, mfma_f32_block(x2, d2, zero)};
  }
  const f32x4_t a30 = of.a(3, 0), a31 = of.a(3, 1), a32 = of.a(3, 2), d3 = of.minus_diag(3);
  const f32x4_t x1 = mfma_f32_block(a10, t0, zero);
  f32x4_t x2 = mfma_f32_block(a20, t0, zero), x3 = mfma_f32_block(a30, t0, zero);
  const f32x4_t t10 = mfma_f32_block(d1, x1, zero);
  x2 = mfma_f32_block(a21, t10, x2);
  x3 = mfma_f32_block(a31, t10, x3);
  const f32x4_t t20 = mfma_f32_block(d2, x2, zero);
  x3 = mfma_f32_block(a32, t20, x3);
  if constexpr (LAST_LATER) return {x3, d3};  // this chain is the longest: its last product is left to the caller
  else return {mfma_f32_block(x3, d3, zero), zero};
}

}  // namespace
}  // namespace msgl
