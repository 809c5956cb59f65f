// Gated delta rule over many tokens per request: chunks of 64 tokens on the matrix cores.
//
// The recurrence of gdn_state.hip (one state row dv of a head, tokens t = 1 .. 64 of a chunk, S the
// state before the chunk, G_t the product of the decays g_1 .. g_t):
//     u_t = beta_t (v_t - G_t <S, k_t> - sum_{i<t} (G_t / G_i) <k_i, k_t> u_i)
//     y_t = G_t <S, q_t> + sum_{i<=t} (G_t / G_i) <k_i, q_t> u_i
//     S'  = G_64 S + sum_i (G_64 / G_i) u_i k_i
// is, for all rows of a head at once, a triangular system (I + A) U = beta (V - G K S^T) with
// A[t][i] = beta_t (G_t / G_i) <k_i, k_t>, i < t: the chunkwise form of the delta rule (Yang et al.,
// "Parallelizing Linear Transformers with the Delta Rule over Sequence Length", 2024, with decays as in
// "Gated Delta Networks", 2024).  T = (I + A)^-1 and P[t][i] = (G_t / G_i) <k_i, q_t> do not depend on
// the state, so the serial part of a chunk is five products.
//
// Token after token a request costs 0.33 us per token whatever the chip has free; here a chunk of 64 costs
// 4.4 us.  Requests of 992, 1581, 4005 and 1601 tokens at hk 16, hv 32: 1353 -> 287 us; one of 1024: 298 -> 78.
//
// Work: one workgroup per (request, value head, half of its 128 rows).  Waves 0-3 ("state" waves, 16
// rows each, S^T in 32 accumulator registers) run the serial part of chunk j; waves 4-7 ("chunk" waves,
// 16 tokens each) make T and P of chunk j + 1 beside them, one of each on a SIMD.  Three slots per
// chunk, a workgroup barrier behind each:
//     slot   state waves, chunk j                 chunk waves
//      1     X = K S^T, Z = Q S^T                  T and P of chunk j and K, Q of chunk j + 1 to LDS
//      2     R = beta (V - G X), U = T R           A, the decay ratios of P, the diagonal blocks of T of chunk j + 1
//      3     Y = G Z + P U, S = G_64 S + K^T U     P, the blocks of T below the diagonal, V of chunk j + 1;
//                                                  decay products of chunk j + 2
// What bounds it: a chunk takes 10.6 K cycles (slots of 3.3, 2.9 and 4.4 K), in which a SIMD has 5.3 K cycles of
// matrix instructions and as many of vector instructions in two chains that wait for their own results, and a
// wave that has the SIMD for itself still pays about 5 cycles per instruction of any kind.  The last wave of a slot is
// a chunk wave in all three, 0.6 K, 0.4 K and 0.5 K cycles behind the slowest state wave.  Hence: fp32 values
// are split by the matrix pipe (see Split: 16 instructions instead of 44), Z and Y are made transposed (4 stores
// of 8 bytes a chunk instead of 16 of 2), V comes by transposing LDS reads, and the chunk waves share the blocks
// out evenly (12.5 -> 10.7 K).  T and P of all chunks in a launch of their own, in parallel, measured the same
// for the longest request of a launch and less for many short ones: their 20 KB per chunk and head cost 40 us
// of writing for the requests above, and LDS and issue time in the serial part.
//
// Precision: fp32 throughout, as in the token kernel.  q, k, v are bf16 and enter the bf16 matrix
// instructions as they are; fp32 operands (S, R, U, T, P) are split into three bf16 parts of 8
// significant bits each, which hold all 24, and multiplied part by part into fp32 accumulators (for
// two split operands the six products above 2^-24 of the result).  The inverse is built from fp32
// matrix instructions.  Decay ratios are products of the decays (no logarithms: a decay may be 0).
//
// Infinities and NaN: the products above run over a whole chunk, zeros of a triangle included, and would carry
// 0 * infinity from a token to the ones before it and from a dim to the others.  So every wave keeps the largest
// magnitude of its U (not finite if v, k, a gate or the state is not, or if T overflowed) and of P on the diagonal
// (not finite if a query is not), and if that is not finite in the end, goes through the request again from the
// state it started with, token by token: what the token kernel gives.  Keeping it costs 0.7 % (286 -> 288 us for the
// requests above); the second pass takes 0.6 us a token (one request of 4005: 0.29 -> 2.8 ms).
//
// Layouts (v_mfma 16x16x32: lane l holds row / column l % 16 and the 8 contraction values of lane group
// g = l / 16; results: column l % 16, rows 4 g + i).  A result used as an operand of the next product
// keeps its registers: the contraction order is permuted to match instead, i.e. lane group g
// contracts over rows 4 g + i of two neighbouring result tiles.  For tokens the columns of T and P are
// stored in that order; for S^T the transposing LDS reads of K (4 tokens x 16 dims) pick their dims so
// that result tile 2 s + h holds dims 32 s + 8 g + 4 h + i, which makes the pair (2 s, 2 s + 1) of a lane
// 8 consecutive dims, the natural order of K and Q.
#include "gdn_params.h"
#include "prefill_tile_common.h"

namespace msgl {
namespace {

constexpr int kChunk = 64;        // tokens per chunk
constexpr int kRowsPerWg = 64;    // dv rows of a workgroup
constexpr int kRanked = 512;      // requests ranked by length (one per thread)

// T and P as operands: fragment f of row block m and contraction step c (32 columns), those that are not
// zero; lane x16 + 16 g of a fragment holds row x16, columns 32 c + 4 g .. and 32 c + 16 + 4 g ..
constexpr int kFragments = 6;
__device__ constexpr int fragment(int m, int c) { return c == 0 ? m : m + 2; }

struct ChunkLds {
  uint16_t k[2][kChunk][kDK], q[2][kChunk][kDK];  // 16-byte pieces of a row in swizzled order (see piece())
  uint16_t v[kChunk][kRowsPerWg];
  u32x4_t t[3][kFragments][64], p[3][kFragments][64];  // T and P in three bf16 parts
  float a[kChunk][68];            // A of the chunk being prepared (blocks on and below the diagonal)
  float diag[4][16][20];          // inverses of the diagonal blocks of I + A
  // per token, chunks j .. j + 2: beta, G, and tail_i = G_64 / G_i
  float beta[3][kChunk], gamma[3][kChunk], tail[3][kChunk];
  // of the chunk being prepared: the decays; products over the block of 16 up to a token, behind it, and
  // over its quad up to it; products over whole blocks and over the quads of each block
  float g[kChunk], pre[kChunk], suf[kChunk], quad_pre[kChunk], block[4], quad[16];
  float total[3];                 // G_64, chunks j .. j + 2 (last: the arrays above are read 16 bytes at a time)
  int request;
  alignas(16) float p_largest[4 * 64];  // per lane of the chunk waves: largest() of P's diagonal blocks, all chunks
};

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

__device__ __forceinline__ void state_waves(const GdnParams& p, ChunkLds& lds, int start, int end, int slot, int hv,
                                            int row, int column) {
  const int lane = lane_id(), x16 = lane & 15, g = lane >> 4;
  const int n_chunks = (end - start + kChunk - 1) / kChunk;
  f32x4_t s[8];  // s[2 c + h][i]: dim 32 c + 8 g + 4 h + i of row `row + x16`
  float* srow = state_row(slot, hv, row);
#pragma unroll
  for (int c = 0; c < 8; ++c) s[c] = *reinterpret_cast<const f32x4_t*>(srow + 32 * (c >> 1) + 4 * (c & 1));

  // a lane's part of Y: of token 16 m + x16 the rows 4 g ..
  const uint32_t y_step = (uint32_t)p.hv * kDV * 2u, y_lane = x16 * y_step + 8 * g;
  char* ybase = reinterpret_cast<char*>(p.y + ((int64_t)start * p.hv + hv) * kDV + row);
  const Picker pick;
  // places of K's and Q's pieces in LDS: as operands, row x16, and transposed, row `trow`, per 32 dims
  const int trow = 4 * g + (x16 >> 2);
  uint32_t at[4], kt_at[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    at[c] = x16 * kDK + 8 * piece(x16, 4 * c + g);
    kt_at[c] = trow * kDK + 8 * piece(trow, 4 * c + (x16 & 3));
  }
  struct Rows {
    bf16x8_t k[4], q[4];
  };
  auto load_rows = [&](int par, int c, Rows& r) {
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      r.k[m] = operand(&lds.k[par][16 * m][0] + at[c]);
      r.q[m] = operand(&lds.q[par][16 * m][0] + at[c]);
    }
  };
  __builtin_amdgcn_s_setprio(1);  // before the chunk waves, but in slot 2, where those have the longer way
  slot_barrier();  // K, Q of chunk 0
  slot_barrier();  // A of chunk 0
  slot_barrier();  // what T of chunk 0 is made of

  Rows rows[2];
  load_rows(0, 0, rows[0]);
  Split sp = split(pick, s[0], s[1]);
  float most = 0.f;  // largest() of every U
  for (int j = 0, tri = 0; j < n_chunks; ++j, tri = tri == 2 ? 0 : tri + 1) {
    const int par = j & 1;
    // ---- slot 1 ----------------------------------------------------------------------------
    f32x4_t x[4], z[4];  // X, and Z transposed: a lane's four values are neighbours in a row of Y
#pragma unroll
    for (int m = 0; m < 4; ++m) x[m] = z[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (c < 3) load_rows(par, c + 1, rows[(c + 1) & 1]);
      fence();
      const Rows& r = rows[c & 1];
      auto step = [&](bf16x8_t part) {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          x[m] = product<false>(r.k[m], part, x[m]);
          z[m] = product<true>(r.q[m], part, z[m]);
        }
      };
      const Split now = sp;
      step(now.lo);
      if (c < 3) sp = split(pick, s[2 * c + 2], s[2 * c + 3]);
      step(now.mid);
      step(now.hi);
      fence();
    }
    slot_barrier();
    // ---- slot 2 ----------------------------------------------------------------------------
    Triangle tp;
    load_triangle<0, 4>(lds.t, tp);
    f32x4_t u[4];
    {
      f32x4_t r[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const f32x4_t bet = *reinterpret_cast<const f32x4_t*>(&lds.beta[tri][16 * m + 4 * g]);
        const f32x4_t gam = *reinterpret_cast<const f32x4_t*>(&lds.gamma[tri][16 * m + 4 * g]);
        const u32x2_t v = lds_read_tr16(reinterpret_cast<const unsigned char*>(&lds.v[16 * m + trow][column + 4 * (x16 & 3)]));
#pragma unroll
        for (int i = 0; i < 4; ++i)
          r[m][i] = (bf16_bits_to_f32(i & 1 ? v[i >> 1] >> 16 : v[i >> 1] & 0xffffu) - gam[i] * x[m][i]) * bet[i];
        u[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
      load_triangle<4, 6>(lds.t, tp);
      const Split rs0 = split(pick, r[0], r[1]);
      const Split rs1 = split(pick, r[2], r[3]);
      triangle_first<false>(tp, rs0, u);
      triangle_second<false>(tp, rs1, u);
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) z[m] *= lds.gamma[tri][16 * m + x16];
    fence();
    load_triangle<0, 4>(lds.p, tp);
    slot_barrier();
    // ---- slot 3 ----------------------------------------------------------------------------
    const uint16_t* k = &lds.k[par][0][0];
    auto load_kt = [&](int n, bf16x8_t (&ka)[4]) {  // K transposed: tokens 32 (n % 2) .., dims 64 (n / 2) ..
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = 4 * (n >> 1) + i;
        const uint16_t* a = k + kt_at[c >> 1] + 4 * (c & 1) + 32 * (n & 1) * kDK;
        const u32x2_t a0 = lds_read_tr16(reinterpret_cast<const unsigned char*>(a));
        const u32x2_t a1 = lds_read_tr16(reinterpret_cast<const unsigned char*>(a + 16 * kDK));
        ka[i] = as_bf16x8(u32x4_t{a0[0], a0[1], a1[0], a1[1]});
      }
    };
    bf16x8_t ka[2][4];
    f32x4_t tail[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) tail[m] = *reinterpret_cast<const f32x4_t*>(&lds.tail[tri][16 * m + 4 * g]);
    const float total = lds.total[tri];
    load_triangle<4, 6>(lds.p, tp);
    load_kt(0, ka[0]);
    load_kt(1, ka[1]);
    const Split us0 = split(pick, u[0], u[1]);
    const Split us1 = split(pick, u[2], u[3]);
    fence();
    triangle_first<true>(tp, us0, z);
    const Split ut0 = split(pick, u[0] * tail[0], u[1] * tail[1]);
    const Split ut1 = split(pick, u[2] * tail[2], u[3] * tail[3]);
#pragma unroll
    for (int c = 0; c < 8; ++c) s[c] *= total;
#pragma unroll
    for (int m = 0; m < 4; ++m) most = largest(u[m], most);
    fence();
    triangle_second<true>(tp, us1, z);
    auto steps = [&](int n, const Split& b) {
      auto step = [&](bf16x8_t part) {
#pragma unroll
        for (int i = 0; i < 4; ++i) s[4 * (n >> 1) + i] = mfma_16x16x32(ka[n & 1][i], part, s[4 * (n >> 1) + i]);
      };
      step(b.lo);
      step(b.mid);
      step(b.hi);
    };
    steps(0, ut0);
    fence();
    load_kt(2, ka[0]);
    steps(1, ut1);
    fence();
    load_kt(3, ka[1]);
    steps(2, ut0);
    char* to = ybase + (int64_t)j * kChunk * y_step;
    const int left = end - start - j * kChunk;
    auto store = [&](int m) {
      *reinterpret_cast<u32x2_t*>(to + (y_lane + 16 * m * y_step)) = u32x2_t{pack_bf16x2(z[m][0], z[m][1]), pack_bf16x2(z[m][2], z[m][3])};
    };
    if (left >= kChunk) {
#pragma unroll
      for (int m = 0; m < 4; ++m) store(m);
    } else {
#pragma unroll
      for (int m = 0; m < 4; ++m)
        if (16 * m + x16 < left) store(m);
    }
    fence();
    load_rows(par ^ 1, 0, rows[0]);  // of chunk j + 1 (of no use behind the last chunk)
    steps(3, ut1);
    sp = split(pick, s[0], s[1]);
    slot_barrier();
  }
  most = largest(*reinterpret_cast<const f32x4_t*>(&lds.p_largest[4 * lane]), most);
  if (__builtin_expect(!__all(splits(most)), 0)) {
    wait_all_vm();  // the stores of Y: the same places are written again
    token_by_token(start, end, slot, hv, row);
    return;
  }
  srow = state_row(slot, hv, row);
#pragma unroll
  for (int c = 0; c < 8; ++c) *reinterpret_cast<f32x4_t*>(srow + 32 * (c >> 1) + 4 * (c & 1)) = s[c];
}

// A value from another lane of the row of 16, 1 where there is none.  DPP control C: 0x110 + n the lane n below,
// 0x100 + n the lane n above.
template <int C>
__device__ __forceinline__ float row_shift(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0x3f800000, __builtin_bit_cast(int, x), C, 0xf, 0xf, false));
}
// Lane t of every row of 16 lanes, in all of them.
template <int T>
__device__ __forceinline__ float row_broadcast(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x150 + T, 0xf, 0xf, true));
}
// Inverse of I + A for a 16 x 16 block: lane x16 holds row x16 of the strictly lower A and, of the inverse,
// columns 4 g .. 4 g + 3 of that row.  Row T is final when its turn comes and is taken off the rows below it.
template <int T>
__device__ __forceinline__ void eliminate(const float (&a)[16], f32x4_t& inv) {
#pragma unroll
  for (int n = 0; n < 4; ++n) inv[n] = __builtin_fmaf(-a[T], row_broadcast<T>(inv[n]), inv[n]);
  if constexpr (T < 14) eliminate<T + 1>(a, inv);
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
struct Inverse {
  const ChunkLds& lds;
  int x16, g;
  __device__ __forceinline__ explicit Inverse(const ChunkLds& l) : lds(l), x16(lane_id() & 15), g(lane_id() >> 4) {}
  __device__ __forceinline__ f32x4_t a(int r, int k) const { return *reinterpret_cast<const f32x4_t*>(&lds.a[16 * r + x16][16 * k + 4 * g]); }
  __device__ __forceinline__ f32x4_t minus_diag(int r) const { return -*reinterpret_cast<const f32x4_t*>(&lds.diag[r][x16][4 * g]); }
  __device__ __forceinline__ f32x4_t diag_plain(int r) const {
    f32x4_t d;
#pragma unroll
    for (int n = 0; n < 4; ++n) d[n] = lds.diag[r][4 * g + n][x16];
    return d;
  }
};

__device__ __forceinline__ void chunk_waves(const GdnParams& p, ChunkLds& lds, int start, int end, int hv,
                                            int wg_row, int w) {
  const int lane = lane_id(), x16 = lane & 15, g = lane >> 4;
  const Picker pick;
  const int n_chunks = (end - start + kChunk - 1) / kChunk;
  const int hk = hv / p.hv_per_hk;
  // this wave's 16 tokens of K and Q, four rows per load, and every token's gates: scalar bases at the
  // request's first token, 32-bit offsets
  const char* kbase = reinterpret_cast<const char*>(p.k + (int64_t)start * p.k_stride0 + hk * kDK);
  const char* qbase = reinterpret_cast<const char*>(p.q + (int64_t)start * p.q_stride0 + hk * kDK);
  const char* gbase = reinterpret_cast<const char*>(p.g + (int64_t)start * p.hv + hv);
  const char* bbase = reinterpret_cast<const char*>(p.beta + (int64_t)start * p.hv + hv);
  const uint32_t k_step = (uint32_t)p.k_stride0 * 2u, q_step = (uint32_t)p.q_stride0 * 2u, g_step = (uint32_t)p.hv * 2u;
  // V of the workgroup's rows, 8 tokens a load, straight to LDS; rows past the request's end: the last row
  // (beta is zero there)
  const char* vbase = reinterpret_cast<const char*>(p.v + (int64_t)start * p.v_stride0 + hv * kDV + wg_row);
  const uint32_t v_step = (uint32_t)p.v_stride0 * 2u, v_lds = (uint32_t)(uintptr_t)MSGL_LDS_PTR(uint16_t, &lds.v[16 * w][0]);
  auto fetch_v = [&](int first) {
    const char* base = vbase + (int64_t)(first - start) * v_step;
#pragma unroll
    for (int n = 0; n < 2; ++n)
      lds_direct_b128(__builtin_amdgcn_readfirstlane(v_lds + 1024 * n), base,
                      min((uint32_t)(16 * w + 8 * n + (lane >> 3)), (uint32_t)(end - 1 - first)) * v_step + 16 * (lane & 7));
  };
  u32x4_t kr[4], qr[4];
  uint32_t graw, braw;
  auto fetch = [&](int first) {
    const char* kb = kbase + (int64_t)(first - start) * k_step;
    const char* qb = qbase + (int64_t)(first - start) * q_step;
    const uint32_t last = end - 1 - first;
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const uint32_t t = min((uint32_t)(16 * w + 4 * n + g), last);
      kr[n] = ld_global_b128(kb + (t * k_step + 16 * x16));
      qr[n] = ld_global_b128(qb + (t * q_step + 16 * x16));
    }
    const uint32_t t = min((uint32_t)lane, last) * g_step;
    graw = *reinterpret_cast<const uint16_t*>(gbase + (int64_t)(first - start) * g_step + t);
    braw = *reinterpret_cast<const uint16_t*>(bbase + (int64_t)(first - start) * g_step + t);
  };
  auto stage = [&](int first, int par) {  // rows past the request's end are zero
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const int t = 16 * w + 4 * n + g;
      const u32x4_t zero = {0u, 0u, 0u, 0u};
      const bool in = first + t < end;
      *reinterpret_cast<u32x4_t*>(&lds.k[par][t][8 * piece(t, x16)]) = in ? kr[n] : zero;
      *reinterpret_cast<u32x4_t*>(&lds.q[par][t][8 * piece(t, x16)]) = in ? qr[n] : zero;
    }
  };
  // decay products of a chunk from the gates fetched with it: the last wave's work, it has the least to do
  // beside T
  auto decays = [&](int first, int tri) {
    const bool in = first + lane < end;
    const float gv = in ? bf16_bits_to_f32(graw) : 1.0f, bv = in ? bf16_bits_to_f32(braw) : 0.0f;
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
    lds.beta[tri][lane] = bv;
    lds.gamma[tri][lane] = before * pre;
    lds.tail[tri][lane] = suf * behind;
    lds.g[lane] = gv;
    lds.pre[lane] = pre;
    lds.suf[lane] = suf;
    lds.quad_pre[lane] = quad_pre;
    if (x16 == 15) lds.block[g] = pre;
    if ((lane & 3) == 3) lds.quad[lane >> 2] = quad_pre;
    if (lane == 0) lds.total[tri] = b0 * b1 * b2 * b3;
  };
  // The ten blocks (r, c) of A and P on and below the diagonal: every wave its diagonal block and one
  // more, waves 1 and 2 two.  Results are transposed (lane: token t = 16 r + x16, tokens i = 16 c + 4 g + n), so that a
  // lane's four values are neighbours in a row of A and of P.
  const int n_blocks = w == 0 || w == 3 ? 2 : 3;
  auto block_row = [&](int n) { return n == 0 ? w : n == 1 ? (w == 0 ? 3 : w) : (w == 2 ? 2 : 3); };
  auto block_col = [&](int n) { return n == 0 ? w : n == 1 ? (w == 3 ? 1 : 0) : (w == 1 ? 2 : 1); };
  f32x4_t pp[3];  // the ratios of P of these blocks, then P
  float most = 0.f;  // largest() of P's diagonal block, every chunk
  f32x4_t inv;    // the inverse of the diagonal block: row x16, columns 4 g ..
  auto products = [&](int par, int tri) {
    struct Block {
      bf16x8_t kc[4], kr[4];
      f32x4_t col;
      float row, beta;
    };
    auto load = [&](int r, int c, Block& x) {
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        x.kc[d] = operand(&lds.k[par][16 * c + x16][8 * piece(x16, 4 * d + g)]);
        x.kr[d] = operand(&lds.k[par][16 * r + x16][8 * piece(x16, 4 * d + g)]);
      }
      x.beta = lds.beta[tri][16 * r + x16];
      x.row = r == c ? lds.quad_pre[16 * r + x16] : lds.pre[16 * r + x16];
      x.col = *reinterpret_cast<const f32x4_t*>(r == c ? &lds.g[16 * r + 4 * g] : &lds.suf[16 * c + 4 * g]);
    };
    auto dots = [&](const Block& x) {
      f32x4_t kk = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < 4; ++d) kk = mfma_16x16x32(x.kc[d], x.kr[d], kk);
      return kk;
    };
    // G_t / G_i of a block below the diagonal: token t's block up to it, whole blocks, token i's block behind it
    auto below_block = [&](int n, int r, int c, const Block& x, const f32x4_t& kk) {
      float row = x.row;
      if (c < 1 && r > 1) row *= lds.block[1];
      if (c < 2 && r > 2) row *= lds.block[2];
      const f32x4_t ratio = row * x.col;
      pp[n] = ratio;
      *reinterpret_cast<f32x4_t*>(&lds.a[16 * r + x16][16 * c + 4 * g]) = x.beta * ratio * kk;
    };
    Block b0, b1, b2;
    const int r1 = block_row(1), c1 = block_col(1), r2 = block_row(2), c2 = block_col(2);
    load(w, w, b0);
    load(r1, c1, b1);
    const f32x4_t kk0 = dots(b0);
    {
      // on the diagonal: token t's quad up to it and the quads between, then token by token down the columns
      float far = b0.row;
      if (g < 1 && x16 >= 8) far *= lds.quad[4 * w + 1];
      if (g < 2 && x16 >= 12) far *= lds.quad[4 * w + 2];
      f32x4_t ratio, a;
      ratio[3] = (x16 >> 2) > g ? far : 1.0f;
#pragma unroll
      for (int i = 2; i >= 0; --i) ratio[i] = ratio[i + 1] * (4 * g + i + 1 <= x16 ? b0.col[i + 1] : 1.0f);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i] = 4 * g + i < x16 ? b0.beta * ratio[i] * kk0[i] : 0.f;
        pp[0][i] = 4 * g + i <= x16 ? ratio[i] : 0.f;
      }
      *reinterpret_cast<f32x4_t*>(&lds.a[16 * w + x16][16 * w + 4 * g]) = a;
    }
    float arow[16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4_t a = *reinterpret_cast<const f32x4_t*>(&lds.a[16 * w + x16][16 * w + 4 * i]);
#pragma unroll
      for (int e = 0; e < 4; ++e) arow[4 * i + e] = a[e];
    }
#pragma unroll
    for (int n = 0; n < 4; ++n) inv[n] = x16 == 4 * g + n ? 1.0f : 0.0f;
    if (n_blocks > 2) {
      load(r2, c2, b2);
      const f32x4_t kk1 = dots(b1), kk2 = dots(b2);
      eliminate<0>(arow, inv);
      below_block(1, r1, c1, b1, kk1);
      below_block(2, r2, c2, b2, kk2);
    } else {
      const f32x4_t kk1 = dots(b1);
      eliminate<0>(arow, inv);
      below_block(1, r1, c1, b1, kk1);
    }
    *reinterpret_cast<f32x4_t*>(&lds.diag[w][x16][4 * g]) = inv;
  };
  auto finish_p = [&](int par) {  // P = ratios times <k, q>
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      if (n >= n_blocks) break;
      f32x4_t qk = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < 4; ++d)
        qk = mfma_16x16x32(operand(&lds.k[par][16 * block_col(n) + x16][8 * piece(x16, 4 * d + g)]),
                           operand(&lds.q[par][16 * block_row(n) + x16][8 * piece(x16, 4 * d + g)]), qk);
      pp[n] *= qk;
    }
    most = largest(pp[0], most);
  };
  // Blocks of T below the diagonal, two waves with the first column: (1, 0) and (2, 0); (2, 1) and (3, 1); (3, 2);
  // (3, 0).  Everything a chain needs from LDS is asked for before it starts.
  f32x4_t below[2];
  auto inverse = [&]() {
    const Inverse of(lds);
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    if (w == 2) {
      const f32x4_t a32 = of.a(3, 2), t2 = of.diag_plain(2), d3 = of.minus_diag(3);
      below[0] = mfma_f32_block(mfma_f32_block(a32, t2, zero), d3, zero);
    } else if (w == 1) {
      const f32x4_t a21 = of.a(2, 1), a31 = of.a(3, 1), a32 = of.a(3, 2), t1 = of.diag_plain(1), d2 = of.minus_diag(2), d3 = of.minus_diag(3);
      const f32x4_t x2 = mfma_f32_block(a21, t1, zero);
      f32x4_t x3 = mfma_f32_block(a31, t1, zero);
      const f32x4_t t21 = mfma_f32_block(d2, x2, zero);
      below[0] = mfma_f32_block(x2, d2, zero);
      x3 = mfma_f32_block(a32, t21, x3);
      below[1] = mfma_f32_block(x3, d3, zero);
    } else {
      const f32x4_t a10 = of.a(1, 0), a20 = of.a(2, 0), a21 = of.a(2, 1), t0 = of.diag_plain(0), d1 = of.minus_diag(1), d2 = of.minus_diag(2);
      if (w == 0) {
        const f32x4_t x1 = mfma_f32_block(a10, t0, zero);
        f32x4_t x2 = mfma_f32_block(a20, t0, zero);
        const f32x4_t t10 = mfma_f32_block(d1, x1, zero);
        below[0] = mfma_f32_block(x1, d1, zero);
        x2 = mfma_f32_block(a21, t10, x2);
        below[1] = mfma_f32_block(x2, d2, zero);
      } else {
        const f32x4_t a30 = of.a(3, 0), a31 = of.a(3, 1), a32 = of.a(3, 2), d3 = of.minus_diag(3);
        const f32x4_t x1 = mfma_f32_block(a10, t0, zero);
        f32x4_t x2 = mfma_f32_block(a20, t0, zero), x3 = mfma_f32_block(a30, t0, zero);
        const f32x4_t t10 = mfma_f32_block(d1, x1, zero);
        x2 = mfma_f32_block(a21, t10, x2);
        x3 = mfma_f32_block(a31, t10, x3);
        const f32x4_t t20 = mfma_f32_block(d2, x2, zero);
        x3 = mfma_f32_block(a32, t20, x3);
        below[0] = mfma_f32_block(x3, d3, zero);
      }
    }
  };
  auto store_t = [&]() {
    split_store(pick, inv, lds.t, w, w);
    const int r = w == 0 ? 1 : w == 1 ? 2 : 3, c = w == 1 ? 1 : w == 2 ? 2 : 0;
    split_store(pick, below[0], lds.t, r, c);
    if (w < 2) split_store(pick, below[1], lds.t, r + 1, c);
  };
  auto store_p = [&]() {
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      if (n >= n_blocks) break;
      split_store(pick, pp[n], lds.p, block_row(n), block_col(n));
    }
  };

  fetch(start);
  stage(start, 0);
  if (w == 2) decays(start, 0);
  slot_barrier();
  fetch_v(start);
  if (n_chunks > 1) fetch(start + kChunk);
  products(0, 0);
  slot_barrier();
  finish_p(0);
  inverse();
  if (w == 2 && n_chunks > 1) decays(start + kChunk, 1);
  slot_barrier();
  int tri = 1;  // of chunk j + 1, modulo 3
  for (int j = 0; j < n_chunks; ++j) {
    const int next = start + (j + 1) * kChunk, par = (j + 1) & 1;
    const bool more = j + 1 < n_chunks, two = j + 2 < n_chunks;
    store_t();
    store_p();
    wait_all_vm();  // V of chunk j is in LDS
    if (more) stage(next, par);
    if (two) fetch(next + kChunk);
    slot_barrier();
    __builtin_amdgcn_s_setprio(2);
    if (more) products(par, tri);
    __builtin_amdgcn_s_setprio(0);
    slot_barrier();
    tri = tri == 2 ? 0 : tri + 1;
    if (more) {
      fetch_v(next);
      finish_p(par);
      inverse();
    }
    if (w == 2 && two) decays(next + kChunk, tri);
    if (!more) lds.p_largest[64 * w + lane] = most;
    slot_barrier();
  }
}

// Workgroup -> (request, value head, half): the workgroups that read the same K and Q rows (the value
// heads of a key head, both halves) get ids of one residue modulo 8, so one L2 serves them; requests go
// longest first where there are more workgroups than compute units.
__global__ __launch_bounds__(512) void gdn_chunk_kernel(GdnParams p, int ranked) {
  __shared__ __attribute__((aligned(16))) ChunkLds lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int halves = kDV / kRowsPerWg;
  const int sharing = p.hv_per_hk * halves, hk_n = p.hv / p.hv_per_hk;
  int group, member;  // group = (request, key head)
  const int groups = p.batch * hk_n;
  if (groups % 8 == 0) {
    const int seq = blockIdx.x >> 3;
    group = (seq / sharing) * 8 + (blockIdx.x & 7);
    member = seq % sharing;
  } else {
    group = blockIdx.x / sharing;
    member = blockIdx.x % sharing;
  }
  int b = group / hk_n;
  const int hv = (group - b * hk_n) * p.hv_per_hk + member / halves;
  const int row = (member % halves) * kRowsPerWg;
  if (ranked) {
    int* lens = reinterpret_cast<int*>(&lds.k[0][0][0]);
    const int tid = threadIdx.x;
    int mine = 0;
    if (tid < p.batch) lens[tid] = mine = p.qo_indptr[tid + 1] - p.qo_indptr[tid];
    __syncthreads();
    if (tid < p.batch) {
      int rank = 0;
      for (int o = 0; o < p.batch; ++o) rank += (lens[o] > mine || (lens[o] == mine && o < tid)) ? 1 : 0;
      if (rank == b) lds.request = tid;
    }
    __syncthreads();
    b = lds.request;
    __syncthreads();
  }
  b = __builtin_amdgcn_readfirstlane(b);
  const int start = p.qo_indptr[b], end = min(p.qo_indptr[b + 1], p.tokens);
  if (end <= start) return;  // the whole workgroup: the state stays as it is
  // the blocks of T and P above the diagonal that are read are never written: zero from here on
  for (int i = threadIdx.x; i < (int)(sizeof(lds.t) + sizeof(lds.p)) / 16; i += 512)
    reinterpret_cast<u32x4_t*>(&lds.t[0][0][0])[i] = u32x4_t{0u, 0u, 0u, 0u};
  if (wave < 4) state_waves(p, lds, start, end, __builtin_amdgcn_readfirstlane(p.slot_ids[b]), hv, row + 16 * wave, 16 * wave);
  else chunk_waves(p, lds, start, end, hv, row, wave - 4);
}

}  // namespace

int launch_gdn_chunks(const GdnParams& p, hipStream_t stream) {
  const int64_t blocks = (int64_t)p.batch * p.hv * (kDV / kRowsPerWg);
  if (blocks > 0x7fffffffLL) return MSGL_ERR_SHAPE;
  const int ranked = p.batch > 1 && p.batch <= kRanked && blocks > device_cus();
  hipLaunchKernelGGL(gdn_chunk_kernel, dim3((unsigned)blocks), dim3(512), 0, stream, p, ranked);
  return check_launch();
}

}  // namespace msgl
