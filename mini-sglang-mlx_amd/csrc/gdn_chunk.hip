// Gated delta rule over many tokens per request: chunks of 64 tokens on the matrix cores, in one launch.  (Requests of several
// hundred tokens take two where there is memory for the systems below: gdn_long.hip.)
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
// 4.3 us, or 3.2 us in pairs of waves (below).  Requests of 992, 1581, 4005 and 1601 tokens at hk 16, hv 32:
// 1353 -> 217 us (283 without pairs); one of 2000: 147 -> 109.
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
// What bounds it: a chunk takes 10.4 K cycles (slots of 3.4, 2.6 and 4.3 K), in which a SIMD has 5.3 K cycles of
// matrix instructions and as many of vector instructions in two chains that wait for their own results, and a
// wave that has the SIMD for itself still pays about 5 cycles per instruction of any kind.  The last wave of a slot is
// a chunk wave in slots 1 and 3, some 0.4 K cycles behind the slowest state wave.  Hence: fp32 values
// are split by the matrix pipe (see Split: 16 instructions instead of 44), Z and Y are made transposed (4 stores
// of 8 bytes a chunk instead of 16 of 2), V comes by transposing LDS reads, the chunk waves share the blocks
// out evenly (12.5 -> 10.7 K), and what a block needs from LDS is read whether it is used or not (no branches, so the
// reads of several blocks go out together: 10.6 -> 10.4 K).
//
// Pairs: the longest request's chain ends a launch when the others have left their compute units, and a launch of few
// requests never fills the chip.  Such requests go on four workgroups a value head, of 32 rows: waves 0-1 are state
// waves, and waves 2-3 ("output" waves) take what the next chunk does not wait for, Z and Y, from the S and U that
// their state wave leaves in LDS, and P:
//     slot   state waves, chunk j          output waves                  chunk waves
//      1     X, R                           Z, two blocks of P to LDS      T of chunk j, K and Q of chunk j + 1 to LDS
//      2     U, two blocks of A of j + 1    P of chunk j + 1               A, the diagonal blocks of T of chunk j + 1
//      3     S                              Y, three blocks of P to LDS    the other blocks of T of chunk j + 1, V of j + 2
// A chunk takes 7.7 K cycles (slots of 2.5, 2.4 and 2.7 K, every role 1.9-2.6 K of each).  It is 1.5 times the work of
// the chip for a chunk, so a launch that fills the compute units evenly has no pairs (see in_pairs()).
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
#include "gdn_chunk_tiles.h"

namespace msgl {
namespace {

constexpr int kRowsPerWg = 64;    // dv rows of a workgroup
constexpr int kRowsPaired = 32;   // where output waves take half of the state waves' work

template <bool PAIRED>
struct ChunkLds {
  uint16_t k[2][kChunk][kDK], q[2][kChunk][kDK];  // 16-byte pieces of a row in swizzled order (see piece())
  uint16_t v[PAIRED ? 2 : 1][kChunk][PAIRED ? kRowsPaired : kRowsPerWg];
  u32x4_t t[3][kFragments][64], p[3][kFragments][64];  // T and P in three bf16 parts
  float a[kChunk][68];            // A of the chunk being prepared (blocks on and below the diagonal)
  float diag[4][16][20];          // inverses of the diagonal blocks of I + A
  __device__ __forceinline__ const float* a_row(int r, int c, int row) const { return &a[16 * r + row][16 * c]; }
  __device__ __forceinline__ const float* diagonal_row(int r, int row) const { return diag[r][row]; }
  // per token, chunks j .. j + 2: beta, G, and tail_i = G_64 / G_i
  float beta[3][kChunk], gamma[3][kChunk], tail[3][kChunk];
  // of the chunk being prepared: the decays; products over the block of 16 up to a token, behind it, and
  // over its quad up to it; products over whole blocks and over the quads of each block
  float g[kChunk], pre[kChunk], suf[kChunk], quad_pre[kChunk], block[4], quad[16];
  float total[3];                 // G_64, chunks j .. j + 2 (last: the arrays above are read 16 bytes at a time)
  int request;
  alignas(16) float p_largest[4 * 64];  // per lane of the waves that make P: largest() of P's diagonal blocks, all chunks
};
struct PairedLds : ChunkLds<true> {
  f32x4_t s[2][8][64], u[2][4][64];  // a state wave's S and U for its output wave, registers as they are
};

template <bool PAIRED, typename Lds>
__device__ __forceinline__ void state_waves(const GdnParams& p, Lds& lds, int start, int end, int slot, int hv,
                                            int row, int column) {
  const int lane = lane_id(), x16 = lane & 15, g = lane >> 4;
  const int n_chunks = (end - start + kChunk - 1) / kChunk;
  f32x4_t s[8];  // s[2 c + h][i]: dim 32 c + 8 g + 4 h + i of row `row + x16`
  float* srow = state_row(slot, hv, row);
#pragma unroll
  for (int c = 0; c < 8; ++c) s[c] = *reinterpret_cast<const f32x4_t*>(srow + 32 * (c >> 1) + 4 * (c & 1));

  const Outputs y(p, start, end, hv, row);
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
      if constexpr (!PAIRED) r.q[m] = operand(&lds.q[par][16 * m][0] + at[c]);
    }
  };
  auto hand_over = [&](f32x4_t (*to)[64], const f32x4_t* from, int n) {
#pragma unroll
    for (int i = 0; i < n; ++i) to[i][lane] = from[i];
  };
  if constexpr (PAIRED) hand_over(lds.s[column >> 4], s, 8);
  __builtin_amdgcn_s_setprio(1);  // before the chunk waves, but in slot 2, where those have the longer way
  auto a_block = [&](int par, int tri) {  // (3, 2), and the other state wave (2, 1)
    const int r = column ? 2 : 3, c = r - 1;
    BelowBlock x;
    x.load(lds, lds.k[par], lds.beta[tri], r, c);
    x.store(lds, r, c, block_dots(x.kc, x.kr));
  };
  slot_barrier();  // K, Q of chunk 0
  if constexpr (PAIRED) a_block(0, 0);
  slot_barrier();  // A of chunk 0
  slot_barrier();  // what T of chunk 0 is made of

  Rows rows[2];
  load_rows(0, 0, rows[0]);
  Split sp = split(pick, s[0], s[1]);
  float most = 0.f;  // largest() of every U
  for (int j = 0, tri = 0; j < n_chunks; ++j, tri = tri == 2 ? 0 : tri + 1) {
    const int par = j & 1;
    Triangle tp;
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
          if constexpr (!PAIRED) z[m] = product<true>(r.q[m], part, z[m]);
        }
      };
      const Split now = sp;
      step(now.lo);
      if (c < 3) sp = split(pick, s[2 * c + 2], s[2 * c + 3]);
      step(now.mid);
      step(now.hi);
      fence();
    }
    Split rs0, rs1;
    auto make_r = [&]() {
      f32x4_t r[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const f32x4_t bet = *reinterpret_cast<const f32x4_t*>(&lds.beta[tri][16 * m + 4 * g]);
        const f32x4_t gam = *reinterpret_cast<const f32x4_t*>(&lds.gamma[tri][16 * m + 4 * g]);
        const u32x2_t v = lds_read_tr16(reinterpret_cast<const unsigned char*>(&lds.v[PAIRED ? par : 0][16 * m + trow][column + 4 * (x16 & 3)]));
#pragma unroll
        for (int i = 0; i < 4; ++i)
          r[m][i] = (bf16_bits_to_f32(i & 1 ? v[i >> 1] >> 16 : v[i >> 1] & 0xffffu) - gam[i] * x[m][i]) * bet[i];
      }
      if constexpr (!PAIRED) load_triangle<4, 6>(lds.t, tp);
      rs0 = split(pick, r[0], r[1]);
      rs1 = split(pick, r[2], r[3]);
    };
    if constexpr (PAIRED) make_r();
    slot_barrier();
    // ---- slot 2 ----------------------------------------------------------------------------
    if constexpr (PAIRED) a_block(par ^ 1, tri == 2 ? 0 : tri + 1);  // of chunk j + 1 (of no use behind the last one)
    load_triangle<0, PAIRED ? 6 : 4>(lds.t, tp);
    if constexpr (!PAIRED) make_r();
    f32x4_t u[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) u[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    triangle_first<false>(tp, rs0, u);
    triangle_second<false>(tp, rs1, u);
    f32x4_t tail[4];
    Split ut0, ut1;
    auto take_tail = [&]() {
#pragma unroll
      for (int m = 0; m < 4; ++m) tail[m] = *reinterpret_cast<const f32x4_t*>(&lds.tail[tri][16 * m + 4 * g]);
    };
    auto weigh = [&]() {
      ut0 = split(pick, u[0] * tail[0], u[1] * tail[1]);
      ut1 = split(pick, u[2] * tail[2], u[3] * tail[3]);
    };
    if constexpr (PAIRED) {
      hand_over(lds.u[column >> 4], u, 4);
    } else {
#pragma unroll
      for (int m = 0; m < 4; ++m) z[m] *= lds.gamma[tri][16 * m + x16];
      fence();
      load_triangle<0, 4>(lds.p, tp);
    }
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
    take_tail();
    const float total = lds.total[tri];
    if constexpr (!PAIRED) load_triangle<4, 6>(lds.p, tp);
    load_kt(0, ka[0]);
    load_kt(1, ka[1]);
    Split us1;
    if constexpr (!PAIRED) {
      const Split us0 = split(pick, u[0], u[1]);
      us1 = split(pick, u[2], u[3]);
      fence();
      triangle_first<true>(tp, us0, z);
    }
    weigh();
#pragma unroll
    for (int c = 0; c < 8; ++c) s[c] *= total;
#pragma unroll
    for (int m = 0; m < 4; ++m) most = largest(u[m], most);
    fence();
    if constexpr (!PAIRED) triangle_second<true>(tp, us1, z);
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
    if constexpr (!PAIRED) y.store(j, z);
    fence();
    load_rows(par ^ 1, 0, rows[0]);  // of chunk j + 1 (of no use behind the last chunk)
    steps(3, ut1);
    sp = split(pick, s[0], s[1]);
    if constexpr (PAIRED) hand_over(lds.s[column >> 4], s, 8);
    slot_barrier();
  }
  if constexpr (PAIRED) slot_barrier();  // the output waves' stores are done
  most = largest(*reinterpret_cast<const f32x4_t*>(&lds.p_largest[4 * (PAIRED ? lane & 31 : lane)]), most);
  if (__builtin_expect(!__all(splits(most)), 0)) {
    wait_all_vm();  // the stores of Y: the same places are written again
    token_by_token(start, end, slot, hv, row);
    return;
  }
  srow = state_row(slot, hv, row);
#pragma unroll
  for (int c = 0; c < 8; ++c) *reinterpret_cast<f32x4_t*>(srow + 32 * (c >> 1) + 4 * (c & 1)) = s[c];
}

template <bool PAIRED, typename Lds>
__device__ __forceinline__ void chunk_waves(const GdnParams& p, Lds& lds, int start, int end, int hv,
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
  // V of the workgroup's rows, 8 tokens a load (16 of half as many rows), straight to LDS; rows past the request's end: the last row
  // (beta is zero there)
  const char* vbase = reinterpret_cast<const char*>(p.v + (int64_t)start * p.v_stride0 + hv * kDV + wg_row);
  const uint32_t v_step = (uint32_t)p.v_stride0 * 2u, v_lds = (uint32_t)(uintptr_t)MSGL_LDS_PTR(uint16_t, &lds.v[0][16 * w][0]);
  auto fetch_v = [&](int first, int par = 0) {
    const char* base = vbase + (int64_t)(first - start) * v_step;
    constexpr int kLanes = PAIRED ? 4 : 8;  // a token
#pragma unroll
    for (int n = 0; n < kLanes / 4; ++n)
      lds_direct_b128(__builtin_amdgcn_readfirstlane(v_lds + 1024 * n + par * (uint32_t)sizeof(lds.v[0])), base,
                      min((uint32_t)(16 * w + 8 * n + lane / kLanes), (uint32_t)(end - 1 - first)) * v_step + 16 * (lane % kLanes));
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
    decay_products(lds, gv, bv, lds.beta[tri], lds.gamma[tri], lds.tail[tri], lds.total[tri]);
  };
  // The ten blocks (r, c) of A and P on and below the diagonal: every wave its diagonal block and one
  // more, waves 1 and 2 two (PAIRED: the state waves have those).  Results are transposed (lane: token t = 16 r + x16, tokens i = 16 c + 4 g + n), so that a
  // lane's four values are neighbours in a row of A and of P.
  const int n_blocks = PAIRED || w == 0 || w == 3 ? 2 : 3;
  auto block_row = [&](int n) { return n == 0 ? w : n == 1 ? (w == 0 ? 3 : w) : (w == 2 ? 2 : 3); };
  auto block_col = [&](int n) { return n == 0 ? w : n == 1 ? (w == 3 ? 1 : 0) : (w == 1 ? 2 : 1); };
  f32x4_t pp0, pp1, pp2;  // the ratios of P of these blocks, then P
  float most = 0.f;  // largest() of P's diagonal block, every chunk
  f32x4_t inv;    // the inverse of the diagonal block: row x16, columns 4 g ..
  auto products = [&](int par, int tri) {
    BelowBlock b0, b1, b2;
    const int r1 = block_row(1), c1 = block_col(1), r2 = block_row(2), c2 = block_col(2);
    b0.load(lds, lds.k[par], lds.beta[tri], w, w);
    b1.load(lds, lds.k[par], lds.beta[tri], r1, c1);
    const f32x4_t kk0 = block_dots(b0.kc, b0.kr);
    {
      const f32x4_t ratio = b0.decays.diagonal(lds, w);
      f32x4_t a;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i] = 4 * g + i < x16 ? -b0.beta * ratio[i] * kk0[i] : 0.f;  // negated, as eliminate() takes it
        if constexpr (!PAIRED) pp0[i] = 4 * g + i <= x16 ? ratio[i] : 0.f;
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
    // (no two branches of a lambda end in stores to different captures: those become one store to a chosen address,
    // and the captures go to scratch memory)
    if (n_blocks > 2) {
      b2.load(lds, lds.k[par], lds.beta[tri], r2, c2);
      const f32x4_t kk1 = block_dots(b1.kc, b1.kr), kk2 = block_dots(b2.kc, b2.kr);
      eliminate<0>(arow, inv);
      pp2 = b2.store(lds, r2, c2, kk2);
      pp1 = b1.store(lds, r1, c1, kk1);
    } else {
      const f32x4_t kk1 = block_dots(b1.kc, b1.kr);
      eliminate<0>(arow, inv);
      pp1 = b1.store(lds, r1, c1, kk1);
    }
    *reinterpret_cast<f32x4_t*>(&lds.diag[w][x16][4 * g]) = inv;
  };
  auto finish_p = [&](int par) {  // P = ratios times <k, q>
    auto times_dots = [&](int n, f32x4_t& x) {
      bf16x8_t k[4], q[4];
      load_block_rows(lds.k[par], block_col(n), k);
      load_block_rows(lds.q[par], block_row(n), q);
      x *= block_dots(k, q);
    };
    times_dots(0, pp0);
    times_dots(1, pp1);
    if (n_blocks > 2) times_dots(2, pp2);
    most = largest(pp0, most);
  };
  Below below;
  auto store_t = [&]() {
    f32x4_t first = below.first;
    if (PAIRED && w == 3) first = mfma_f32_block(first, below.second, f32x4_t{0.f, 0.f, 0.f, 0.f});
    split_store(pick, inv, lds.t, w, w);
    const int r = w == 0 ? 1 : w == 1 ? 2 : 3, c = w == 1 ? 1 : w == 2 ? 2 : 0;
    split_store(pick, first, lds.t, r, c);
    if (w < 2) split_store(pick, below.second, lds.t, r + 1, c);
  };
  auto store_p = [&]() {
    split_store(pick, pp0, lds.p, block_row(0), block_col(0));
    split_store(pick, pp1, lds.p, block_row(1), block_col(1));
    if (n_blocks > 2) split_store(pick, pp2, lds.p, block_row(2), block_col(2));
  };

  fetch(start);
  stage(start, 0);
  if (w == 2) decays(start, 0);
  slot_barrier();
  fetch_v(start);
  if (n_chunks > 1) fetch(start + kChunk);
  products(0, 0);
  slot_barrier();
  if constexpr (!PAIRED) finish_p(0);
  below = blocks_below<PAIRED>(lds, w);
  if (w == 2 && n_chunks > 1) decays(start + kChunk, 1);
  if constexpr (PAIRED) {
    wait_all_vm();  // V of chunk 0 is in LDS
    if (n_chunks > 1) fetch_v(start + kChunk, 1);
  }
  slot_barrier();
  int tri = 1;  // of chunk j + 1, modulo 3
  for (int j = 0; j < n_chunks; ++j) {
    const int next = start + (j + 1) * kChunk, par = (j + 1) & 1;
    const bool more = j + 1 < n_chunks, two = j + 2 < n_chunks;
    store_t();
    if constexpr (!PAIRED) store_p();
    wait_all_vm();  // V of chunk j (PAIRED: j + 1) is in LDS
    if (more) stage(next, par);
    if (two) fetch(next + kChunk);
    slot_barrier();
    __builtin_amdgcn_s_setprio(2);
    if (more) products(par, tri);
    __builtin_amdgcn_s_setprio(0);
    slot_barrier();
    tri = tri == 2 ? 0 : tri + 1;
    if (PAIRED && two) fetch_v(next + kChunk, j & 1);
    if (more) {
      if constexpr (!PAIRED) fetch_v(next);
      if constexpr (!PAIRED) finish_p(par);
      below = blocks_below<PAIRED>(lds, w);
    }
    if (w == 2 && two) decays(next + kChunk, tri);
    if (!PAIRED && !more) lds.p_largest[64 * w + lane] = most;
    slot_barrier();
  }
  if constexpr (PAIRED) slot_barrier();
}

// The half of a state wave's work that the next chunk does not wait for, and P: slot 1 of a chunk P to LDS and
// Z = Q S^T, slot 2 P of the next chunk, slot 3 Y = G Z + P U.  S and U come from the state wave, one slot behind it.
template <int w>
__device__ __forceinline__ void output_waves(const GdnParams& p, PairedLds& lds, int start, int end, int hv, int row) {
  const int lane = lane_id(), x16 = lane & 15, g = lane >> 4;
  const int n_chunks = (end - start + kChunk - 1) / kChunk;
  const Outputs y(p, start, end, hv, row);
  const Picker pick;
  // the blocks of P: wave 0 has (0, 0), (1, 1), (1, 0), (2, 0) and (2, 1), wave 1 (2, 2), (3, 3), (3, 0), (3, 1) and (3, 2)
  constexpr int block_row[5] = {2 * w, 2 * w + 1, w ? 3 : 1, w ? 3 : 2, w ? 3 : 2};
  constexpr int block_col[5] = {2 * w, 2 * w + 1, 0, w ? 1 : 0, w ? 2 : 1};
  constexpr int kColumns = w ? 4 : 2, kFirstRow = w ? 2 : 0, kRows = w ? 2 : 3;  // of K, of Q
  f32x4_t pp[5];
  float most = 0.f;  // largest() of P's diagonal blocks, every chunk
  auto make_p = [&](int par) {
    bf16x8_t k[kColumns][4], q[kRows][4];
#pragma unroll
    for (int c = 0; c < kColumns; ++c) load_block_rows(lds.k[par], c, k[c]);
#pragma unroll
    for (int r = 0; r < kRows; ++r) load_block_rows(lds.q[par], kFirstRow + r, q[r]);
#pragma unroll
    for (int n = 0; n < 5; ++n) {
      const int r = block_row[n], c = block_col[n];
      Decays decays;
      decays.load(lds, r, c);
      f32x4_t ratio;
      if (n < 2) {
        ratio = decays.diagonal(lds, r);
#pragma unroll
        for (int i = 0; i < 4; ++i) ratio[i] = 4 * g + i <= x16 ? ratio[i] : 0.f;
      } else {
        ratio = decays.below(lds, r, c);
      }
      pp[n] = ratio * block_dots(k[c], q[r - kFirstRow]);
      if (n < 2) most = largest(pp[n], most);
    }
  };
  auto store_p = [&](int from, int to) {
#pragma unroll
    for (int n = 0; n < 5; ++n)
      if (n >= from && n < to) split_store(pick, pp[n], lds.p, block_row[n], block_col[n]);
  };
  uint32_t at[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) at[c] = x16 * kDK + 8 * piece(x16, 4 * c + g);
  slot_barrier();
  make_p(0);
  slot_barrier();
  store_p(0, 3);
  slot_barrier();
  for (int j = 0, tri = 0; j < n_chunks; ++j, tri = tri == 2 ? 0 : tri + 1) {
    const int par = j & 1;
    f32x4_t z[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) z[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      bf16x8_t q[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) q[m] = operand(&lds.q[par][16 * m][0] + at[c]);
      const Split sp = split(pick, lds.s[w][2 * c][lane], lds.s[w][2 * c + 1][lane]);
      auto step = [&](bf16x8_t part) {
#pragma unroll
        for (int m = 0; m < 4; ++m) z[m] = product<true>(q[m], part, z[m]);
      };
      step(sp.lo);
      step(sp.mid);
      step(sp.hi);
    }
    store_p(3, 5);
    slot_barrier();
    Triangle tp;
    load_triangle<0, 6>(lds.p, tp);
#pragma unroll
    for (int m = 0; m < 4; ++m) z[m] *= lds.gamma[tri][16 * m + x16];
    if (j + 1 < n_chunks) make_p(par ^ 1);
    slot_barrier();
    const Split us0 = split(pick, lds.u[w][0][lane], lds.u[w][1][lane]);
    const Split us1 = split(pick, lds.u[w][2][lane], lds.u[w][3][lane]);
    triangle_first<true>(tp, us0, z);
    triangle_second<true>(tp, us1, z);
    y.store(j, z);
    store_p(0, 3);  // of the next chunk (of no use behind the last one)
    slot_barrier();
  }
  lds.p_largest[64 * w + lane] = most;
  wait_all_vm();  // the state waves may have to write the same places again
  slot_barrier();
}

// Requests in pairs: the `n` longest, each on four workgroups a value head instead of two and so with two of the
// `slots` that a request without takes one of.  As many as leave a slot for every request; and beyond that down to the
// i-th longest, if the rest (chunks on the slots that are left, and what the last one of them may stick out) ends
// before it: 3/4 of the time that it takes without.
__device__ __forceinline__ bool in_pairs(int i, int chunks, int rest, int shortest, int batch, int slots) {
  const int left = slots - 2 * (i + 1);
  return i < slots - batch || (left > 0 && 4 * (rest + (left - 1) * shortest) <= 3 * left * chunks);
}
// How many there are at most.  Where these do not all fit beside the others, workgroups of places that stay empty wait
// for a compute unit at the end of the launch: 1.3 us, which launches of short requests are spared.
constexpr int kPairsMeanTokens = 768;
inline int most_in_pairs(const GdnParams& p, int64_t cus) {
  const int64_t slots = cus / (p.hv * (kDV / kRowsPerWg));
  const int64_t long_ones = p.tokens >= (int64_t)kPairsMeanTokens * p.batch ? (slots - 1) / 2 : 0;
  return p.batch > 64 ? 0 : (int)std::min<int64_t>(p.batch, std::max<int64_t>({slots - p.batch, long_ones, 0}));
}

// Workgroup -> (place, value head, half or quarter of its rows): the workgroups that read the same K and Q rows (the
// value heads of a key head, their halves) get ids of one residue modulo 8, so one L2 serves them; a request in
// pairs has two places.  Requests go longest first where there are more workgroups than compute units or some may go
// in pairs.
__global__ __launch_bounds__(512) void gdn_chunk_kernel(GdnParams p, int ranked, int places, int slots) {
  __shared__ union {
    ChunkLds<false> whole;
    PairedLds paired;
    struct {
      int length[kRanked], request;
    } order;
  } lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int halves = kDV / kRowsPerWg;
  const int sharing = p.hv_per_hk * halves, hk_n = p.hv / p.hv_per_hk;
  int group, member;  // group = (place, key head)
  const int groups = places * hk_n;
  if (groups % 8 == 0) {
    const int seq = blockIdx.x >> 3;
    group = (seq / sharing) * 8 + (blockIdx.x & 7);
    member = seq % sharing;
  } else {
    group = blockIdx.x / sharing;
    member = blockIdx.x % sharing;
  }
  const int place = group / hk_n, half = member % halves;
  const int hv = (group - place * hk_n) * p.hv_per_hk + member / halves;
  int b = place, n_paired = 0;
  int start, end;
  if (p.batch <= 64 && (ranked || places > p.batch)) {  // every wave for itself, a request per lane
    const int lane = lane_id(), at = min(lane, p.batch - 1);
    const int from = p.qo_indptr[at], to = p.qo_indptr[at + 1];
    const int length = lane < p.batch ? max(0, to - from) : -1;
    int rank = 0, rest = 0, shortest = 0x7fffffff;
    for (int o = 0; o < p.batch; ++o) {
      const int other = __builtin_amdgcn_readlane(length, o), chunks = (other + kChunk - 1) / kChunk;
      const bool before = other > length || (other == length && o < lane);
      rank += before ? 1 : 0;
      rest += before || o == lane ? 0 : chunks;
      shortest = min(shortest, chunks);
    }
    const bool pairs = lane < p.batch && rank < places - p.batch &&
                       in_pairs(rank, (length + kChunk - 1) / kChunk, rest, shortest, p.batch, slots);
    while (__ballot(pairs && rank >= n_paired)) ++n_paired;
    const int wanted = place < 2 * n_paired ? place >> 1 : place - n_paired;
    const uint64_t found = __ballot(lane < p.batch && rank == wanted);
    if (!found) return;  // a place for a request in pairs that there is not: the whole workgroup
    b = __builtin_ctzll(found);
    start = __builtin_amdgcn_readlane(from, b);
    end = __builtin_amdgcn_readlane(to, b);
  } else {
    if (ranked) {
      const int tid = threadIdx.x;
      int mine = 0;
      if (tid < p.batch) lds.order.length[tid] = mine = p.qo_indptr[tid + 1] - p.qo_indptr[tid];
      __syncthreads();
      if (tid < p.batch) {
        int rank = 0;
        for (int o = 0; o < p.batch; ++o) rank += (lds.order.length[o] > mine || (lds.order.length[o] == mine && o < tid)) ? 1 : 0;
        if (rank == b) lds.order.request = tid;
      }
      __syncthreads();
      b = lds.order.request;
      __syncthreads();
    }
    b = __builtin_amdgcn_readfirstlane(b);
    start = p.qo_indptr[b];
    end = p.qo_indptr[b + 1];
  }
  end = min(end, p.tokens);
  if (end <= start) return;  // the whole workgroup: the state stays as it is
  const int slot = __builtin_amdgcn_readfirstlane(p.slot_ids[b]);
  // the blocks of T and P above the diagonal that are read are never written: zero from here on
  auto clear = [](auto& t, auto& p) {
    for (int i = threadIdx.x; i < (int)(sizeof(t) + sizeof(p)) / 16; i += 512)
      reinterpret_cast<u32x4_t*>(&t[0][0][0])[i] = u32x4_t{0u, 0u, 0u, 0u};
  };
  if (place < 2 * n_paired) {
    const int row = (place & 1) * kRowsPerWg + half * kRowsPaired;
    clear(lds.paired.t, lds.paired.p);
    if (wave < 2) state_waves<true>(p, lds.paired, start, end, slot, hv, row + 16 * wave, 16 * wave);
    else if (wave == 2) output_waves<0>(p, lds.paired, start, end, hv, row);
    else if (wave == 3) output_waves<1>(p, lds.paired, start, end, hv, row + 16);
    else chunk_waves<true>(p, lds.paired, start, end, hv, row, wave == 6 ? 3 : wave == 7 ? 2 : wave - 4);
  } else {
    const int row = half * kRowsPerWg;
    clear(lds.whole.t, lds.whole.p);
    if (wave < 4) state_waves<false>(p, lds.whole, start, end, slot, hv, row + 16 * wave, 16 * wave);
    else chunk_waves<false>(p, lds.whole, start, end, hv, row, wave - 4);
  }
}

}  // namespace

int launch_gdn_chunks(const GdnParams& p, hipStream_t stream) {
  const int64_t cus = device_cus();
  const int64_t places = p.batch + most_in_pairs(p, cus);
  const int64_t blocks = places * p.hv * (kDV / kRowsPerWg);
  if (blocks > 0x7fffffffLL) return MSGL_ERR_SHAPE;
  const int ranked = p.batch > 1 && p.batch <= kRanked && blocks > cus;
  hipLaunchKernelGGL(gdn_chunk_kernel, dim3((unsigned)blocks), dim3(512), 0, stream, p, ranked, (int)places, (int)(cus / (p.hv * (kDV / kRowsPerWg))));
  return check_launch();
}

}  // namespace msgl
