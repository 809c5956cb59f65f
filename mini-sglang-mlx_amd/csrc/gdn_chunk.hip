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
// 5.2 us.  Requests of 992, 1581, 4005 and 1601 tokens at hk 16, hv 32: 1353 -> 330 us; one of 1024: 298 -> 90.
//
// Work: one workgroup per (request, value head, half of its 128 rows).  Waves 0-3 ("state" waves, 16
// rows each, S^T in 32 accumulator registers) run the serial part of chunk j; waves 4-7 ("chunk" waves,
// 16 tokens each) make T and P of chunk j + 1 beside them, one of each on a SIMD.  Three slots per
// chunk, a workgroup barrier behind each:
//     slot   state waves, chunk j                 chunk waves
//      1     X = K S^T, Z = Q S^T                  P of chunk j and K, Q of chunk j + 1 to LDS
//      2     R = beta (V - G X), U = T R           A, P and the diagonal blocks of T of chunk j + 1
//      3     Y = G Z + P U, S = G_64 S + K^T U     the blocks of T below the diagonal; T of chunk j + 1 to LDS;
//                                                  decay products of chunk j + 2
// What bounds it: a chunk takes 12.5 K cycles (slots of 3.1, 3.9 and 5.0 K), of which the matrix pipe is busy
// 4.4 K, LDS 5.2 K and the vector ALU about 5 K: three chains that depend on each other, on one wave each per
// SIMD.  Operands are asked for a step, and across the barriers a slot, before they are used, and the splits
// stand between the matrix instructions.
//
// Precision: fp32 throughout, as in the token kernel.  q, k, v are bf16 and enter the bf16 matrix
// instructions as they are; fp32 operands (S, R, U, T, P) are split into three bf16 parts of 8
// significant bits each, which hold all 24, and multiplied part by part into fp32 accumulators (for
// two split operands the six products above 2^-24 of the result).  The inverse is built from fp32
// matrix instructions.  Decay ratios are products of the decays (no logarithms: a decay may be 0).
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
// Rows of 304 bytes: 16 rows at one column lie in 16 different groups of four banks, and so do, all but
// three, the 4 rows x 4 columns of a transposing read (rows of 272 bytes: 4 of those in one group).
constexpr int kRowPad = 152;
constexpr int kRanked = 512;      // requests ranked by length (one per thread)

struct ChunkLds {
  uint16_t k[2][kChunk][kRowPad];
  uint16_t q[2][kChunk][kRowPad];
  uint16_t t[3][kChunk][72];      // T and P in three bf16 parts, columns in contraction order
  uint16_t p[3][kChunk][72];
  float a[kChunk][68];            // A of the chunk being prepared (blocks on and below the diagonal)
  float diag[4][16][20];          // inverses of the diagonal blocks of I + A
  // per token, chunks j .. j + 2: beta, G, and tail_i = G_64 / G_i
  float beta[3][kChunk], gamma[3][kChunk], tail[3][kChunk];
  // of the chunk being prepared: the decays; products over the block of 16 up to a token, behind it, and
  // over its quad up to it; products over whole blocks and over the quads of each block
  float g[kChunk], pre[kChunk], suf[kChunk], quad_pre[kChunk], block[4], quad[16];
  float total[3];                 // G_64, chunks j .. j + 2 (last: the arrays above are read 16 bytes at a time)
  int request;
};

// Eight fp32 values as three operands of bf16 parts: x = hi + mid + lo (each cut, so exact).
struct Split {
  bf16x8_t hi, mid, lo;
};
__device__ __forceinline__ float upper(float x) {
  return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) & 0xffff0000u);
}
__device__ __forceinline__ Split split(f32x4_t a, f32x4_t b) {
  u32x4_t hi, mid, lo;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float x0 = j < 2 ? a[2 * j] : b[2 * j - 4], x1 = j < 2 ? a[2 * j + 1] : b[2 * j - 3];
    const float y0 = x0 - upper(x0), y1 = x1 - upper(x1);
    const float z0 = y0 - upper(y0), z1 = y1 - upper(y1);
    hi[j] = pack_hi16(__builtin_bit_cast(uint32_t, x0), __builtin_bit_cast(uint32_t, x1));
    mid[j] = pack_hi16(__builtin_bit_cast(uint32_t, y0), __builtin_bit_cast(uint32_t, y1));
    lo[j] = pack_hi16(__builtin_bit_cast(uint32_t, z0), __builtin_bit_cast(uint32_t, z1));
  }
  return Split{as_bf16x8(hi), as_bf16x8(mid), as_bf16x8(lo)};
}
// Four neighbouring values of a row of T or P, in three parts.
__device__ __forceinline__ void split_store(f32x4_t x, uint16_t (*m)[kChunk][72], int row, int col) {
  f32x4_t y, z;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float f = x[i], rest = f - upper(f);
    y[i] = rest;
    z[i] = rest - upper(rest);
  }
  auto cut = [](f32x4_t f) {
    const u32x4_t u = __builtin_bit_cast(u32x4_t, f);
    return u32x2_t{pack_hi16(u[0], u[1]), pack_hi16(u[2], u[3])};
  };
  *reinterpret_cast<u32x2_t*>(&m[0][row][col]) = cut(x);
  *reinterpret_cast<u32x2_t*>(&m[1][row][col]) = cut(y);
  *reinterpret_cast<u32x2_t*>(&m[2][row][col]) = cut(z);
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

// Column of tokens 16 c + 4 q .. + 3 of a chunk in the rows of T and P (see Layouts).
__device__ __forceinline__ int token_column(int c, int q) { return 32 * (c >> 1) + 8 * q + 4 * (c & 1); }

// Operands of the row blocks of T or P that reach contraction step c (m = 2 c .. 3), in three parts.
struct Triangle {
  bf16x8_t hi[4], mid[4], lo[4];
};
__device__ __forceinline__ void load_triangle(const uint16_t (*m0)[kChunk][72], int c, Triangle& t) {
  const int x16 = lane_id() & 15, g = lane_id() >> 4;
#pragma unroll
  for (int m = 2 * c; m < 4; ++m) {
    t.hi[m] = operand(&m0[0][16 * m + x16][32 * c + 8 * g]);
    t.mid[m] = operand(&m0[1][16 * m + x16][32 * c + 8 * g]);
    t.lo[m] = operand(&m0[2][16 * m + x16][32 * c + 8 * g]);
  }
}
// acc += M B for contraction step C of M (row blocks m = 2 C .. 3), B split: the six products above 2^-24,
// smallest first, the row blocks side by side.
template <int C>
__device__ __forceinline__ void triangle_product(const Triangle& t, const Split& b, f32x4_t (&acc)[4]) {
  auto step = [&](const bf16x8_t (&part)[4], const bf16x8_t& b0) {
#pragma unroll
    for (int m = 2 * C; m < 4; ++m) acc[m] = mfma_16x16x32(part[m], b0, acc[m]);
  };
  step(t.lo, b.hi);
  step(t.mid, b.mid);
  step(t.hi, b.lo);
  step(t.mid, b.hi);
  step(t.hi, b.mid);
  step(t.hi, b.hi);
}
// Scheduling of what stands between two fences: N times one matrix instruction and V vector instructions
// behind it.  A wave alone issues a vector instruction every 5 cycles and a matrix instruction every 16, so
// two or three of the former run in the shadow of each of the latter, if they stand there.
template <int N, int V>
__device__ __forceinline__ void interleave() {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, V, 0);
  }
}
__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }

__device__ __forceinline__ void state_waves(const GdnParams& p, ChunkLds& lds, int start, int end, int slot, int hv,
                                            int row) {
  const int lane = lane_id(), x16 = lane & 15, g = lane >> 4;
  const int n_chunks = (end - start + kChunk - 1) / kChunk;
  float* srow = p.state + (int64_t)slot * p.state_stride0 + ((int64_t)hv * kDV + row + x16) * kDK + 8 * g;
  f32x4_t s[8];  // s[2 c + h][i]: dim 32 c + 8 g + 4 h + i of row `row + x16`
#pragma unroll
  for (int c = 0; c < 8; ++c) s[c] = *reinterpret_cast<const f32x4_t*>(srow + 32 * (c >> 1) + 4 * (c & 1));

  // V and Y of tokens 16 m + 4 g + i of a chunk: one scalar base per chunk, 32-bit offsets of the rows
  const uint16_t* vrow = p.v + (int64_t)start * p.v_stride0 + hv * kDV + row;
  const int64_t y_stride = (int64_t)p.hv * kDV;
  uint16_t* yrow = p.y + (int64_t)start * y_stride + (int64_t)hv * kDV + row;
  const uint32_t v_step = (uint32_t)p.v_stride0 * 2u, y_step = (uint32_t)y_stride * 2u;
  uint32_t v_lane = 4 * g * v_step + 2 * x16, y_lane = 4 * g * y_step + 2 * x16;
  uint32_t v[16];
  auto load_v = [&](int j) {
    const int last = end - 1 - start - j * kChunk;
    const char* base = reinterpret_cast<const char*>(vrow + (int64_t)j * kChunk * p.v_stride0);
    uint32_t off[16];
    asm volatile("" : "+v"(v_lane));  // the offsets are made here and now, not kept in 16 registers
    if (last >= kChunk - 1) {
#pragma unroll
      for (int n = 0; n < 16; ++n) off[n] = v_lane + (16 * (n >> 2) + (n & 3)) * v_step;
    } else {  // rows past the request's end: its last row (counted as zero where it is used)
#pragma unroll
      for (int n = 0; n < 16; ++n) off[n] = min(16 * (n >> 2) + 4 * g + (n & 3), last) * v_step + 2 * x16;
    }
    // in assembly: loads the compiler knows it packs in pairs, and waits for, where they are issued
#pragma unroll
    for (int n = 0; n < 16; ++n) asm volatile("global_load_ushort %0, %1, %2" : "=v"(v[n]) : "v"(off[n]), "s"(base));
  };
  auto wait_v = [&]() {
    asm volatile("s_waitcnt vmcnt(0)"
                 : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]),
                   "+v"(v[8]), "+v"(v[9]), "+v"(v[10]), "+v"(v[11]), "+v"(v[12]), "+v"(v[13]), "+v"(v[14]), "+v"(v[15]));
  };
  slot_barrier();  // K, Q of chunk 0
  slot_barrier();  // A, P of chunk 0
  slot_barrier();  // T of chunk 0

  // transposing reads of K: token 4 g + x16 / 4 of a tile, dims 8 (x16 % 4) .. of a block of 32
  const int kt_lane = (4 * g + (x16 >> 2)) * kRowPad + 8 * (x16 & 3);
  struct Rows {
    bf16x8_t k[4], q[4];
  };
  auto load_rows = [&](int par, int c, Rows& r) {
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      r.k[m] = operand(&lds.k[par][16 * m + x16][32 * c + 8 * g]);
      r.q[m] = operand(&lds.q[par][16 * m + x16][32 * c + 8 * g]);
    }
  };
  Rows rows[2];
  load_rows(0, 0, rows[0]);
  for (int j = 0, tri = 0; j < n_chunks; ++j, tri = tri == 2 ? 0 : tri + 1) {
    const int first = start + j * kChunk, par = j & 1;
    Triangle tp[2];
    // ---- slot 1 ----------------------------------------------------------------------------
    load_v(j);
    f32x4_t x[4], z[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) x[m] = z[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    Split sp = split(s[0], s[1]);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (c < 3) load_rows(par, c + 1, rows[(c + 1) & 1]);
      fence();
      const Rows& r = rows[c & 1];
      auto step = [&](bf16x8_t part) {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          x[m] = mfma_16x16x32(r.k[m], part, x[m]);
          z[m] = mfma_16x16x32(r.q[m], part, z[m]);
        }
      };
      step(sp.lo);
      step(sp.mid);
      step(sp.hi);
      if (c < 3) {
        sp = split(s[2 * c + 2], s[2 * c + 3]);
        interleave<24, 2>();
      }
      fence();
    }
    slot_barrier();
    // ---- slot 2 ----------------------------------------------------------------------------
    load_triangle(lds.t, 0, tp[0]);
    wait_v();
    if (first + kChunk > end) {
#pragma unroll
      for (int n = 0; n < 16; ++n) v[n] = first + 16 * (n >> 2) + 4 * g + (n & 3) < end ? v[n] : 0u;
    }
    f32x4_t u[4];
    {
      f32x4_t r[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const f32x4_t bet = *reinterpret_cast<const f32x4_t*>(&lds.beta[tri][16 * m + 4 * g]);
        const f32x4_t gam = *reinterpret_cast<const f32x4_t*>(&lds.gamma[tri][16 * m + 4 * g]);
#pragma unroll
        for (int i = 0; i < 4; ++i) r[m][i] = (bf16_bits_to_f32(v[4 * m + i]) - gam[i] * x[m][i]) * bet[i];
        z[m] *= gam;
        u[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
      load_triangle(lds.t, 1, tp[1]);
      const Split rs0 = split(r[0], r[1]);
      fence();
      triangle_product<0>(tp[0], rs0, u);
      const Split rs1 = split(r[2], r[3]);
      interleave<24, 2>();
      fence();
      load_triangle(lds.p, 0, tp[0]);
      triangle_product<1>(tp[1], rs1, u);
    }
    slot_barrier();
    // ---- slot 3 ----------------------------------------------------------------------------
    const uint16_t* kt = &lds.k[par][0][0] + kt_lane;
    auto load_kt = [&](int n, bf16x8_t (&ka)[4]) {  // contraction step n / 2, dims 64 (n % 2) ..
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = 4 * (n & 1) + i;
        const uint16_t* at = kt + 32 * (c >> 1) + 4 * (c & 1) + 32 * (n >> 1) * kRowPad;
        const u32x2_t a0 = lds_read_tr16(reinterpret_cast<const unsigned char*>(at));
        const u32x2_t a1 = lds_read_tr16(reinterpret_cast<const unsigned char*>(at + 16 * kRowPad));
        ka[i] = as_bf16x8(u32x4_t{a0[0], a0[1], a1[0], a1[1]});
      }
    };
    load_triangle(lds.p, 1, tp[1]);
    {
      const Split us0 = split(u[0], u[1]);
      fence();
      triangle_product<0>(tp[0], us0, z);
      const Split us1 = split(u[2], u[3]);
      interleave<24, 2>();
      fence();
      bf16x8_t ka[2][4];
      load_kt(0, ka[0]);
      f32x4_t tail[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) tail[m] = *reinterpret_cast<const f32x4_t*>(&lds.tail[tri][16 * m + 4 * g]);
      const float total = lds.total[tri];
      triangle_product<1>(tp[1], us1, z);
#pragma unroll
      for (int c = 0; c < 8; ++c) s[c] *= total;
      const Split ut0 = split(u[0] * tail[0], u[1] * tail[1]);
      interleave<12, 5>();
      fence();
      auto step = [&](int n, bf16x8_t part) {
#pragma unroll
        for (int i = 0; i < 4; ++i) s[4 * (n & 1) + i] = mfma_16x16x32(ka[n & 1][i], part, s[4 * (n & 1) + i]);
      };
      auto steps = [&](int n, const Split& b) {
        step(n, b.lo);
        step(n, b.mid);
        step(n, b.hi);
      };
      load_kt(1, ka[1]);
      steps(0, ut0);
      const Split ut1 = split(u[2] * tail[2], u[3] * tail[3]);
      interleave<12, 4>();
      fence();
      load_kt(2, ka[0]);
      steps(1, ut0);
      fence();
      load_kt(3, ka[1]);
      steps(2, ut1);
      fence();
      load_rows(par ^ 1, 0, rows[0]);  // of chunk j + 1 (of no use behind the last chunk)
      steps(3, ut1);
      char* base = reinterpret_cast<char*>(yrow + (int64_t)j * kChunk * y_stride);
      asm volatile("" : "+v"(y_lane));
      const bool whole = first + kChunk <= end;
#pragma unroll
      for (int n = 0; n < 16; ++n) {
        const uint16_t bits = __builtin_bit_cast(uint16_t, (__bf16)z[n >> 2][n & 3]);
        uint16_t* to = reinterpret_cast<uint16_t*>(base + (y_lane + (16 * (n >> 2) + (n & 3)) * y_step));
        if (whole) *to = bits;
        else if (first + 16 * (n >> 2) + 4 * g + (n & 3) < end) *to = bits;
      }
    }
    slot_barrier();
  }
#pragma unroll
  for (int c = 0; c < 8; ++c) *reinterpret_cast<f32x4_t*>(srow + 32 * (c >> 1) + 4 * (c & 1)) = s[c];
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

// Column block W of T below the diagonal: T_rW = -T_rr X_r, X_r = sum over W <= k < r of A_rk T_kW.  T_rW is
// made twice, as the operand of the rows below it and transposed, four neighbours of a row to a lane, for
// LDS.  Everything the chain needs from LDS is asked for before it starts.
template <int W>
__device__ __forceinline__ void column_block(ChunkLds& lds) {
  const int x16 = lane_id() & 15, g = lane_id() >> 4;
  f32x4_t a[4][4], d[4], tk[4];
#pragma unroll
  for (int n = 0; n < 4; ++n) tk[W][n] = lds.diag[W][4 * g + n][x16];
#pragma unroll
  for (int r = W + 1; r < 4; ++r) {
#pragma unroll
    for (int k = W; k < r; ++k) a[r][k] = *reinterpret_cast<const f32x4_t*>(&lds.a[16 * r + x16][16 * k + 4 * g]);
    d[r] = *reinterpret_cast<const f32x4_t*>(&lds.diag[r][x16][4 * g]);
  }
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  f32x4_t x[4];
#pragma unroll
  for (int r = W + 1; r < 4; ++r) x[r] = mfma_f32_block(a[r][W], tk[W], zero);
#pragma unroll
  for (int r = W + 1; r < 4; ++r) {
    const f32x4_t minus = -d[r];
    if (r < 3) {
      tk[r] = mfma_f32_block(minus, x[r], zero);
#pragma unroll
      for (int n = r + 1; n < 4; ++n) x[n] = mfma_f32_block(a[n][r], tk[r], x[n]);
    }
    split_store(mfma_f32_block(x[r], minus, zero), lds.t, 16 * r + x16, token_column(W, g));
  }
}

__device__ __forceinline__ void chunk_waves(const GdnParams& p, ChunkLds& lds, int start, int end, int hv, int w) {
  const int lane = lane_id(), x16 = lane & 15, g = lane >> 4;
  const int n_chunks = (end - start + kChunk - 1) / kChunk;
  const int hk = hv / p.hv_per_hk;
  // this wave's 16 tokens of K and Q, four rows per load, and every token's gates: scalar bases at the
  // request's first token, 32-bit offsets
  const char* kbase = reinterpret_cast<const char*>(p.k + (int64_t)start * p.k_stride0 + hk * kDK);
  const char* qbase = reinterpret_cast<const char*>(p.q + (int64_t)start * p.q_stride0 + hk * kDK);
  const char* gbase = reinterpret_cast<const char*>(p.g + (int64_t)start * p.hv + hv);
  const char* bbase = reinterpret_cast<const char*>(p.beta + (int64_t)start * p.hv + hv);
  const uint32_t k_step = (uint32_t)p.k_stride0 * 2u, q_step = (uint32_t)p.q_stride0 * 2u, g_step = (uint32_t)p.hv * 2u;
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
      *reinterpret_cast<u32x4_t*>(&lds.k[par][t][8 * x16]) = in ? kr[n] : zero;
      *reinterpret_cast<u32x4_t*>(&lds.q[par][t][8 * x16]) = in ? qr[n] : zero;
    }
  };
  // decay products of a chunk from the gates fetched with it: the last wave's work, it has the least to do
  // beside T
  auto decays = [&](int first, int tri) {
    const bool in = first + lane < end;
    const float gv = in ? bf16_bits_to_f32(graw) : 1.0f, bv = in ? bf16_bits_to_f32(braw) : 0.0f;
    float pre = gv, suf = gv, quad_pre = gv;
#pragma unroll
    for (int n = 1; n < 16; n <<= 1) {
      const float a = __shfl_up(pre, n, 16), b = __shfl_down(suf, n, 16);
      if (n < 4) {
        const float q = __shfl_up(quad_pre, n, 4);
        if ((x16 & 3) >= n) quad_pre *= q;
      }
      if (x16 >= n) pre *= a;
      if (x16 + n < 16) suf *= b;
    }
    const float after = __shfl_down(suf, 1, 16);
    suf = x16 == 15 ? 1.0f : after;
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
  // The ten blocks (r, c) of A and P on and below the diagonal: every wave its diagonal block, waves 0-2
  // two more.  Results are transposed (lane: token t = 16 r + x16, tokens i = 16 c + 4 g + n), so that a
  // lane's four values are neighbours in a row of A and of P.
  const int n_blocks = w == 3 ? 1 : 3;
  auto block_row = [&](int n) { return n == 0 ? w : n == 1 ? (w == 0 ? 3 : w) : (w == 2 ? 2 : 3); };
  auto block_col = [&](int n) { return n == 0 ? w : n == 1 ? 0 : (w == 1 ? 2 : 1); };
  f32x4_t pp[3];  // P of these blocks
  f32x4_t inv;    // the inverse of the diagonal block: row x16, columns 4 g ..
  auto products = [&](int par, int tri) {
    struct Block {
      bf16x8_t kc[4], kr[4], qr[4];
      f32x4_t col;
      float row, beta;
    };
    auto load = [&](int r, int c, Block& x) {
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        x.kc[d] = operand(&lds.k[par][16 * c + x16][32 * d + 8 * g]);
        x.kr[d] = operand(&lds.k[par][16 * r + x16][32 * d + 8 * g]);
        x.qr[d] = operand(&lds.q[par][16 * r + x16][32 * d + 8 * g]);
      }
      x.beta = lds.beta[tri][16 * r + x16];
      x.row = r == c ? lds.quad_pre[16 * r + x16] : lds.pre[16 * r + x16];
      x.col = *reinterpret_cast<const f32x4_t*>(r == c ? &lds.g[16 * r + 4 * g] : &lds.suf[16 * c + 4 * g]);
    };
    auto dots = [&](const Block& x, f32x4_t& kk, f32x4_t& qk) {
      kk = qk = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        kk = mfma_16x16x32(x.kc[d], x.kr[d], kk);
        qk = mfma_16x16x32(x.kc[d], x.qr[d], qk);
      }
    };
    // G_t / G_i of a block below the diagonal: token t's block up to it, whole blocks, token i's block behind it
    auto below = [&](int n, int r, int c, const Block& x, const f32x4_t& kk, const f32x4_t& qk) {
      float row = x.row;
      if (c < 1 && r > 1) row *= lds.block[1];
      if (c < 2 && r > 2) row *= lds.block[2];
      const f32x4_t ratio = row * x.col;
      pp[n] = ratio * qk;
      *reinterpret_cast<f32x4_t*>(&lds.a[16 * r + x16][16 * c + 4 * g]) = x.beta * ratio * kk;
    };
    Block b0, b1, b2;
    f32x4_t kk0, qk0, kk1, qk1, kk2, qk2;
    const int r1 = block_row(1), c1 = block_col(1), r2 = block_row(2), c2 = block_col(2);
    load(w, w, b0);
    if (n_blocks > 1) load(r1, c1, b1);
    dots(b0, kk0, qk0);
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
        pp[0][i] = 4 * g + i <= x16 ? ratio[i] * qk0[i] : 0.f;
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
    if (n_blocks > 1) {
      load(r2, c2, b2);
      dots(b1, kk1, qk1);
      dots(b2, kk2, qk2);
      eliminate<0>(arow, inv);
      below(1, r1, c1, b1, kk1, qk1);
      below(2, r2, c2, b2, kk2, qk2);
    } else {
      eliminate<0>(arow, inv);
    }
    *reinterpret_cast<f32x4_t*>(&lds.diag[w][x16][4 * g]) = inv;
  };
  auto inverse = [&]() {
    split_store(inv, lds.t, 16 * w + x16, token_column(w, g));
    if (w == 0) column_block<0>(lds);
    else if (w == 1) column_block<1>(lds);
    else if (w == 2) column_block<2>(lds);
  };
  auto store_p = [&]() {
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      if (n >= n_blocks) break;
      split_store(pp[n], lds.p, 16 * block_row(n) + x16, token_column(block_col(n), g));
    }
  };

  fetch(start);
  stage(start, 0);
  if (w == 3) decays(start, 0);
  slot_barrier();
  if (n_chunks > 1) fetch(start + kChunk);
  products(0, 0);
  slot_barrier();
  inverse();
  if (w == 3 && n_chunks > 1) decays(start + kChunk, 1);
  slot_barrier();
  int tri = 1;  // of chunk j + 1, modulo 3
  for (int j = 0; j < n_chunks; ++j) {
    const int next = start + (j + 1) * kChunk, par = (j + 1) & 1;
    const bool more = j + 1 < n_chunks, two = j + 2 < n_chunks;
    store_p();
    if (more) stage(next, par);
    if (two) fetch(next + kChunk);
    slot_barrier();
    if (more) products(par, tri);
    slot_barrier();
    tri = tri == 2 ? 0 : tri + 1;
    if (more) inverse();
    if (w == 3 && two) decays(next + kChunk, tri);
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
  if (wave < 4) state_waves(p, lds, start, end, p.slot_ids[b], hv, row + 16 * wave);
  else chunk_waves(p, lds, start, end, hv, wave - 4);
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
