// Gated delta rule over requests of many chunks: the chunks' triangular systems in a launch of their own, all in
// parallel, then the serial part alone.  Notation, layouts, precision and what happens to infinities: gdn_chunk.hip, which does both in
// one launch; results are the same bits.
//
// In one launch every workgroup of a value head, two or four of them, makes the systems of all its chunks beside the serial part, and
// its waves share SIMDs and LDS with those of the chain that the launch waits for: 7.7 K cycles a chunk.  Here a system is made once,
// and the chain is short: 5.2 K cycles a chunk where a request has four workgroups a value head, 7.6 K with two.
//
// gdn_systems_kernel: one workgroup per chunk and value head; 17 us for 63 chunks of 32 heads, 29 us for 130 (before its 15 KiB of A
// and inverses shared their place with K and T and three workgroups more fitted a compute unit: 21 and 37).  Bound by the
// round trips to memory in front of its 5 K cycles of work (its request, K, the gates), then by its stores (3 TB/s).
// gdn_serial_kernel: quarters by the chain of a state wave, 4.7 K of the 5.2 K cycles, 2.6 K of them matrix instructions, at 2.3 GHz (the
// pipe is busy for 23 % of the SIMD cycles with one request, 43 % with the four below); halves where many requests fill the chip by the
// matrix pipe: 1.12-1.15 PFLOP/s of bf16 products at 2.1 GHz, where a large product reaches 1.24.
//
// Both against the one launch, us: one request of 4005 tokens 208 -> 156; of 992, 1581, 4005 and 1601 tokens 232 -> 178; 2000 among five
// short ones 146 -> 95; eight of 1000 158 -> 156.
#include "gdn_chunk_tiles.h"

namespace msgl {
namespace {

// What the serial part needs of a chunk and value head beside k, q and v: its products of decays, and T as operands.
struct Gates {
  float beta[kChunk], gamma[kChunk], tail[kChunk], g[kChunk], pre[kChunk], suf[kChunk], quad_pre[kChunk];  // see ChunkLds
  float block[4], quad[16], total, unused[43];
};
struct ChunkRecord {
  u32x4_t t[3][kFragments][64];
  Gates gates;
};
static_assert(sizeof(Gates) == 2048 && sizeof(ChunkRecord) == 20480, "copied in whole KiB");

// Records of a launch, [chunk][value head]: request b's chunks from start_b / 64 + b on, which leaves room for its last one.
__device__ __forceinline__ int first_record(int start, int b) { return (int)((uint32_t)start / kChunk) + b; }

// The ten blocks of A on and below the diagonal: those on it, then (1, 0), (2, 0), (2, 1), (3, 0), (3, 1), (3, 2)
__device__ constexpr int block_at(int r, int c) { return r == c ? r : 4 + r * (r - 1) / 2 + c; }
struct SystemsLds : Gates {  // (Decays and Inverse name the arrays)
  union {  // one after the other
    uint16_t k[kChunk][kDK];
    float a[10][16][20];  // A's blocks, those on the diagonal -A and then their inverses
    u32x4_t t[3][kFragments][64];
  };
  __device__ __forceinline__ const float* a_row(int r, int c, int row) const { return a[block_at(r, c)][row]; }
  __device__ __forceinline__ const float* diagonal_row(int r, int row) const { return a[r][row]; }
};

__global__ __launch_bounds__(256, 7) void gdn_systems_kernel(GdnParams p, ChunkRecord* records, int chunks) {
  __shared__ SystemsLds lds;
  const int lane = lane_id(), x16 = lane & 15, g = lane >> 4;
  // Workgroup -> (chunk, key head, value head of it): those of one key head get ids of one residue modulo 8, so one L2 serves them
  const int hk_n = p.hv / p.hv_per_hk;
  const int seq = blockIdx.x >> 3, group = (seq / p.hv_per_hk) * 8 + (blockIdx.x & 7);
  // the four waves have unlike amounts of work: they change places from workgroup to workgroup, so that no SIMD gets the longest of all
  const int w = __builtin_amdgcn_readfirstlane(((threadIdx.x >> 6) + seq) & 3);
  if (group >= chunks * hk_n) return;
  const int chunk = group / hk_n, hk = group - chunk * hk_n, hv = hk * p.hv_per_hk + seq % p.hv_per_hk;
  int first = -1, end = 0;
  for (int b0 = 0; b0 < p.batch && first < 0; b0 += kWave) {
    const int b = min(b0 + lane, p.batch - 1);
    const int from = p.qo_indptr[b], to = min(p.qo_indptr[b + 1], p.tokens);
    const int at = chunk - first_record(from, b);
    const uint64_t hit = __ballot(b0 + lane < p.batch && at >= 0 && at * kChunk < to - from);
    if (hit) {
      const int src = __builtin_ctzll(hit);
      first = __builtin_amdgcn_readlane(from, src) + __builtin_amdgcn_readlane(at, src) * kChunk;
      end = __builtin_amdgcn_readlane(to, src);
    }
  }
  if (first < 0) return;  // room behind a request's last chunk: the whole workgroup
  const uint16_t* kbase = p.k + (int64_t)first * p.k_stride0 + hk * kDK;
  const uint32_t last = end - 1 - first;
  uint32_t graw = 0, braw = 0;  // a token per lane
  if (w == 3) {
    const int64_t token = (int64_t)(first + min((uint32_t)lane, last)) * p.hv + hv;
    graw = p.g[token];
    braw = p.beta[token];
  }
  u32x4_t kr[4];  // four whole rows a load (as operands, from 16 rows at once, a load takes four times as long)
#pragma unroll
  for (int n = 0; n < 4; ++n) kr[n] = ld_global_b128(kbase + (int64_t)min((uint32_t)(16 * w + 4 * n + g), last) * p.k_stride0 + 8 * x16);
  if (w == 3) {
    const bool in = first + lane < end;
    decay_products(lds, in ? bf16_bits_to_f32(graw) : 1.0f, in ? bf16_bits_to_f32(braw) : 0.0f, lds.beta, lds.gamma, lds.tail, lds.total);
  }
#pragma unroll
  for (int n = 0; n < 4; ++n) {  // rows past the request's end are zero
    const int t = 16 * w + 4 * n + g;
    *reinterpret_cast<u32x4_t*>(&lds.k[t][8 * piece(t, x16)]) = first + t < end ? kr[n] : u32x4_t{0u, 0u, 0u, 0u};
  }
  __syncthreads();
  // A: every wave its diagonal block and one more, waves 1 and 2 two
  const bool two = w == 1 || w == 2;
  const int r1 = w == 0 ? 3 : w, c1 = w == 3 ? 1 : 0, r2 = w + 1, c2 = w;
  f32x4_t kk0, kk1, kk2 = {0.f, 0.f, 0.f, 0.f};
  {
    bf16x8_t own[4], other[4], third[4];  // rows of block w, of the other one of (r1, c1), of r2
    load_block_rows(lds.k, w, own);
    load_block_rows(lds.k, w == 0 ? 3 : c1, other);
    if (two) load_block_rows(lds.k, r2, third);
    kk0 = block_dots(own, own);
    kk1 = w == 0 ? block_dots(own, other) : block_dots(other, own);
    if (two) kk2 = block_dots(own, third);
  }
  __syncthreads();
  f32x4_t inv;
  {
    auto store_below = [&](int r, int c, f32x4_t dots) {
      Decays decays;
      decays.load(lds, r, c);
      *reinterpret_cast<f32x4_t*>(&lds.a[block_at(r, c)][x16][4 * g]) = lds.beta[16 * r + x16] * decays.below(lds, r, c) * dots;
    };
    Decays decays;
    decays.load(lds, w, w);
    const float beta = lds.beta[16 * w + x16];
    const f32x4_t ratio = decays.diagonal(lds, w);
    f32x4_t a;
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = 4 * g + i < x16 ? -beta * ratio[i] * kk0[i] : 0.f;  // negated, as eliminate() takes it
    float* const own = lds.a[w][x16];
    *reinterpret_cast<f32x4_t*>(own + 4 * g) = a;
    float arow[16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4_t four = *reinterpret_cast<const f32x4_t*>(own + 4 * i);
#pragma unroll
      for (int e = 0; e < 4; ++e) arow[4 * i + e] = four[e];
    }
#pragma unroll
    for (int n = 0; n < 4; ++n) inv[n] = x16 == 4 * g + n ? 1.0f : 0.0f;
    store_below(r1, c1, kk1);
    if (two) store_below(r2, c2, kk2);
    eliminate<0>(arow, inv);
    *reinterpret_cast<f32x4_t*>(own + 4 * g) = inv;
  }
  __syncthreads();
  const Below below = blocks_below<false>(lds, w);
  __syncthreads();
  const Picker pick;
  split_store(pick, inv, lds.t, w, w);
  const int r = w == 0 ? 1 : w == 1 ? 2 : 3, c = w == 1 ? 1 : w == 2 ? 2 : 0;
  split_store(pick, below.first, lds.t, r, c);
  if (w < 2) split_store(pick, below.second, lds.t, r + 1, c);
  else split_store(pick, f32x4_t{0.f, 0.f, 0.f, 0.f}, lds.t, w == 2 ? 0 : 2, w == 2 ? 1 : 3);  // read beside the diagonal blocks
  __syncthreads();
  u32x4_t* to = reinterpret_cast<u32x4_t*>(records + (int64_t)chunk * p.hv + hv);
  constexpr int kT = sizeof(lds.t) / 16;
#pragma unroll
  for (int i = 0; i < (int)sizeof(ChunkRecord) / 16 / 256; ++i) {
    const int at = threadIdx.x + 256 * i;
    to[at] = at < kT ? (&lds.t[0][0][0])[at] : reinterpret_cast<const u32x4_t*>(static_cast<const Gates*>(&lds))[at - kT];
  }
}

// ---- the serial part ----------------------------------------------------------------------------------------
// How a request is spread: its heads in halves or in quarters of their 128 rows, a workgroup each.
//   halves   four waves of 16 rows, each with all that its rows take (X, Z, R, U, Y, S), four that fetch and make P
//   quarters two state waves with X, R, U and S, two output waves with Z and Y, four that fetch and make P
// (Whole heads, eight waves of the first kind, take as long as two halves one after the other: the matrix pipe has no room.)
// A chunk's data come in by themselves while the chunk before is worked on.
template <int ROWS>
struct SerialLds {
  uint16_t k[2][kChunk][kDK], q[2][kChunk][kDK];
  uint16_t v[2][kChunk][ROWS];
  u32x4_t t[ROWS == 32 ? 1 : 2][3][kFragments][64], p[3][kFragments][64];
  Gates gates[2];
  alignas(16) float p_largest[4 * 64];
};
struct QuarterLds : SerialLds<32> {
  f32x4_t s[2][2][8][64], u[2][4][64];  // a state wave's S, before chunk j in s[j % 2], and U for its output wave
};
static_assert(sizeof(SerialLds<64>) <= 160 * 1024 && sizeof(QuarterLds) <= 160 * 1024, "LDS of a compute unit");

// A chunk's data to LDS, 1 KiB a load.  Rows past the request's end: its last row (beta is zero there, and their rows of Y
// are not stored).
template <int ROWS>
struct Fetch {
  const char *k, *q, *v, *records;
  uint32_t k_step, q_step, v_step, record_step;
  int tokens;
  uint32_t to_k, to_q, to_v, to_t, to_gates;
  template <typename Lds>
  __device__ __forceinline__ Fetch(const GdnParams& p, const ChunkRecord* rec, Lds& lds, int b, int start, int end, int hv, int row)
      : k_step((uint32_t)p.k_stride0 * 2u), q_step((uint32_t)p.q_stride0 * 2u), v_step((uint32_t)p.v_stride0 * 2u),
        record_step((uint32_t)p.hv * (uint32_t)sizeof(ChunkRecord)), tokens(end - start) {
    const int hk = hv / p.hv_per_hk;
    k = reinterpret_cast<const char*>(p.k + (int64_t)start * p.k_stride0 + hk * kDK);
    q = reinterpret_cast<const char*>(p.q + (int64_t)start * p.q_stride0 + hk * kDK);
    v = reinterpret_cast<const char*>(p.v + (int64_t)start * p.v_stride0 + hv * kDV + row);
    records = reinterpret_cast<const char*>(rec + (int64_t)first_record(start, b) * p.hv + hv);
    // (the low half of such an address is its place in LDS)
    auto place = [](const void* at) { return (uint32_t)reinterpret_cast<uintptr_t>(at); };
    to_k = place(&lds.k[0][0][0]);
    to_q = place(&lds.q[0][0][0]);
    to_v = place(&lds.v[0][0][0]);
    to_t = place(&lds.t[0][0][0][0]);
    to_gates = place(&lds.gates[0]);
  }
  static __device__ __forceinline__ void load(uint32_t to, const char* base, uint32_t at) {
    lds_direct_b128(__builtin_amdgcn_readfirstlane(to), base, at);
  }
  __device__ __forceinline__ uint32_t row(int chunk, int t) const { return min((uint32_t)t, (uint32_t)(tokens - 1 - chunk * kChunk)); }
  // rows of 256 bytes, four a load, load n of 16
  __device__ __forceinline__ void rows(const char* base, uint32_t step, uint32_t to, int chunk, int n) const {
    const int t = 4 * n + (lane_id() >> 4);
    load(to + (chunk & 1) * (kChunk * kDK * 2u) + 1024 * n, base + (int64_t)chunk * kChunk * step,
         row(chunk, t) * step + 16 * piece(t, lane_id() & 15));
  }
  __device__ __forceinline__ void k_rows(int chunk, int n) const { rows(k, k_step, to_k, chunk, n); }
  __device__ __forceinline__ void q_rows(int chunk, int n) const { rows(q, q_step, to_q, chunk, n); }
  __device__ __forceinline__ void v_rows(int chunk, int n) const {  // load n of ROWS / 8
    constexpr int kLanes = ROWS / 8;  // a token
    const int lane = lane_id(), t = n * (64 / kLanes) + lane / kLanes;
    load(to_v + (chunk & 1) * (kChunk * ROWS * 2u) + 1024 * n, v + (int64_t)chunk * kChunk * v_step, row(chunk, t) * v_step + 16 * (lane % kLanes));
  }
  __device__ __forceinline__ void t_part(int chunk, int n) const {  // of 18
    constexpr uint32_t kSize = sizeof(ChunkRecord) - sizeof(Gates);
    load(to_t + (ROWS == 32 ? 0 : (chunk & 1) * kSize) + 1024 * n, records + (int64_t)chunk * record_step, 1024 * n + 16 * lane_id());
  }
  __device__ __forceinline__ void gates(int chunk, int n) const {  // of 2
    load(to_gates + (chunk & 1) * (uint32_t)sizeof(Gates) + 1024 * n, records + (int64_t)chunk * record_step,
         (uint32_t)(sizeof(ChunkRecord) - sizeof(Gates)) + 1024 * n + 16 * lane_id());
  }
  // Everything of a chunk but T, by wave w of four: 9 loads, gates in front of them
  __device__ __forceinline__ void four_waves(int chunk, int w) const {
    if (w >= 2) gates(chunk, w - 2);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      k_rows(chunk, 4 * w + i);
      q_rows(chunk, 4 * w + i);
    }
#pragma unroll
    for (int i = 0; i < ROWS / 32; ++i) v_rows(chunk, (ROWS / 32) * w + i);
  }
  __device__ __forceinline__ void t_four_waves(int chunk, int w) const {
#pragma unroll
    for (int i = 0; i < 4; ++i) t_part(chunk, 4 * w + i);
    if (w < 2) t_part(chunk, 16 + w);
  }
};

// Block (r, c) of P: what it is made of is asked for apart, so that several blocks' reads are under way together.
struct BlockOfP {
  bf16x8_t k[4], q[4];
  Decays decays;
  template <typename Lds>
  __device__ __forceinline__ void load(const Lds& lds, int par, int r, int c) {
    load_block_rows(lds.k[par], c, k);
    load_block_rows(lds.q[par], r, q);
    decays.load(lds.gates[par], r, c);
  }
  __device__ __forceinline__ f32x4_t below(const Gates& gates, int r, int c) const { return decays.below(gates, r, c) * block_dots(k, q); }
  __device__ __forceinline__ f32x4_t diagonal(const Gates& gates, int r) const {
    const int x16 = lane_id() & 15, g = lane_id() >> 4;
    const f32x4_t dots = block_dots(k, q);
    f32x4_t ratio = decays.diagonal(gates, r);
#pragma unroll
    for (int i = 0; i < 4; ++i) ratio[i] = 4 * g + i <= x16 ? ratio[i] : 0.f;
    return ratio * dots;
  }
};
// Block n of P: those on the diagonal, then (1, 0), (2, 0), (2, 1), (3, 0), (3, 1), (3, 2)
__device__ __forceinline__ int row_of_block(int n) { return n < 4 ? n : n == 4 ? 1 : n < 7 ? 2 : 3; }
__device__ __forceinline__ int column_of_block(int n) { return n < 4 ? n : n == 4 ? 0 : n < 7 ? n - 5 : n - 7; }

// Places of K's and Q's pieces in LDS, as operands (row x16) and transposed (row 4 g + x16 / 4), per 32 dims.
struct Places {
  uint32_t at[4], transposed[4];
  __device__ __forceinline__ Places() {
    const int x16 = lane_id() & 15, g = lane_id() >> 4, trow = 4 * g + (x16 >> 2);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      at[c] = x16 * kDK + 8 * piece(x16, 4 * c + g);
      transposed[c] = trow * kDK + 8 * piece(trow, 4 * c + (x16 & 3));
    }
  }
};
__device__ __forceinline__ void load_operands(const uint16_t (*m)[kDK], uint32_t at, bf16x8_t (&x)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = operand(&m[16 * i][0] + at);
}
// K transposed: tokens 32 (n % 2) .., dims 64 (n / 2) ..
__device__ __forceinline__ void load_transposed(const uint16_t (*m)[kDK], const Places& places, int n, bf16x8_t (&x)[4]) {
  const uint16_t* k = &m[0][0];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = 4 * (n >> 1) + i;
    const uint16_t* a = k + places.transposed[c >> 1] + 4 * (c & 1) + 32 * (n & 1) * kDK;
    const u32x2_t a0 = lds_read_tr16(reinterpret_cast<const unsigned char*>(a));
    const u32x2_t a1 = lds_read_tr16(reinterpret_cast<const unsigned char*>(a + 16 * kDK));
    x[i] = as_bf16x8(u32x4_t{a0[0], a0[1], a1[0], a1[1]});
  }
}

// A wave's 16 state rows and what it does with them.
struct StateRows {
  f32x4_t s[8];  // s[2 c + h][i]: dim 32 c + 8 g + 4 h + i of row `row + x16`
  __device__ __forceinline__ void load(int slot, int hv, int row) {
    const float* from = state_row(slot, hv, row);
#pragma unroll
    for (int c = 0; c < 8; ++c) s[c] = *reinterpret_cast<const f32x4_t*>(from + 32 * (c >> 1) + 4 * (c & 1));
  }
  __device__ __forceinline__ void store(int slot, int hv, int row) const {
    float* to = state_row(slot, hv, row);
#pragma unroll
    for (int c = 0; c < 8; ++c) *reinterpret_cast<f32x4_t*>(to + 32 * (c >> 1) + 4 * (c & 1)) = s[c];
  }
};

// R = beta (V - G X) of a wave's rows, from column `column` of V on: half h of the tokens, as operand.
struct ForR {
  f32x4_t beta[2], gamma[2];
  u32x2_t v[2];
  template <typename Lds>
  __device__ __forceinline__ void load(const Lds& lds, int par, int column, int h) {
    const int x16 = lane_id() & 15, g = lane_id() >> 4, trow = 4 * g + (x16 >> 2);
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      v[m] = lds_read_tr16(reinterpret_cast<const unsigned char*>(&lds.v[par][16 * (2 * h + m) + trow][column + 4 * (x16 & 3)]));
      beta[m] = *reinterpret_cast<const f32x4_t*>(&lds.gates[par].beta[16 * (2 * h + m) + 4 * g]);
      gamma[m] = *reinterpret_cast<const f32x4_t*>(&lds.gates[par].gamma[16 * (2 * h + m) + 4 * g]);
    }
  }
  __device__ __forceinline__ Split make(const Picker& pick, const f32x4_t* x) const {
    f32x4_t r[2];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        r[m][i] = (bf16_bits_to_f32(i & 1 ? v[m][i >> 1] >> 16 : v[m][i >> 1] & 0xffffu) - gamma[m][i] * x[m][i]) * beta[m][i];
    return split(pick, r[0], r[1]);
  }
};
// Half h of U weighed by tail, as operand
__device__ __forceinline__ Split weigh(const Picker& pick, const Gates& gates, const f32x4_t (&u)[4], int h) {
  f32x4_t tail[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) tail[m] = *reinterpret_cast<const f32x4_t*>(&gates.tail[16 * (2 * h + m) + 4 * (lane_id() >> 4)]);
  return split(pick, u[2 * h] * tail[0], u[2 * h + 1] * tail[1]);
}
// N matrix instructions of what lies between two fences, V vector instructions behind each of them: what does not wait for
// the matrix pipe goes out while it is busy.  (Four, the instruction slots of a matrix instruction, so that the chain of a split,
// conversions that wait for products, begins with most of the products still to come: one of 4005 tokens 162 -> 160 us with them than with two.)
template <int N, int V>
__device__ __forceinline__ void weave() {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, V, 0);
  }
}
// s += K^T U for dims 64 (n / 2) .., tokens 32 (n % 2) ..
__device__ __forceinline__ void state_steps(f32x4_t (&s)[8], const bf16x8_t (&k)[4], int n, const Split& u) {
  auto step = [&](bf16x8_t part) {
#pragma unroll
    for (int i = 0; i < 4; ++i) s[4 * (n >> 1) + i] = mfma_16x16x32(k[i], part, s[4 * (n >> 1) + i]);
  };
  step(u.lo);
  step(u.mid);
  step(u.hi);
}

// The end of a wave with state rows: `most` is the largest magnitude of its U, p_largest of P.
template <typename Lds>
__device__ __forceinline__ void finish_rows(const Lds& lds, const StateRows& rows, float most, int start, int end, int slot, int hv, int row) {
  most = largest(*reinterpret_cast<const f32x4_t*>(&lds.p_largest[4 * lane_id()]), most);
  if (__builtin_expect(!__all(splits(most)), 0)) {
    wait_all_vm();  // the stores of Y: the same places are written again
    token_by_token(start, end, slot, hv, row);
    return;
  }
  rows.store(slot, hv, row);
}

// Halves: a wave with its rows and all that they take.
//     part 1   X, Z, R, U; P to LDS        part 2   Y, S
__device__ __forceinline__ void half_rows(const GdnParams& p, SerialLds<64>& lds, int start, int end, int slot, int hv, int row, int column) {
  const int lane = lane_id(), x16 = lane & 15;
  const int n_chunks = (end - start + kChunk - 1) / kChunk;
  StateRows rows;
  rows.load(slot, hv, row);
  f32x4_t (&s)[8] = rows.s;
  const Outputs y(p, start, end, hv, row);
  const Picker pick;
  const Places places;
  float most = 0.f;
  slot_barrier();
  for (int j = 0; j < n_chunks; ++j) {
    const int par = j & 1;
    const Gates& gates = lds.gates[par];
    // ---- X = K S^T, Z = Q S^T (transposed: a lane's four values are neighbours in a row of Y), U = T R
    bf16x8_t kk[2][4], qq[2][4];
    load_operands(lds.k[par], places.at[0], kk[0]);
    load_operands(lds.q[par], places.at[0], qq[0]);
    Split sp = split(pick, s[0], s[1]);
    f32x4_t x[4], z[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) x[m] = z[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (c < 3) {
        load_operands(lds.k[par], places.at[c + 1], kk[(c + 1) & 1]);
        load_operands(lds.q[par], places.at[c + 1], qq[(c + 1) & 1]);
      }
      fence();
      auto step = [&](bf16x8_t part) {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          x[m] = product<false>(kk[c & 1][m], part, x[m]);
          z[m] = product<true>(qq[c & 1][m], part, z[m]);
        }
      };
      const Split now = sp;
      step(now.lo);
      if (c < 3) sp = split(pick, s[2 * c + 2], s[2 * c + 3]);
      step(now.mid);
      step(now.hi);
      fence();
    }
    Triangle tp;
    load_triangle<0, 6>(lds.t[par], tp);
    ForR f0, f1;
    f0.load(lds, par, column, 0);
    f1.load(lds, par, column, 1);
    const Split r0 = f0.make(pick, x), r1 = f1.make(pick, x + 2);
    f32x4_t u[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) u[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    triangle_first<false>(tp, r0, u);
    triangle_second<false>(tp, r1, u);
#pragma unroll
    for (int m = 0; m < 4; ++m) z[m] *= gates.gamma[16 * m + x16];
    slot_barrier();  // P
    // ---- Y = G Z + P U, S = G_64 S + K^T U
    load_triangle<0, 6>(lds.p, tp);
    bf16x8_t kt[2][4];
    load_transposed(lds.k[par], places, 0, kt[0]);
    load_transposed(lds.k[par], places, 1, kt[1]);
    const Split u0 = split(pick, u[0], u[1]), u1 = split(pick, u[2], u[3]);
    fence();
    triangle_first<true>(tp, u0, z);
    const Split ut0 = weigh(pick, gates, u, 0), ut1 = weigh(pick, gates, u, 1);
    const float total = gates.total;
#pragma unroll
    for (int c = 0; c < 8; ++c) s[c] *= total;
#pragma unroll
    for (int m = 0; m < 4; ++m) most = largest(u[m], most);
    fence();
    triangle_second<true>(tp, u1, z);
    state_steps(s, kt[0], 0, ut0);
    fence();
    load_transposed(lds.k[par], places, 2, kt[0]);
    state_steps(s, kt[1], 1, ut1);
    fence();
    load_transposed(lds.k[par], places, 3, kt[1]);
    state_steps(s, kt[0], 2, ut0);
    y.store(j, z);
    fence();
    state_steps(s, kt[1], 3, ut1);
    slot_barrier();
  }
  finish_rows(lds, rows, most, start, end, slot, hv, row);
}
// P by four waves: wave w has its diagonal block and one of (1, 0), (2, 0), (2, 1), (3, 0), the last two also (3, 1) and (3, 2).
struct BlocksOfP {
  f32x4_t one, two;
  template <typename Lds>
  __device__ __forceinline__ f32x4_t make(const Lds& lds, int par, int w) {
    const int r = row_of_block(4 + w), c = column_of_block(4 + w);
    const Gates& gates = lds.gates[par];
    BlockOfP b0, b1, b2;
    b0.load(lds, par, w, w);
    b1.load(lds, par, r, c);
    if (w < 2) {
      one = b1.below(gates, r, c);
      return b0.diagonal(gates, w);
    }
    b2.load(lds, par, 3, w - 1);
    one = b1.below(gates, r, c);
    two = b2.below(gates, 3, w - 1);
    return b0.diagonal(gates, w);
  }
  __device__ __forceinline__ void store(const Picker& pick, f32x4_t diagonal, u32x4_t (*p)[kFragments][64], int w) const {
    split_store(pick, diagonal, p, w, w);
    split_store(pick, one, p, row_of_block(4 + w), column_of_block(4 + w));
    if (w >= 2) split_store(pick, two, p, 3, w - 1);
  }
};
// Halves: what the row waves don't do, by wave w of four.
__device__ __forceinline__ void half_helpers(SerialLds<64>& lds, const Fetch<64>& fetch, int n_chunks, int w) {
  const Picker pick;
  BlocksOfP blocks{};
  float most = 0.f;
  fetch.t_four_waves(0, w);
  fetch.four_waves(0, w);
  wait_all_vm();
  slot_barrier();
  for (int j = 0; j < n_chunks; ++j) {
    if (j + 1 < n_chunks) {
      fetch.t_four_waves(j + 1, w);
      fetch.four_waves(j + 1, w);
    }
    const f32x4_t x = blocks.make(lds, j & 1, w);
    most = largest(x, most);
    blocks.store(pick, x, lds.p, w);
    if (j + 1 == n_chunks) lds.p_largest[64 * w + lane_id()] = most;
    slot_barrier();
    wait_all_vm();
    slot_barrier();
  }
}

// Quarters: X, R, U and S of 16 rows.
//              state waves                          output waves                  helpers
//     part 1   X of tokens 0-31                     Y of chunk j - 1, begun       T to LDS, chunk j + 1 asked for
//     part 2   X of 32-63, R, U                     the rest of it, half of Z     P
//     part 3   S                                    the rest of Z                 P to LDS, T of chunk j + 1 asked for
// S and U go to the output waves through LDS.  With all of Z in part 3 the output waves were the last there, by 0.2 K cycles of
// 5.36 K (one of 4005 tokens 159 -> 156 us, the four above 179.3 -> 177.5).  K, V and Q asked for in a part each, which takes the helpers
// out of the way in part 1: 155.5, but the four 182; K's operands of part 1 read in the part before it: no change.
__device__ __forceinline__ void quarter_state(QuarterLds& lds, int start, int end, int slot, int hv, int row, int w) {
  const int lane = lane_id();
  const int n_chunks = (end - start + kChunk - 1) / kChunk;
  StateRows rows;
  rows.load(slot, hv, row);
  f32x4_t (&s)[8] = rows.s;
  auto hand_over = [&](f32x4_t (*to)[64], const f32x4_t* from, int n) {
#pragma unroll
    for (int i = 0; i < n; ++i) to[i][lane] = from[i];
  };
  const Picker pick;
  const Places places;
  float most = 0.f;
  __builtin_amdgcn_s_setprio(1);
  hand_over(lds.s[0][w], s, 8);
  Split sp[4];  // S as operands
  sp[0] = split(pick, s[0], s[1]);
  sp[1] = split(pick, s[2], s[3]);
  slot_barrier();
  // The order keeps the matrix pipe at work: what a half of the tokens goes through between two products is done
  // beside the other half's.
  for (int j = 0; j < n_chunks; ++j) {
    const int par = j & 1;
    const Gates& gates = lds.gates[par];
    bf16x8_t k[2][4][2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int m = 0; m < 2; ++m) k[h][c][m] = operand(&lds.k[par][32 * h + 16 * m][0] + places.at[c]);
    sp[2] = split(pick, s[4], s[5]);
    sp[3] = split(pick, s[6], s[7]);
    fence();
    f32x4_t x[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) x[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto half_of_x = [&](int h) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        auto step = [&](bf16x8_t part) {
#pragma unroll
          for (int m = 0; m < 2; ++m) x[2 * h + m] = product<false>(k[h][c][m], part, x[2 * h + m]);
        };
        step(sp[c].lo);
        step(sp[c].mid);
        step(sp[c].hi);
      }
    };
    ForR f0, f1;
    f0.load(lds, par, 16 * w, 0);
    f1.load(lds, par, 16 * w, 1);
    half_of_x(0);
    slot_barrier();  // T
    Triangle tp;
    load_triangle<0, 4>(lds.t[0], tp);
    fence();
    half_of_x(1);
    const Split r0 = f0.make(pick, x);
    weave<14, 4>();
    fence();
    load_triangle<4, 6>(lds.t[0], tp);
    f32x4_t u[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) u[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    bf16x8_t kt[4][4];
    load_transposed(lds.k[par], places, 0, kt[0]);
    triangle_first<false>(tp, r0, u);
    const Split r1 = f1.make(pick, x + 2);
    weave<14, 4>();
    fence();
    load_transposed(lds.k[par], places, 2, kt[2]);
    triangle_second<false>(tp, r1, u);
    const Split ut0 = weigh(pick, gates, u, 0);
    const float total = gates.total;
#pragma unroll
    for (int c = 0; c < 8; ++c) s[c] *= total;
    weave<16, 4>();
    slot_barrier();  // P and U of chunk j - 1 have been read
    load_transposed(lds.k[par], places, 1, kt[1]);
    load_transposed(lds.k[par], places, 3, kt[3]);
    state_steps(s, kt[0], 0, ut0);
    state_steps(s, kt[2], 2, ut0);
    const Split ut1 = weigh(pick, gates, u, 1);
    hand_over(lds.u[w], u, 4);
#pragma unroll
    for (int m = 0; m < 4; ++m) most = largest(u[m], most);
    weave<14, 4>();
    fence();
    state_steps(s, kt[1], 1, ut1);
    fence();
    hand_over(lds.s[par ^ 1][w], s, 4);
    state_steps(s, kt[3], 3, ut1);
    sp[0] = split(pick, s[0], s[1]);
    sp[1] = split(pick, s[2], s[3]);
    weave<20, 3>();
    hand_over(lds.s[par ^ 1][w] + 4, s + 4, 4);
    slot_barrier();
  }
  slot_barrier();  // the output waves' stores are done
  most = largest(*reinterpret_cast<const f32x4_t*>(&lds.p_largest[4 * lane]), most);
  if (__builtin_expect(!__all(splits(most)), 0)) {
    token_by_token(start, end, slot, hv, row);
    return;
  }
  rows.store(slot, hv, row);
}
// Quarters: Z and Y of the rows of state wave w.
__device__ __forceinline__ void quarter_output(const GdnParams& p, QuarterLds& lds, int start, int end, int hv, int row, int w) {
  const int lane = lane_id(), x16 = lane & 15;
  const int n_chunks = (end - start + kChunk - 1) / kChunk;
  const Outputs y(p, start, end, hv, row);
  const Picker pick;
  const Places places;
  f32x4_t z[4];
  auto finish = [&](int j, auto between) {  // Y = G Z + P U
    Triangle tp;
    load_triangle<0, 6>(lds.p, tp);
    const Split u0 = split(pick, lds.u[w][0][lane], lds.u[w][1][lane]);
    const Split u1 = split(pick, lds.u[w][2][lane], lds.u[w][3][lane]);
    triangle_first<true>(tp, u0, z);
    between();
    triangle_second<true>(tp, u1, z);
    y.store(j, z);
  };
  slot_barrier();
  for (int j = 0; j < n_chunks; ++j) {
    const int par = j & 1;
    if (j > 0) finish(j - 1, [] { slot_barrier(); });
    else slot_barrier();
#pragma unroll
    for (int m = 0; m < 4; ++m) z[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto half_of_z = [&](auto half) {
      constexpr int c0 = 2 * decltype(half)::value;
      bf16x8_t q[2][4];
      Split sp[2];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        load_operands(lds.q[par], places.at[c0 + c], q[c]);
        sp[c] = split(pick, lds.s[par][w][2 * (c0 + c)][lane], lds.s[par][w][2 * (c0 + c) + 1][lane]);
      }
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        auto step = [&](bf16x8_t part) {
#pragma unroll
          for (int m = 0; m < 4; ++m) z[m] = product<true>(q[c][m], part, z[m]);
        };
        step(sp[c].lo);
        step(sp[c].mid);
        step(sp[c].hi);
      }
    };
    half_of_z(std::integral_constant<int, 0>{});
    slot_barrier();
    half_of_z(std::integral_constant<int, 1>{});
#pragma unroll
    for (int m = 0; m < 4; ++m) z[m] *= lds.gates[par].gamma[16 * m + x16];
    slot_barrier();
  }
  finish(n_chunks - 1, [] {});
  wait_all_vm();  // the state waves may have to write the same places again
  slot_barrier();
}
// Quarters: what the others don't do, by wave w of four.
__device__ __forceinline__ void quarter_helpers(QuarterLds& lds, const Fetch<32>& fetch, int n_chunks, int w) {
  const Picker pick;
  BlocksOfP blocks{};
  float most = 0.f;
  // T's 18 KiB through registers, so that it is there soon after its place is free
  u32x4_t t[5];
  auto load_t = [&](int j) {
#pragma unroll
    for (int i = 0; i < 5; ++i)
      if (i < 4 || w < 2) t[i] = ld_global_b128(fetch.records + (int64_t)j * fetch.record_step + 1024 * (4 * i + w) + 16 * lane_id());
  };
  load_t(0);
  fetch.four_waves(0, w);
  wait_all_vm();
  slot_barrier();
  for (int j = 0; j < n_chunks; ++j) {
    const bool more = j + 1 < n_chunks;
#pragma unroll
    for (int i = 0; i < 5; ++i)
      if (i < 4 || w < 2) (&lds.t[0][0][0][0])[64 * (4 * i + w) + lane_id()] = t[i];
    if (more) fetch.four_waves(j + 1, w);
    slot_barrier();
    const f32x4_t x = blocks.make(lds, j & 1, w);
    most = largest(x, most);
    slot_barrier();
    blocks.store(pick, x, lds.p, w);
    if (more) {
      load_t(j + 1);
      if (w < 2) wait_vm_at_most<5>();  // all but T
      else wait_vm_at_most<4>();
    } else {
      lds.p_largest[64 * w + lane_id()] = most;
    }
    slot_barrier();
  }
  slot_barrier();
}

// Time of a chunk in halves, in quarters (7.6 K and 5.2 K cycles).
constexpr int kCost[2] = {16, 11};

// Which request a place works for and how that is spread, the longest first: every request begins in halves, two places, and the
// one that would end last goes on in quarters, four, if it sticks out of the launch's average and the compute units have room for
// that, or the others, on what it leaves of them (and what the last one of those may stick out), end before it would have.
struct Place {
  int b, part;
  bool quarters;
};
__device__ __forceinline__ bool find_place(const GdnParams& p, int place, int places, int slots, Place* out, int* start, int* end) {
  const int lane = lane_id(), at = min(lane, p.batch - 1);
  const int from = p.qo_indptr[at], to = min(p.qo_indptr[at + 1], p.tokens);
  const int length = lane < p.batch ? max(0, to - from) : -1;
  const int chunks = lane < p.batch ? (length + kChunk - 1) / kChunk : 0;
  bool quarters = false;
  int time = chunks * kCost[0], used = 2 * p.batch;
  int busy = 2 * wave_sum(time), rest = busy, left = slots;  // rest: of those in halves, on `left` places
  const int shortest = wave_min(lane < p.batch ? time : 0x7fffffff);
  while (used + 2 <= places) {
    const int longest = wave_max(time);
    if (longest * slots <= busy + (busy >> 3)) break;
    const int src = __builtin_ctzll(__ballot(time == longest));
    if (__builtin_amdgcn_readlane((int)quarters, src)) break;
    rest -= 2 * longest;
    left -= 4;
    if (used + 2 > slots && (left < 2 || 16 * (rest + (left - 1) * shortest) > 15 * left * longest)) break;
    const int now = __builtin_amdgcn_readlane(chunks, src) * kCost[1];
    used += 2;
    busy += 4 * now - 2 * longest;
    if (lane == src) {
      quarters = true;
      time = now;
    }
  }
  int before = 0;  // places of longer requests
  for (int o = 0; o < p.batch; ++o) {
    const int other = __builtin_amdgcn_readlane(length, o), width = 2 + 2 * __builtin_amdgcn_readlane((int)quarters, o);
    before += other > length || (other == length && o < lane) ? width : 0;
  }
  const uint64_t found = __ballot(lane < p.batch && place >= before && place < before + (quarters ? 4 : 2));
  if (!found) return false;
  const int b = __builtin_ctzll(found);
  out->b = b;
  out->part = place - __builtin_amdgcn_readlane(before, b);
  out->quarters = __builtin_amdgcn_readlane((int)quarters, b) != 0;
  *start = __builtin_amdgcn_readlane(from, b);
  *end = __builtin_amdgcn_readlane(to, b);
  return true;
}

// Workgroup -> (place, key head, value head of it), ids of one residue modulo 8 for what shares K and Q rows.
__global__ __launch_bounds__(512) void gdn_serial_kernel(GdnParams p, const ChunkRecord* records, int places, int slots) {
  __shared__ union {
    SerialLds<64> half;
    QuarterLds quarter;
    struct {
      int length[kRanked], request;
    } order;
  } lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hk_n = p.hv / p.hv_per_hk, groups = places * hk_n;
  int group, member;
  if (groups % 8 == 0) {
    const int seq = blockIdx.x >> 3;
    group = (seq / p.hv_per_hk) * 8 + (blockIdx.x & 7);
    member = seq % p.hv_per_hk;
  } else {
    group = blockIdx.x / p.hv_per_hk;
    member = blockIdx.x % p.hv_per_hk;
  }
  const int place = group / hk_n, hv = (group - place * hk_n) * p.hv_per_hk + member;
  Place at{place >> 1, place & 1, false};
  int start, end;
  if (p.batch <= kWave) {
    if (!find_place(p, place, places, slots, &at, &start, &end)) return;
  } else {
    if (p.batch <= kRanked) {
      const int tid = threadIdx.x;
      int mine = 0;
      if (tid < p.batch) lds.order.length[tid] = mine = p.qo_indptr[tid + 1] - p.qo_indptr[tid];
      __syncthreads();
      if (tid < p.batch) {
        int rank = 0;
        for (int o = 0; o < p.batch; ++o) rank += (lds.order.length[o] > mine || (lds.order.length[o] == mine && o < tid)) ? 1 : 0;
        if (rank == place >> 1) lds.order.request = tid;
      }
      __syncthreads();
      at.b = lds.order.request;
      __syncthreads();
    }
    at.b = __builtin_amdgcn_readfirstlane(at.b);
    start = p.qo_indptr[at.b];
    end = min(p.qo_indptr[at.b + 1], p.tokens);
  }
  if (end <= start) return;  // the whole workgroup: the state stays as it is
  const int slot = __builtin_amdgcn_readfirstlane(p.slot_ids[at.b]);
  const int n_chunks = (end - start + kChunk - 1) / kChunk;
  // the blocks of P above the diagonal that are read are never written: zero from here on
  auto clear = [](auto& m) {
    for (int i = threadIdx.x; i < (int)sizeof(m) / 16; i += 512) reinterpret_cast<u32x4_t*>(&m[0][0][0])[i] = u32x4_t{0u, 0u, 0u, 0u};
  };
  if (!at.quarters) {
    const int row = 64 * at.part;
    clear(lds.half.p);
    if (wave < 4) half_rows(p, lds.half, start, end, slot, hv, row + 16 * wave, 16 * wave);
    else half_helpers(lds.half, Fetch<64>(p, records, lds.half, at.b, start, end, hv, row), n_chunks, wave - 4);
  } else {
    const int row = 32 * at.part;
    clear(lds.quarter.p);
    if (wave < 2) quarter_state(lds.quarter, start, end, slot, hv, row + 16 * wave, wave);
    else if (wave < 4) quarter_output(p, lds.quarter, start, end, hv, row + 16 * (wave - 2), wave - 2);
    else quarter_helpers(lds.quarter, Fetch<32>(p, records, lds.quarter, at.b, start, end, hv, row), n_chunks, wave - 4);
  }
}

int64_t chunk_records(int64_t tokens, int64_t batch) { return tokens / kChunk + batch; }

}  // namespace

size_t gdn_long_workspace_bytes(int64_t tokens, int64_t batch, int64_t hv) {
  return (size_t)(chunk_records(tokens, batch) * hv) * sizeof(ChunkRecord);
}

int launch_gdn_long(const GdnParams& p, void* workspace, hipStream_t stream) {
  ChunkRecord* const records = static_cast<ChunkRecord*>(workspace);
  const int64_t chunks = chunk_records(p.tokens, p.batch), hk = p.hv / p.hv_per_hk;
  const int64_t systems = (chunks * hk + 7) / 8 * 8 * p.hv_per_hk;
  const int64_t slots = std::max<int64_t>(device_cus() / p.hv, 1);
  // two for every request; more as far as they make one round, or for two requests where there are more rounds
  const int64_t places = p.batch > kWave ? 2 * p.batch : std::min<int64_t>(4 * p.batch, std::max<int64_t>(slots, 2 * p.batch + 4));
  const int64_t blocks = places * p.hv;
  if (systems > 0x7fffffffLL || blocks > 0x7fffffffLL) return MSGL_ERR_SHAPE;
  hipLaunchKernelGGL(gdn_systems_kernel, dim3((unsigned)systems), dim3(256), 0, stream, p, records, (int)chunks);
  hipLaunchKernelGGL(gdn_serial_kernel, dim3((unsigned)blocks), dim3(512), 0, stream, p, records, (int)places, (int)slots);
  return check_launch();
}

}  // namespace msgl
