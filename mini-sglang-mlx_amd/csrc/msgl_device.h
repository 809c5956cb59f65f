// Device-side building blocks shared by the gfx950 paged-attention kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace msgl {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kWave = 64;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegInf = -__builtin_inff();

// 16-byte global load / store of 8 bf16 (one lane's MFMA operand slice).
__device__ __forceinline__ u32x4_t ld_global_b128(const void* p) {
  return *reinterpret_cast<const u32x4_t*>(p);
}
// The same of what nobody reads again soon: the line leaves the caches first.  A wave's loads of whole 128-byte lines this way, 16 KiB after
// 16 KiB: 4 GiB at 6.7-7.0 TB/s, plain loads 5.9-6.1; of halves of lines, whose other half another load asks for, 5.2-6.1.  (From the caches 12 and 25.)
__device__ __forceinline__ u32x4_t ld_stream_b128(const void* p) { return __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p)); }
__device__ __forceinline__ void st_global_b128(void* p, u32x4_t v) {
  *reinterpret_cast<u32x4_t*>(p) = v;
}
// Rows of a result, 256 bytes of each: what is still in the L2 caches when a kernel ends is written back then, with nothing beside it.  240 extends at
// head_dim 128 and 256, those of 16-50 us 1.012 and 1.019 (geometric mean; 12 prompts of up to 113 tokens 15.1 -> 13.8, 7 of up to 80 15.5 ->
// 14.5), longer ones 1.00.  Whole lines only: in pieces of 32 bytes the rows of workgroups that stay cost head_dim 256 3-5 %.
__device__ __forceinline__ void st_stream_b128(void* p, u32x4_t v) { __builtin_nontemporal_store(v, reinterpret_cast<u32x4_t*>(p)); }

__device__ __forceinline__ bf16x8_t as_bf16x8(u32x4_t v) {
  return __builtin_bit_cast(bf16x8_t, v);
}

// Two fp32 -> packed bf16x2 (round to nearest even); lowers to v_cvt_pk_bf16_f32.
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  bf16x2_t p;
  p[0] = (__bf16)lo;
  p[1] = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, p);
}

// Optimisation barrier on one register value: it must be computed before this point and
// is treated as modified after it.
__device__ __forceinline__ void pin(float& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void pin(uint32_t& x) { asm volatile("" : "+v"(x)); }

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// v_perm_b32: result byte i = byte sel[i] of the 8-byte value {hi:lo} (lo = bytes 0..3).
__device__ __forceinline__ uint32_t perm_b32(uint32_t hi, uint32_t lo, uint32_t sel) {
  return __builtin_amdgcn_perm(hi, lo, sel);
}
// {a.lo16, b.lo16} and {a.hi16, b.hi16}: the two halves of a 2x2 transpose of 16-bit lanes.
__device__ __forceinline__ uint32_t pack_lo16(uint32_t a, uint32_t b) {
  return perm_b32(b, a, 0x05040100u);
}
__device__ __forceinline__ uint32_t pack_hi16(uint32_t a, uint32_t b) {
  return perm_b32(b, a, 0x07060302u);
}

// D(16x16 f32) += A(16x32 bf16) * B(32x16 bf16).
//   A: lane l holds A[l%16][8*(l/16) .. +8]      B: lane l holds B[8*(l/16) .. +8][l%16]
//   D: lane l holds D[4*(l/16) + i][l%16], i = 0..3
__device__ __forceinline__ f32x4_t mfma_16x16x32(bf16x8_t a, bf16x8_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// D(32x32 f32) += A(32x16 bf16) * B(16x32 bf16).
//   A: lane l holds A[l%32][8*(l/32) .. +8]      B: lane l holds B[8*(l/32) .. +8][l%32]
//   D: lane l holds D[8*(i/4) + 4*(l/32) + i%4][l%32], i = 0..15
__device__ __forceinline__ f32x16_t mfma_32x32x16(bf16x8_t a, bf16x8_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// The same product on raw 16-bit operands: bf16 or, with F16, IEEE half.
template <bool F16>
__device__ __forceinline__ f32x4_t mfma_16x16x32_raw(u32x4_t a, u32x4_t b, f32x4_t c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  else
    return mfma_16x16x32(as_bf16x8(a), as_bf16x8(b), c);
}
// Two fp32 -> packed 16-bit pair, round to nearest even.
template <bool F16>
__device__ __forceinline__ uint32_t pack_16x2(float lo, float hi) {
  if constexpr (F16) {
    f16x2_t p;
    p[0] = (_Float16)lo;
    p[1] = (_Float16)hi;
    return __builtin_bit_cast(uint32_t, p);
  } else {
    return pack_bf16x2(lo, hi);
  }
}

__device__ __forceinline__ int lane_id() { return threadIdx.x & (kWave - 1); }

// ---- values of other lanes, without LDS (a shuffle through LDS costs about 100 cycles, these 5 to 10) -------------
// All lanes of the wave have to be active.
// DPP control C, 0 where there is no such lane: 0xB1 lane ^ 1, 0x4E lane ^ 2, 0x141 mirror in 8, 0x140 mirror in 16,
// 0x110 + n the lane n below and 0x120 + n the lane n below with rotation, in 16.
template <int C>
__device__ __forceinline__ int dpp(int v) {
  return __builtin_amdgcn_update_dpp(0, v, C, 0xf, 0xf, true);
}
template <int C>
__device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, dpp<C>(__builtin_bit_cast(int, v)));
}
// For M = 16 and 32: the swap leaves a row's (half's) value and its partner's in the two results.
template <int M>
__device__ __forceinline__ float max_across(float v) {  // of lanes l and l ^ M
  const uint32_t x = __builtin_bit_cast(uint32_t, v);
  if constexpr (M == 16) {
    const auto s = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    return fmaxf(__builtin_bit_cast(float, (uint32_t)s[0]), __builtin_bit_cast(float, (uint32_t)s[1]));
  } else {
    const auto s = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return fmaxf(__builtin_bit_cast(float, (uint32_t)s[0]), __builtin_bit_cast(float, (uint32_t)s[1]));
  }
}
template <int M>
__device__ __forceinline__ float sum_across(float v) {  // of lanes l and l ^ M
  const uint32_t x = __builtin_bit_cast(uint32_t, v);
  if constexpr (M == 16) {
    const auto s = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    return __builtin_bit_cast(float, (uint32_t)s[0]) + __builtin_bit_cast(float, (uint32_t)s[1]);
  } else {
    const auto s = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return __builtin_bit_cast(float, (uint32_t)s[0]) + __builtin_bit_cast(float, (uint32_t)s[1]);
  }
}
// Sum over a row of 16 lanes, in the order of a butterfly: once the lanes of a group of 4 (of 8) agree, the mirrors
// in 8 (in 16) are as good as lane ^ 4 (lane ^ 8).
__device__ __forceinline__ float row_sum16(float v) {
  v += dpp<0xB1>(v);
  v += dpp<0x4E>(v);
  v += dpp<0x141>(v);
  v += dpp<0x140>(v);
  return v;
}
__device__ __forceinline__ float row_max16(float v) {
  v = fmaxf(v, dpp<0xB1>(v));
  v = fmaxf(v, dpp<0x4E>(v));
  v = fmaxf(v, dpp<0x141>(v));
  return fmaxf(v, dpp<0x140>(v));
}
// The value of lane N of a row of 16 lanes, in all of them
template <int N>
__device__ __forceinline__ float of_row_lane(float v) {
  return dpp<0x150 + N>(v);
}
__device__ __forceinline__ int row_max16(int v) {
  v = max(v, dpp<0x128>(v));
  v = max(v, dpp<0x124>(v));
  v = max(v, dpp<0x122>(v));
  return max(v, dpp<0x121>(v));
}
// The largest and the smallest value of a wave, in a scalar register.
__device__ __forceinline__ int wave_max(int v) {
  v = row_max16(v);
  return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
             max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}
__device__ __forceinline__ int wave_min(int v) { return ~wave_max(~v); }
// Wave-wide sum (a scalar) and inclusive prefix sum: a prefix sum inside each row of 16 lanes, the rows' totals
// through scalar registers.
__device__ __forceinline__ int row_scan(int v) {
  v += dpp<0x111>(v);
  v += dpp<0x112>(v);
  v += dpp<0x114>(v);
  v += dpp<0x118>(v);
  return v;
}
__device__ __forceinline__ int wave_sum(int v) {
  v = row_scan(v);
  return __builtin_amdgcn_readlane(v, 15) + __builtin_amdgcn_readlane(v, 31) + __builtin_amdgcn_readlane(v, 47) +
         __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ int wave_inclusive_scan(int v) {
  v = row_scan(v);
  const int r0 = __builtin_amdgcn_readlane(v, 15), r1 = __builtin_amdgcn_readlane(v, 31), r2 = __builtin_amdgcn_readlane(v, 47);
  const int row = lane_id() >> 4;
  return v + (row > 0 ? r0 : 0) + (row > 1 ? r1 : 0) + (row > 2 ? r2 : 0);
}

// A kernel's parameters come through the scalar cache, 64 bytes at a time, from memory that no cache of the compute unit has
// seen: a wave that reads them where it needs them waits half a microsecond each time.  Called while the first load of a
// kernel's own is under way, this has all the lines of the first BYTES asked for together.  (The registers are nobody's: only the lines are wanted.)
template <int BYTES>
__device__ __forceinline__ void fetch_parameters() {
  static_assert(BYTES > 0 && BYTES <= 512, "eight lines");
  const auto at = __builtin_amdgcn_kernarg_segment_ptr();
  constexpr int kLast = (BYTES - 4) & ~3;
  constexpr auto line = [](int i) { return 64 * i < kLast ? 64 * i : kLast; };
  uint32_t r0, r1, r2, r3, r4, r5, r6, r7;
  asm volatile(
      "s_load_dword %0, %8, %9\n\ts_load_dword %1, %8, %10\n\ts_load_dword %2, %8, %11\n\ts_load_dword %3, %8, %12\n\t"
      "s_load_dword %4, %8, %13\n\ts_load_dword %5, %8, %14\n\ts_load_dword %6, %8, %15\n\ts_load_dword %7, %8, %16\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&s"(r0), "=&s"(r1), "=&s"(r2), "=&s"(r3), "=&s"(r4), "=&s"(r5), "=&s"(r6), "=&s"(r7)
      : "s"(at), "n"(line(0)), "n"(line(1)), "n"(line(2)), "n"(line(3)), "n"(line(4)), "n"(line(5)), "n"(line(6)), "n"(line(7))
      : "memory");
}

// Measurement aid: when `dst` is given, thread 0 of workgroup 0 leaves the shader cycles and the
// 100 MHz wall ticks between its construction and its destruction (every way out of the kernel) in
// dst[0], dst[1]: cycles / ticks x 0.1 is the shader clock in GHz while the kernel ran.  (Both
// counters are read by the same wave: the cycle counters of different compute units are unrelated.)
struct ClockProbe {
  long long* dst;
  long long c0, w0;
  __device__ __forceinline__ explicit ClockProbe(long long* d)
      : dst((d != nullptr && blockIdx.x == 0 && threadIdx.x == 0) ? d : nullptr), c0(0), w0(0) {
    if (dst != nullptr) {
      c0 = clock64();
      w0 = wall_clock64();
    }
  }
  __device__ __forceinline__ ~ClockProbe() {
    if (dst != nullptr) {
      dst[0] = clock64() - c0;
      dst[1] = wall_clock64() - w0;
    }
  }
};

}  // namespace msgl
