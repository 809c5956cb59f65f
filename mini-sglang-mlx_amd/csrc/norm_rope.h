// RMS norm and rotary embedding of one head by 16 lanes, shared by the kernel that does nothing else
// (qk_norm_rope_store.hip) and the decode launch that does it on the way (paged_shares.hip): the same operations in
// the same order, so the same bits.
#pragma once
#include "msgl_device.h"

namespace msgl {

// Lane j of the 16 holds elements E j .. E j + E - 1 of both halves of the head (E = D / 32), so the rotation
// pairs are lane-local.
template <int E>
struct HalfRow;  // E bf16 values as one load
template <>
struct HalfRow<4> { typedef u32x2_t type; };
template <>
struct HalfRow<8> { typedef u32x4_t type; };

// Angle of rotation pair `i` at a position, before the sine and the cosine.
template <int D>
__device__ __forceinline__ float rope_angle(float position, int i, float log2_base) {
  return position * exp2f(-((float)i / (float)(D / 2)) * log2_base);
}

template <int D>
__device__ __forceinline__ void norm_rope_head(typename HalfRow<D / 32>::type& lo, typename HalfRow<D / 32>::type& hi,
                                               const typename HalfRow<D / 32>::type& wl,
                                               const typename HalfRow<D / 32>::type& wh, const float (&cs)[D / 32],
                                               const float (&sn)[D / 32], float eps) {
  constexpr int E = D / 32;
  auto value = [](const typename HalfRow<E>::type& r, int e) {
    const uint32_t w = r[e >> 1];
    return __builtin_bit_cast(float, (e & 1) ? w & 0xffff0000u : w << 16);
  };
  auto round = [](float f) { return (float)(__bf16)f; };
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < E; ++e) ss += value(lo, e) * value(lo, e) + value(hi, e) * value(hi, e);
  ss = row_sum16(ss);
  const float norm = rsqrtf(ss * (1.0f / D) + eps);
#pragma unroll
  for (int e = 0; e < E; e += 2) {
    float ol[2], oh[2];
#pragma unroll
    for (int o = 0; o < 2; ++o) {
      // normalised value and weighted value each pass through bf16, as they do when the norm is a kernel of its
      // own with a bf16 result
      const float yl = round(value(wl, e + o) * round(value(lo, e + o) * norm));
      const float yh = round(value(wh, e + o) * round(value(hi, e + o) * norm));
      ol[o] = yl * cs[e + o] - yh * sn[e + o];
      oh[o] = yl * sn[e + o] + yh * cs[e + o];
    }
    lo[e >> 1] = pack_bf16x2(ol[0], ol[1]);
    hi[e >> 1] = pack_bf16x2(oh[0], oh[1]);
  }
}

}  // namespace msgl
