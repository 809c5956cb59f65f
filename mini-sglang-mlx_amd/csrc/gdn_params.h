// Launch parameters and small pieces shared by the gated delta-rule kernels (gdn_state.hip: token after
// token; gdn_short.hip and gdn_chunk.hip: chunks of 16 and of 64 tokens on the matrix cores; gdn_long.hip:
// chunks of 64 in two launches).
#pragma once
#include "msgl_device.h"
#include "msgl_internal.h"

namespace msgl {

constexpr int kDK = 128, kDV = 128;

struct GdnParams {
  float* state;
  uint16_t* y;
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const uint16_t* g;
  const uint16_t* beta;
  const int32_t* slot_ids;
  const int32_t* qo_indptr;
  int64_t state_stride0, q_stride0, k_stride0, v_stride0;
  int32_t batch, hv, hv_per_hk, tokens, single_token;
};

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t b) { return __builtin_bit_cast(float, b << 16); }

int launch_gdn_short(const GdnParams& p, hipStream_t stream);
int launch_gdn_chunks(const GdnParams& p, hipStream_t stream);
size_t gdn_long_workspace_bytes(int64_t tokens, int64_t batch, int64_t hv);
int launch_gdn_long(const GdnParams& p, void* workspace, hipStream_t stream);

}  // namespace msgl
