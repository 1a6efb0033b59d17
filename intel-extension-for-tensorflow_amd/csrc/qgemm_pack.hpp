// The last step of the epilogues that keep 16 consecutive channels of a row in one lane (qgemm_stream.hip, qconv_direct.hip).
#ifndef ITEXHIP_QGEMM_PACK_HPP_
#define ITEXHIP_QGEMM_PACK_HPP_

#include "qgemm_common.hpp"

namespace itexhip {

// What follows scale and bias: nothing (saturation does it), max(v, 0), or min(max(v, lo), hi).
enum : int { kPostNone = 0, kPostRelu = 1, kPostClip = 2 };

// 4 values -> 4 bytes.  v_cvt_pk_u8_f32 rounds to nearest even, saturates to 0 .. 255 and puts the byte into place in one
// instruction: for every fp32 value but NaN the byte that clamp, magic-number add and permute give (compared over all 2^32
// patterns on the device); a value that may be NaN is clamped first, as there.
template <int OUT_T, int POST>
__device__ __forceinline__ uint32_t pack_bytes(const float (&v)[4]) {
  if constexpr (OUT_T == ITEXHIP_QUINT8) {
    uint32_t w = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      w = __builtin_amdgcn_cvt_pk_u8_f32(POST == kPostNone ? __builtin_amdgcn_fmed3f(v[i], 0.0f, 255.0f) : v[i], i, w);
    return w;
  } else {
    return static_cast<uint32_t>(epilogue_pack<OUT_T>(v4i{__float_as_int(v[0]), __float_as_int(v[1]), __float_as_int(v[2]), __float_as_int(v[3])}).x);
  }
}

}  // namespace itexhip
#endif  // ITEXHIP_QGEMM_PACK_HPP_
