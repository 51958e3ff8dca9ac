// Steps on the 16 channels a lane holds, shared by the quantizers and by the attention kernel where it quantizes Q itself.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/ksana_sage_hip.h"

namespace ksana_sage {

template <int DT>
__device__ __forceinline__ void widen8(const uint4& raw, float* out) {
  const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (DT == KSANA_SAGE_BF16) {
      out[2 * i] = __uint_as_float(w[i] << 16);
      out[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    } else {
      typedef _Float16 h2 __attribute__((ext_vector_type(2)));
      h2 p = __builtin_bit_cast(h2, w[i]);
      out[2 * i] = (float)p[0];
      out[2 * i + 1] = (float)p[1];
    }
  }
}

// rne(x * inv) as int8, sixteen at a time, the product exact: one fused multiply-add onto 1.5 * 2^23, where the fp32
// grid is the integers, rounds the exact sum to nearest, ties to even, and leaves the two's-complement int8 in the low
// byte.  No clamp: |x| <= amax and inv = fl(127 / amax) keep |x * inv| below 127.5.  One instruction per value plus
// three byte-gathers per four.
__device__ __forceinline__ uint4 pack_int8x16(const float* x, float inv) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t z[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) z[j] = __float_as_uint(__fmaf_rn(x[4 * i + j], inv, 12582912.0f));
    const uint32_t lo = __builtin_amdgcn_perm(z[1], z[0], 0x0c0c0400u);  // bytes 0, 1 <- low bytes of z0, z1
    const uint32_t hi = __builtin_amdgcn_perm(z[3], z[2], 0x04000c0cu);  // bytes 2, 3 <- low bytes of z2, z3
    w[i] = lo | hi;
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

}  // namespace ksana_sage
