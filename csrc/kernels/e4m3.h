// Decoding of e4m3 weight codes in registers (fp8_gemm.hip, stream_gemm.hip).
#pragma once

#include "common.h"

namespace mx {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Eight codes (lo: the first four) -> bf16, exactly: the hardware's pair conversion with scale one, 4 instructions
// where decoding by byte permutes, masks and shifts took 20 (28672 x 4096, 4 rows,
// stream_gemm: 28.8 -> 25.8 us).
__device__ __forceinline__ u16x8 dequant8(uint32_t lo, uint32_t hi) {
  return __builtin_bit_cast(u16x8, u32x4{
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.f, false)),
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.f, true)),
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.f, false)),
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.f, true))});
}

}  // namespace mx
