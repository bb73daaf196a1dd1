// MFMA helpers shared by the attention kernels (gfx950, 64-wide waves).
#pragma once

#include <type_traits>

#include "dsp_common.h"

namespace dsp_mfma {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct Bf16Tag {};
struct F16Tag {};

// One v_mfma_f32_16x16x32_{bf16,f16}: c += a . b with 8 packed 16-bit values per lane in
// each operand (lane l: row l % 16, k range 8 * (l / 16) .. +8).
template <typename Tag>
__device__ __forceinline__ f32x4 mfma32(dsp_u32x4 a, dsp_u32x4 b, f32x4 c) {
  if constexpr (std::is_same<Tag, Bf16Tag>::value)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// fp32 -> the cache dtype, round to nearest even.
template <typename Tag>
__device__ __forceinline__ uint16_t narrow(float f) {
  if constexpr (std::is_same<Tag, Bf16Tag>::value)
    return dsp_f32_to_bf16(f);
  else
    return dsp_f32_to_f16(f);
}

template <typename Tag>
__device__ __forceinline__ float widen(uint16_t b) {
  if constexpr (std::is_same<Tag, Bf16Tag>::value)
    return dsp_bf16lo(b);
  else
    return dsp_f16lo(b);
}

__device__ __forceinline__ uint32_t pack2(uint16_t lo, uint16_t hi) {
  return uint32_t(lo) | (uint32_t(hi) << 16);
}

// Eight fp32 values as a 16-bit MFMA operand and, kSplit, the operand of what that rounding
// left over: hi + lo holds a probability to 16 bits (bf16) or 22 (fp16), so two MFMAs over
// them give P.V as fp32 probabilities would, for the shapes whose probabilities are fp32.
template <typename Tag, bool kSplit>
__device__ __forceinline__ void pack8(const float (&p)[8], dsp_u32x4& hi, dsp_u32x4& lo) {
  uint16_t h[8], l[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    h[i] = narrow<Tag>(p[i]);
    l[i] = kSplit ? narrow<Tag>(p[i] - widen<Tag>(h[i])) : uint16_t(0);
  }
  hi = dsp_u32x4{pack2(h[0], h[1]), pack2(h[2], h[3]), pack2(h[4], h[5]), pack2(h[6], h[7])};
  lo = dsp_u32x4{pack2(l[0], l[1]), pack2(l[2], l[3]), pack2(l[4], l[5]), pack2(l[6], l[7])};
}

}  // namespace dsp_mfma
