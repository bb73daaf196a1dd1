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

__device__ __forceinline__ uint32_t pack2(uint16_t lo, uint16_t hi) {
  return uint32_t(lo) | (uint32_t(hi) << 16);
}

// Eight fp32 probabilities as kTerms 16-bit MFMA operands.  One: their rounding.  More: each
// operand takes the leading bits of what the ones before it left over, the last one its
// rounding.  Three hold all 24 bits of an fp32 value: P.V over them is P.V of fp32
// probabilities, for the shapes whose probabilities are fp32 (two hold 16 bits in bf16, 22 in
// fp16; with the third the 256-wide prefill tile takes 91 us instead of 82 at 4 x 200 tokens over
// 1999, 24 slot-table decodes 21.9 instead of 20.9).
// The leading bits are cut, not rounded, and an operand of a p above 0 is kept above 0 (by the
// least number, 2^-100 or the last bit kept), so that an infinity in V meets positive factors
// only: a 0 or a negative one would make NaN of it.
// bf16 has fp32's exponents.  fp16 ends at 2^-24, so more than one term expects p * p_scale
// there, at most 2^15: with three p <= 1 and the last bit kept is 2^-39, whatever p's size; with
// two p <= 2^8 (a lagging maximum) and 2^-31.  The row sum takes the same factor, and the
// division by it cancels the two.
template <typename Tag, int kTerms>
constexpr float p_scale() {
  return kTerms == 1 || std::is_same<Tag, Bf16Tag>::value ? 1.f : kTerms == 2 ? 128.f : 32768.f;
}

template <typename Tag, int kTerms>
__device__ __forceinline__ void pack8(const float* p, dsp_u32x4 (&t)[kTerms]) {
  if constexpr (kTerms == 1) {
    uint16_t h[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) h[i] = narrow<Tag>(p[i]);
    t[0] = dsp_u32x4{pack2(h[0], h[1]), pack2(h[2], h[3]), pack2(h[4], h[5]), pack2(h[6], h[7])};
    return;
  }
  constexpr bool kBf16 = std::is_same<Tag, Bf16Tag>::value;
  constexpr float kLeast = kBf16 ? 0x1p-100f : 0x1p-24f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float rest[2] = {p[2 * i], p[2 * i + 1]};
    const float least[2] = {fminf(rest[0], kLeast), fminf(rest[1], kLeast)};
#pragma unroll
    for (int k = 0; k < kTerms; ++k) {
      if (k + 1 == kTerms) {
        t[k][i] = pack2(narrow<Tag>(rest[0]), narrow<Tag>(rest[1]));
        break;
      }
      float cut[2];
      if constexpr (kBf16) {
        const uint32_t a = __float_as_uint(rest[0]), b = __float_as_uint(rest[1]);
        t[k][i] = (a >> 16) | (b & 0xffff0000u);
        cut[0] = __uint_as_float(a & 0xffff0000u);
        cut[1] = __uint_as_float(b & 0xffff0000u);
      } else {
        t[k][i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(rest[0], rest[1]));
        cut[0] = dsp_f16lo(t[k][i]);
        cut[1] = dsp_f16hi(t[k][i]);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) rest[j] = fmaxf(rest[j] - cut[j], least[j]);
    }
  }
}

// The low n bits, n clamped to 0..32.
__device__ __forceinline__ uint32_t low_bits(int n) {
  return n >= 32 ? ~0u : (n <= 0 ? 0u : (1u << n) - 1u);
}

// Orders a wave's LDS accesses before and after it across its lanes.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Zeros the rows of a V slab (rows of CPR 16-byte chunks, the layout that kLoads 1-KiB DMA loads
// wrote) whose bit of `keep` is not set: keys that count for no row, whose slab rows hold
// another key's values or the pool's slot 0 and would get infinities past a probability of 0.
template <int CPR, int kLoads>
__device__ __forceinline__ void zero_rows(char* slab, uint32_t keep) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < kLoads; ++i)
    if (!((keep >> (i * (64 / CPR) + lane / CPR)) & 1u))
      *reinterpret_cast<dsp_u32x4*>(slab + i * 1024 + 16 * lane) = dsp_u32x4{0u, 0u, 0u, 0u};
}

// ---- infinities and NaN of V on tiles whose rows see different keys.  A key that a row does not
// see has probability 0, but 0 * inf is NaN.  So in chunks that some row does not see whole,
// such values are found (any_nonfinite), added to the rows that see them (odd_operand against
// kHuge for every key seen) and cleared in LDS (clear_nonfinite) before P.V.
template <typename Tag>
constexpr uint32_t exp_bits() {  // an infinity's bits; above it, NaN
  return std::is_same<Tag, Bf16Tag>::value ? 0x7f80u : 0x7c00u;
}
constexpr uint32_t kHuge = 0x7f00u;  // 2^127 in bf16: its square overflows the accumulator

// Whether any lane's part of the kLoads KiB at `slab` holds an infinity or NaN (wave-uniform).
template <typename Tag, int kLoads>
__device__ __forceinline__ bool any_nonfinite(const char* slab) {
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  u16x2 top = {0, 0};
#pragma unroll 4
  for (int i = 0; i < kLoads; ++i) {
    const dsp_u32x4 v =
        *reinterpret_cast<const dsp_u32x4*>(slab + i * 1024 + 16 * (threadIdx.x & 63));
#pragma unroll
    for (int j = 0; j < 4; ++j)
      top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, v[j] & 0x7fff7fffu));
  }
  return __ballot(top[0] >= exp_bits<Tag>() || top[1] >= exp_bits<Tag>()) != 0;
}

template <typename Tag, int kLoads>
__device__ __forceinline__ void clear_nonfinite(char* slab) {
#pragma unroll 4
  for (int i = 0; i < kLoads; ++i) {
    dsp_u32x4* p = reinterpret_cast<dsp_u32x4*>(slab + i * 1024 + 16 * (threadIdx.x & 63));
    dsp_u32x4 v = *p;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if ((v[j] & 0x7fffu) >= exp_bits<Tag>()) v[j] &= 0xffff0000u;
      if ((v[j] & 0x7fff0000u) >= exp_bits<Tag>() << 16) v[j] &= 0xffffu;
    }
    *p = v;
  }
}

// A bf16 operand (whatever the cache's type: the lane layouts are the same) of kHuge where v is
// +inf or NaN (minus false), of -kHuge where it is -inf or NaN (minus true), 0 elsewhere.  The
// MFMA of both with kHuge for the keys a row sees adds inf, -inf, or inf - inf = NaN to it (the
// bf16 MFMA rounds a product to infinity before it adds it to an infinite sum).
template <typename Tag>
__device__ __forceinline__ dsp_u32x4 odd_operand(dsp_u32x4 v, bool minus) {
  auto code = [minus](uint32_t h) {
    const bool odd = minus ? (h & 0x7fffu) > exp_bits<Tag>() || h == (0x8000u | exp_bits<Tag>())
                           : (h & 0x7fffu) > exp_bits<Tag>() || h == exp_bits<Tag>();
    return odd ? kHuge | (minus ? 0x8000u : 0u) : 0u;
  };
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = code(v[j] & 0xffffu) | code(v[j] >> 16) << 16;
  return v;
}

}  // namespace dsp_mfma
