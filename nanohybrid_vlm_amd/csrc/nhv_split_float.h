// Products of floats on the bfloat16 matrix cores: 2^16 times a float as the sum of three bfloat16 numbers.
//
// high = 2^16 x rounded to 8 bits, middle = (2^16 x - high) rounded, rest = 2^16 x - high - middle. Both differences are exact (a
// float has 24 bits; each part takes 8 and its sign one more), and so is the rest's conversion: high + middle + rest = 2^16 x, bit
// for bit. That holds for every float, denormals too: floats end at 2^-149, the bfloat16 denormals (which the instructions used
// here keep) at 2^-133, and the factor brings the one to the other. (Without it the parts of x below 2^-109 lost what lies under
// 2^-133: products of entries near 1e-34 were off by 2.8e-7, near 1e-36 by 2.7e-5.) At the other end 2^16 x is infinite from
// 2^112 on, as is a sum of products from 2^96 on.
#pragma once
#include "nhv_common.h"

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef bf16_t bf16x2 __attribute__((ext_vector_type(2)));
typedef bf16_t bf16x4 __attribute__((ext_vector_type(4)));
typedef bf16_t bf16x8 __attribute__((ext_vector_type(8)));

constexpr float SPLIT_SCALE = 0x1p16f;                   // of an operand
constexpr float SPLIT_UNSCALE = 0x1p-32f;                // of a sum of products

struct SplitFloats4 { bf16x4 high, middle, rest; };
struct SplitFloats8 { bf16x8 high, middle, rest; };

// (a, b) rounded to bfloat16, and what that leaves of them in their place, exactly either way.
// DOTS: by a dot product with (-1, 0), one instruction where the widening and the subtraction are two. (The two pairs come from scalar
// registers that the compiler does not see through: it would write the first as the inline constant -1.0, which the instruction reads
// as another pair, and every first entry's parts came out wrong.) It does not run beside matrix instructions, which the two do where
// these leave room: 32x32x16 ones (1,500 x 12,288 . 2048 454 us, with dots 20 more), not the 16x16x32 ones of the other kernels
// (6 x 2048 . 2048 9.4 us without dots, 8.7 with; 1 x 2048 . 6144 18.8, 17.6; 20 x 3072 . 1001, whose loads the compiler then leaves in
// scratch memory, 46 and 16).
template <bool DOTS>
__device__ __forceinline__ bf16x2 take_high(float& a, float& b) {
  const bf16x2 high = __builtin_convertvector((f32x2{a, b}), bf16x2);
  if constexpr (DOTS) {
    uint32_t first = 0x0000bf80u, second = 0xbf800000u;
    asm("" : "+s"(first));
    asm("" : "+s"(second));
    a = __builtin_amdgcn_fdot2_f32_bf16(high, __builtin_bit_cast(bf16x2, first), a, false);
    b = __builtin_amdgcn_fdot2_f32_bf16(high, __builtin_bit_cast(bf16x2, second), b, false);
  } else {
    const uint32_t bits = __builtin_bit_cast(uint32_t, high);
    a -= __builtin_bit_cast(float, bits << 16);
    b -= __builtin_bit_cast(float, bits & 0xffff0000u);
  }
  return high;
}

template <bool DOTS>
__device__ __forceinline__ SplitFloats4 split_floats(f32x4 v) {
  SplitFloats4 p;
#pragma unroll
  for (int i = 0; i < 4; i += 2) {
    float a = v[i] * SPLIT_SCALE, b = v[i + 1] * SPLIT_SCALE;
    const bf16x2 high = take_high<DOTS>(a, b), middle = take_high<DOTS>(a, b), rest = __builtin_convertvector((f32x2{a, b}), bf16x2);
    p.high[i] = high[0], p.high[i + 1] = high[1];
    p.middle[i] = middle[0], p.middle[i + 1] = middle[1];
    p.rest[i] = rest[0], p.rest[i + 1] = rest[1];
  }
  return p;
}

template <bool DOTS>
__device__ __forceinline__ SplitFloats8 split_floats(f32x4 v0, f32x4 v1) {
  const SplitFloats4 p = split_floats<DOTS>(v0), q = split_floats<DOTS>(v1);
  return {__builtin_shufflevector(p.high, q.high, 0, 1, 2, 3, 4, 5, 6, 7),
          __builtin_shufflevector(p.middle, q.middle, 0, 1, 2, 3, 4, 5, 6, 7),
          __builtin_shufflevector(p.rest, q.rest, 0, 1, 2, 3, 4, 5, 6, 7)};
}

// eight entries whose parts lie PLANE entries apart (in LDS)
template <int PLANE>
__device__ __forceinline__ SplitFloats8 split_at(const bf16_t* p) {
  return {*reinterpret_cast<const bf16x8*>(p), *reinterpret_cast<const bf16x8*>(p + PLANE),
          *reinterpret_cast<const bf16x8*>(p + 2 * PLANE)};
}

// One of the six products of a block of 32 k: the one of the high parts goes to `high`, the five small ones to `low`.
__device__ __forceinline__ void split_product(int step, const SplitFloats8& a, const SplitFloats8& b, f32x4& high, f32x4& low) {
  if (step == 0) low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.middle, b.middle, low, 0, 0, 0);
  if (step == 1) low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.rest, b.high, low, 0, 0, 0);
  if (step == 2) low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.high, b.rest, low, 0, 0, 0);
  if (step == 3) low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.middle, b.high, low, 0, 0, 0);
  if (step == 4) low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.high, b.middle, low, 0, 0, 0);
  if (step == 5) high = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.high, b.high, high, 0, 0, 0);
}

// The same of a block of 16 k and 32 x 32 outputs. The matrix instructions add up eight k (a lane group's) at a time, one group's after
// another's, so that two of these in a row give the bits of one of the above.
__device__ __forceinline__ void split_product(int step, const SplitFloats8& a, const SplitFloats8& b, f32x16& high, f32x16& low) {
  if (step == 0) low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.middle, b.middle, low, 0, 0, 0);
  if (step == 1) low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.rest, b.high, low, 0, 0, 0);
  if (step == 2) low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.high, b.rest, low, 0, 0, 0);
  if (step == 3) low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.middle, b.high, low, 0, 0, 0);
  if (step == 4) low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.high, b.middle, low, 0, 0, 0);
  if (step == 5) high = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.high, b.high, high, 0, 0, 0);
}
