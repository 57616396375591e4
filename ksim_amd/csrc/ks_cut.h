// fp32 values as sums of three bf16 values, for products of fp32 operands on the bf16 matrix instructions (ks_mlp.hip, ks_gru.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace ks {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;  // a 16-byte register vector (plain vector type, so arrays of it stay in registers)

// An fp32 value is cut into three bf16 values (Henry, Tang and Heinecke, ARITH 2019) whose sum is the value itself: its upper 16 bits (8 bits of mantissa, so infinities and NaN
// stay in the first part), the rest, below 2^-7 of it, rounded to bf16, and what that leaves, below 2^-16 and at most 8 bits.  Of the nine
// products of two cut values the eight that reach 2^-24 of the result are added up: the largest in an accumulator of its own, with one rounding
// per 16 k where the fp32 instruction has eight, the other seven, below 2^-6 of it, in a second one; the ninth is below 2^-32.  A reduction of
// one term, or one term among zeros, then rounds once, as the fp32 product does (without the products of second and third parts, 2^-23 each at
// most, it was 3.9 roundings off), and longer ones round less than on the fp32 instruction: relative error against 64 bits, in 2^-24,
// 0.43 -> 0.43 for 1 term, 0.73 -> 0.46 for 5, 3.4 -> 1.1 for 128, 6.5 -> 2.0 for 475.  Eight instructions replace eight of twice their time.
// Range: bf16 ends at 2^-133, so a value below 2^-110 loses what lies under 2^-134 of it: at most 2^-133 times the other operand.
__device__ __forceinline__ unsigned pack_bf16(float lo, float hi) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}

// the three parts of two values, each part's two bf16 in one register
__device__ __forceinline__ void cut_pair(float a, float b, unsigned (&out)[3]) {
#pragma clang fp contract(off)  // a product that comes in is rounded before it is cut
  const unsigned ua = __builtin_bit_cast(unsigned, a), ub = __builtin_bit_cast(unsigned, b);
  out[0] = __builtin_amdgcn_perm(ub, ua, 0x07060302);  // the upper halves
  a -= __builtin_bit_cast(float, ua & 0xffff0000u);
  b -= __builtin_bit_cast(float, ub & 0xffff0000u);
  const unsigned w = pack_bf16(a, b);
  out[1] = w;
  out[2] = pack_bf16(a - __builtin_bit_cast(float, w << 16), b - __builtin_bit_cast(float, w & 0xffff0000u));
}

// eight values to PARTS fragments; PARTS = 1 rounds them to bf16
template <int PARTS>
__device__ __forceinline__ void cut_bf16(const float (&v)[8], u32x4 (&out)[PARTS]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if constexpr (PARTS == 1) {
      out[0][q] = pack_bf16(v[2 * q], v[2 * q + 1]);
    } else {
      unsigned part[3];
      cut_pair(v[2 * q], v[2 * q + 1], part);
      out[0][q] = part[0]; out[1][q] = part[1]; out[2][q] = part[2];
    }
  }
}

// Where the products overflow, or an operand was infinite or NaN, the first parts alone decide: the others of an infinity are NaN.
__device__ __forceinline__ float join_cut(float acc, float low) { return fabsf(acc) < __builtin_inff() ? acc + low : acc; }

}  // namespace ks
