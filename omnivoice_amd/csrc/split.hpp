// Float32 products on the bf16 matrix cores.
//
// A float32 value is the sum of three bf16 parts, each the rounding of what
// the ones before it leave (hi, mid, lo: 8 + 8 + 8 significant bits; see the
// end of this comment for the largest and the smallest values), and six
// of the nine products of two such triples are summed in float32: hi hi in
// one accumulator; hi mid, mid hi, mid mid, hi lo and lo hi in a second one,
// added at the end. What is left out is below 2^-24 of the product, half a
// unit in the last place of float32, and a 16-deep product rounds its sum
// once where the float32 matrix cores' 2-deep one rounds eight times, so the
// sum is nearer to the exact one than theirs. At 16 times the rate of
// v_mfma_f32_32x32x2_f32, six products are 2.7 times its throughput.
//
// Finite values of 0x1.FFp127 (3.396e38) and more round to infinity in the
// first part. Operands that are split once and stored (weights, the
// attention's heads) hold it to bf16's largest value. A convolution's input
// is split for every tile, without the three operations more a value; there
// such a value makes the sum infinite or NaN. Every sum that is not finite,
// for this reason or another, is formed again in double, from the values
// themselves.
// At the other end bf16's parts stop at 2^-133: an operand is kept to 2^-24
// of itself, but to no less than 2^-134, which is more below 2^-110. (The
// matrix cores take and keep bf16's subnormal values.)
#ifndef OMNIVOICE_AMD_SPLIT_HPP_
#define OMNIVOICE_AMD_SPLIT_HPP_

#include <hip/hip_runtime.h>

#include "common.hpp"

namespace ovg {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

// Two values as a packed bf16 pair (to nearest even), the first in the low
// half, and what the pair leaves of them.
__device__ __forceinline__ unsigned RoundPair(floatx2 v) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ floatx2 Rest(floatx2 v, unsigned pair) {
  return floatx2{v[0] - __builtin_bit_cast(float, pair << 16),
                 v[1] - __builtin_bit_cast(float, pair & 0xFFFF0000U)};
}

// What the first part is rounded from: finite values of 0x1.FFp127 and more,
// which would round to infinity, are held to bf16's largest one and have the
// difference in the other parts.
__device__ __forceinline__ float First(float v) {
  constexpr float kMost = 0x1.FEp127F;
  return fabsf(v) < __builtin_inff() ? fminf(fmaxf(v, -kMost), kMost) : v;
}

// Eight values as the three parts of one 16-byte matrix-core operand, of any
// float32 (WIDE) or of those below 0x1.FFp127. An infinite or NaN value has
// it in the first part and NaN in the others, which only the second
// accumulator sees.
template <bool WIDE>
__device__ __forceinline__ void Split8(const float* v, uintx4* part) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    floatx2 rest{v[2 * q], v[2 * q + 1]};
    part[0][q] = RoundPair(WIDE ? floatx2{First(rest[0]), First(rest[1])} : rest);
    rest = Rest(rest, part[0][q]);
    part[1][q] = RoundPair(rest);
    rest = Rest(rest, part[1][q]);
    part[2][q] = RoundPair(rest);
  }
}

// 32x32x16 bf16 MFMA, the layout of Mfma32 (common.hpp).
__device__ __forceinline__ floatx16 MfmaBf16(uintx4 a, uintx4 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// The sum of the two accumulators; the first alone where it is infinite or
// NaN (the second is NaN wherever an operand was infinite).
__device__ __forceinline__ float Join(float main, float rest) {
  return __builtin_isfinite(main) ? main + rest : main;
}

// A kernel's parameters (its only argument), read again: what the rare code
// for sums that are not finite uses of them needs no scalar registers before
// it. With those kept from a kernel's start its launches took 0.2 us longer.
template <typename Params>
__device__ __forceinline__ const Params& ParamsAgain() {
  using Kernarg = __attribute__((address_space(4))) const Params;
  auto at = reinterpret_cast<std::uintptr_t>(
      (__attribute__((address_space(4))) const void*)__builtin_amdgcn_kernarg_segment_ptr());
  asm volatile("" : "+s"(at));
  return *(const Params*)reinterpret_cast<Kernarg*>(at);
}

}  // namespace ovg

#endif  // OMNIVOICE_AMD_SPLIT_HPP_
