// split_bf16.h — fp32 products on the bf16 matrix cores without giving up fp32 precision.
//
// A float's 24 significand bits are exactly the sum of three bf16 values (8 bits each, the
// second and third rounded to nearest, so their signs vary): x = h + m + l. The product of two
// floats is then nine bf16 products, each exact in the matrix core's fp32 accumulation; the
// three smallest (m*l, l*m, l*l: together under 2^-23 of the product, of either sign) are left
// out, the other six are v_mfma_f32_32x32x16_bf16. Registers only, random operands: 1760 TFLOP/s of
// bf16 are 293 of these against 147 of v_mfma_f32_32x32x2_f32.
//
// Accumulation. The bf16 instruction aligns its 16 products and the accumulator to the largest of
// them and drops what falls off the end, downwards: added straight into a long sum, that costs
// more than the fp32 instruction's roundings (relative error of a 3x3 convolution over 64
// channels against float64: 3.6e-7, fp32 3.0e-7), and every step leaves a small negative bias. So
// the six products of a step are summed from zero, where little falls off, and added to the
// accumulator by an ordinary fp32 addition (1.3e-7); and the steps take turns between the product
// and its negative, which is subtracted, so that the biases cancel (without that, a weight gradient
// over 65536 pixels had a mean error of 5e-7 of its size).
//
// Range, low end: the third part of a float below 2^-110 would lie below bf16's normal numbers. Both
// operands are split times X3_SCALE, at which every part of every float, denormals included, is a
// normal bf16, and the addition behind a step's products takes the scale out again (powers of two:
// not a bit of an ordinary sum changes).
// High end: an operand that is infinite, NaN or above 2^104, and a sum above 2^80, leaves an infinity or
// NaN in every sum that it is part of, where fp32 would give one, or a number. Each wave looks at its
// finished sums, and those that are infinite or NaN are computed again with v_mfma_f32_32x32x2_f32,
// operands straight from memory, until each of them is NaN or complete (x3_redo): in a net that has
// diverged that is after some operands. Finite sums pay one multiplication each for the look. us with
// every input NaN / with ordinary ones: convolution 32 -> 64 of 64x64, batch 64, forward and backward 269 /
// 223; a step of the VGG-style stack after it has diverged (all weights of three layers NaN, 7 of 128
// filters of the fourth) / on finite values 4600 / 4340.
#pragma once
#include "common.h"

namespace tdh {
namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16_x3 __attribute__((ext_vector_type(16)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

constexpr int X3_PARTS = 3;  // h, m, l
constexpr float X3_SCALE   = 0x1p24f;   // of both operands when they are split
constexpr float X3_UNSCALE = 0x1p-48f;  // of a product of the two

// two floats to packed bf16 (round to nearest even), the first in the low half
__device__ __forceinline__ uint32_t pack_bf16(const float a, const float b) {
  const floatx2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ float low_bf16(const uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float high_bf16(const uint32_t p) { return __uint_as_float(p & 0xffff0000u); }

// the three parts of two floats (X3_SCALE times the operands)
__device__ __forceinline__ void split_pair(const float a, const float b, uint32_t (&part)[X3_PARTS]) {
  part[0]        = pack_bf16(a, b);
  const float ra = a - low_bf16(part[0]), rb = b - high_bf16(part[0]);
  part[1]        = pack_bf16(ra, rb);
  part[2]        = pack_bf16(ra - low_bf16(part[1]), rb - high_bf16(part[1]));
}

// acc[i][j] += sign * (a[i] * b[j]) of the unscaled operands over the 16*KS reduction indices of KS
// steps, smallest products first; sign is 1 or -1
template <int TM, int TN, int KS>
__device__ __forceinline__ void mfma_x3(floatx16_x3 (&acc)[TM][TN], const bf16x8 (&a)[KS][TM][X3_PARTS],
                                        const bf16x8 (&b)[KS][TN][X3_PARTS], const float sign) {
  constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    floatx16_x3 sum[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) sum[j] = floatx16_x3{};
#pragma unroll
    for (int q = 0; q < 6; ++q)
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          sum[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s][i][pa[q]], b[s][j][pb[q]], sum[j], 0, 0, 0);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = __builtin_fmaf(sum[j][r], sign * X3_UNSCALE, acc[i][j][r]);
      asm volatile("" : "+v"(acc[i][j]));  // (here and now: deferred, the sums pile up in memory)
    }
  }
}
template <int TM, int TN>
__device__ __forceinline__ void mfma_x3(floatx16_x3 (&acc)[TM][TN], const bf16x8 (&a)[TM][X3_PARTS],
                                        const bf16x8 (&b)[TN][X3_PARTS], const float sign) {
  mfma_x3<TM, TN, 1>(acc, reinterpret_cast<const bf16x8(&)[1][TM][X3_PARTS]>(a),
                     reinterpret_cast<const bf16x8(&)[1][TN][X3_PARTS]>(b), sign);
}

template <int N>
__device__ __forceinline__ bool x3_all_nan(const floatx16_x3 (&sum)[N]) {
  bool all = true;
#pragma unroll
  for (int b = 0; b < N; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) all = all && sum[b][r] != sum[b][r];
  return __all(all) != 0;
}
// A wave's N blocks of finished sums: the elements that are in use (element r of block b: used(b, r)) and
// infinite or NaN are computed once more. add_up(sum) adds all their products to sum, or stops when
// x3_all_nan(sum). The other elements stay as they are; in sum they are NaN.
template <int N, class Used, class AddUp>
__device__ __forceinline__ void x3_redo(floatx16_x3 (&acc)[N], const Used &used, const AddUp &add_up) {
  float probe = 0.0f;   // 0 * infinity and 0 * NaN are NaN
#pragma unroll
  for (int b = 0; b < N; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) probe = __builtin_fmaf(acc[b][r], 0.0f, probe);
  if (__builtin_expect(__any(!(probe == 0.0f)) == 0, 1)) return;
  uint32_t bad[N];
  floatx16_x3 sum[N];
#pragma unroll
  for (int b = 0; b < N; ++b) {
    bad[b] = 0;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      bad[b] |= (used(b, r) && !(__builtin_fabsf(acc[b][r]) <= 3.402823466e+38f) ? 1u : 0u) << r;
      sum[b][r] = bad[b] >> r & 1u ? 0.0f : __builtin_nanf("");
    }
  }
  add_up(sum);
#pragma unroll
  for (int b = 0; b < N; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[b][r] = bad[b] >> r & 1u ? sum[b][r] : acc[b][r];
}

}  // namespace
}  // namespace tdh
