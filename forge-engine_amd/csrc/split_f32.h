// float32 products on the matrix cores' bfloat16 instruction.  Every operand is the sum of three bfloat16 numbers, x = x0 + x1 + x2
// exactly (24 bits of a float32 are three times eight; each part the rounding of what the parts before leave), and of the nine
// products of the parts the six largest are added up in float32: x0 y0 + x0 y1 + x1 y0 + x1 y1 + x0 y2 + x2 y0.  The three left out
// are below 2^-25 of |x y| together, where a product rounded to float32 is off by half as much; what a sum loses otherwise is the
// rounding of its own steps, of which there are fewer.
//
// A part of a number that is infinite, or rounds to that, is no number, and so is every sum that it is part of: a result that is not
// finite is made again in float32 alone, product by product.  A bfloat16 number's last bit is 2^-133 at the least: a number below 2^-110 loses
// up to 2^-134 with its last part.  (Operands scaled by 2^16 ahead of the split lose nothing; the two instructions a pair cost the product
// of 700 x 4,096 x 1,024 46.5 -> 49.6 us, for numbers that beside any of ordinary size do not reach a sum's last bit.)
#pragma once
#include "common.h"

namespace split_f32 {

typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float floatx4;
typedef __attribute__((ext_vector_type(4))) unsigned int uintx4;

// (-1, 0) and (0, -1), which a dot product subtracts one part of a pair with, exactly.  The compiler must not see them: it makes a
// constant of -1.0 of the first, which the instruction takes for a pair of them.
struct Minus {
  bf16x2 first, second;
};
__device__ __forceinline__ Minus minus() {
  unsigned low = 0x0000bf80u, high = 0xbf800000u;
  asm("" : "+s"(low));
  asm("" : "+s"(high));
  return {__builtin_bit_cast(bf16x2, low), __builtin_bit_cast(bf16x2, high)};
}

// two floats as three pairs of bfloat16: 3.5 instructions each
__device__ __forceinline__ void split2(float x0, float x1, const Minus& minus, unsigned& high, unsigned& middle, unsigned& low) {
  const bf16x2 h = {(__bf16)x0, (__bf16)x1};
  const float r0 = __builtin_amdgcn_fdot2_f32_bf16(h, minus.first, x0, false), r1 = __builtin_amdgcn_fdot2_f32_bf16(h, minus.second, x1, false);
  const bf16x2 m = {(__bf16)r0, (__bf16)r1};
  const float s0 = __builtin_amdgcn_fdot2_f32_bf16(m, minus.first, r0, false), s1 = __builtin_amdgcn_fdot2_f32_bf16(m, minus.second, r1, false);
  const bf16x2 l = {(__bf16)s0, (__bf16)s1};
  high = __builtin_bit_cast(unsigned, h);
  middle = __builtin_bit_cast(unsigned, m);
  low = __builtin_bit_cast(unsigned, l);
}
// a lane's eight elements of an operand of the 16x16x32 instruction
__device__ __forceinline__ void split8(floatx4 u, floatx4 v, const Minus& minus, bf16x8 (&parts)[3]) {
  uintx4 p[3];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    unsigned a, b, c;
    split2(u[2 * e], u[2 * e + 1], minus, a, b, c);
    p[0][e] = a; p[1][e] = b; p[2][e] = c;
    split2(v[2 * e], v[2 * e + 1], minus, a, b, c);
    p[0][2 + e] = a; p[1][2 + e] = b; p[2][2 + e] = c;
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) parts[i] = __builtin_bit_cast(bf16x8, p[i]);
}

// The same, the same bits, in 5.5 instructions each of the kind that runs beside the matrix cores.  (The dot product with (-1, 0) takes a part off its number in one instruction instead of two, but holds
// those up: a step of 128 x 128 2.25 -> 2.08 us.  Where splitting itself is the bound, as in gemm_split, that form is the faster one.)
__device__ __forceinline__ void split2(float x0, float x1, unsigned& high, unsigned& middle, unsigned& low) {
  high = __builtin_bit_cast(unsigned, bf16x2{(__bf16)x0, (__bf16)x1});
  const float r0 = x0 - __uint_as_float(high << 16), r1 = x1 - __uint_as_float(high & 0xffff0000u);
  middle = __builtin_bit_cast(unsigned, bf16x2{(__bf16)r0, (__bf16)r1});
  const float s0 = r0 - __uint_as_float(middle << 16), s1 = r1 - __uint_as_float(middle & 0xffff0000u);
  low = __builtin_bit_cast(unsigned, bf16x2{(__bf16)s0, (__bf16)s1});
}
__device__ __forceinline__ void split8(floatx4 u, floatx4 v, bf16x8 (&parts)[3]) {
  uintx4 p[3];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    unsigned a, b, c;
    split2(u[2 * e], u[2 * e + 1], a, b, c);
    p[0][e] = a; p[1][e] = b; p[2][e] = c;
    split2(v[2 * e], v[2 * e + 1], a, b, c);
    p[0][2 + e] = a; p[1][2 + e] = b; p[2][2 + e] = c;
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) parts[i] = __builtin_bit_cast(bf16x8, p[i]);
}

// acc(i) += first operand b x second operands a[i], i < COUNT, over 32 of K.  The products of the first parts go into the long sum; the
// others, a 2^8th of their size, are added up by themselves first, so that the long sum is rounded twice for all six and not six
// times.  (The instruction cuts off what an addend has below the last bit of a larger one, downwards: a sum that the small products
// begin and the large ones end is too small by 3e-8 on the average, which the layers of a model add up.)
template <int COUNT, typename Acc>
__device__ __forceinline__ void add_products(const bf16x8 (&a)[COUNT][3], const bf16x8 (&b)[3], Acc acc) {
  constexpr int OF_A[5] = {2, 0, 1, 1, 0}, OF_B[5] = {0, 2, 1, 0, 1};
  floatx4 sum[COUNT];
#pragma unroll
  for (int p = 0; p < 5; ++p)
#pragma unroll
    for (int i = 0; i < COUNT; ++i)
      sum[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[OF_B[p]], a[i][OF_A[p]], p == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : sum[i], 0, 0, 0);
#pragma unroll
  for (int i = 0; i < COUNT; ++i) acc(i) = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[0], a[i][0], acc(i), 0, 0, 0);
#pragma unroll
  for (int i = 0; i < COUNT; ++i) acc(i) += sum[i];
}

// The same with the sum of the others kept apart to the end.
__device__ __forceinline__ void add_products_apart(const bf16x8 (&a)[3], const bf16x8 (&b)[3], floatx4& large, floatx4& small) {
  small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[0], a[2], small, 0, 0, 0);
  large = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[0], a[0], large, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[2], a[0], small, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[1], a[1], small, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[0], a[1], small, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[1], a[0], small, 0, 0, 0);
}

__device__ __forceinline__ bool finite(float v) { return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u; }
// The sum product by product, up to where it stays no number.  (A request gone wrong brings a row of those beside the others: 700 x 4,096 x
// 1,024 with one such row 1,080 -> 75 us, 300 x 2,048 x 6,144 of nothing else 11,900 -> 133; an infinity keeps the whole walk.)
__device__ __forceinline__ float dot(const float* x, const float* y, int count) {
  float sum = 0.f;
  for (int k = 0; k < count && sum == sum; k += 8) {
    const int end = min(k + 8, count);
    for (int i = k; i < end; ++i) sum = __fmaf_rn(x[i], y[i], sum);
  }
  return sum;
}

}  // namespace split_f32
