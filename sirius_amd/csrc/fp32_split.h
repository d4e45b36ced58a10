// fp32 products on the bf16 matrix pipes.
//
// An fp32 value is the exact sum of three bf16 values (8 + 8 + 8 bits of mantissa): x = x0 + x1 + x2 with x0 = x rounded to
// bf16, x1 = the rest rounded to bf16, x2 = what is left.  Of the nine products of two such sums eight go through
// v_mfma_f32_32x32x16_bf16, which accumulates in fp32: 256 cycles for a 32 x 32 x 16 product instead of the 512 of eight
// v_mfma_f32_32x32x2_f32.  The ninth, x2 y2, is below 2^-36 of the product, less than what the sum of the small products is rounded by.
//
// Error: the seven small products have an accumulator of their own, 2^-8 of the size of the other, so that the large one is
// rounded once per 16 reduction elements (fp32 MFMA: once per element), and a sum of one product is rounded as fp32 rounds it.  Norm of
// the error against 64 bits over the norm of the result, 128 x 128 tiles, in units of 1e-7, with fp32 MFMA and in parts:
//   normal x normal over 136 / 768 / 4608:   2.1 / 4.9 / 12.2   and 0.7 / 1.6 / 4.2
//   ReLU'd x normal:                         1.5 / 3.5 / 8.6    and 0.5 / 1.2 / 3.5
// (In one accumulator 4.2 over 768.)  Without x1 y2 and x2 y1 a sum of one product is off by 0.62 units in the last place instead of 0.5.
// Rounding the parts matters: cut off instead, they leave out products of one sign (uniform x uniform over 4608: 116 for 6.3).
// Time: taking a pair of values apart is 11 vector instructions, which pass behind the multiplies; what is left of a small product is
// its operands' way to the CU.
// Range: bf16 has the exponents of fp32, but a first part may be larger than its value (by 2^-9 of it), and with it a first product or
// a sum of them: these overflow up to 0.8 % below the largest fp32 value, and a value that rounds to 2^128 is an infinity in its
// first part.  Infinities and NaN among the operands come out as NaN (inf - inf).  So a kernel that finds a sum that is not finite,
// infinity or NaN, adds all of them up again with fp32 MFMA, whose result counts then: where fp32 has infinities too that costs
// the second pass only.
// Below 2^-110 (7.7e-34) the last parts of a value are bf16 denormals: such an operand keeps an absolute error of up to 2^-134.
#pragma once

#include "kernels.h"
#include <cfloat>

namespace tch {

struct Split8 {
  bf16x8_t part[3];
};

// a pair of values into the bits of its parts
__device__ inline void split_pair(float v0, float v1, uint32_t (&w)[3]) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const f32x2_t v = {v0, v1};
    w[k] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
    if (k < 2) {   // exact
      v0 -= __uint_as_float(w[k] << 16);
      v1 -= __uint_as_float(w[k] & 0xffff0000u);
    }
  }
}

__device__ inline void split4(const Chunk& c, uint2 (&w)[3]) {
  uint32_t a[3], b[3];
  split_pair(c.f[0], c.f[1], a);
  split_pair(c.f[2], c.f[3], b);
#pragma unroll
  for (int k = 0; k < 3; ++k) w[k] = make_uint2(a[k], b[k]);
}

// eight reduction elements of one operand row: `lo` and `hi` are two chunks of four
__device__ inline Split8 split8(const Chunk& lo, const Chunk& hi) {
  Split8 s;
  uint2 a[3], b[3];
  split4(lo, a);
  split4(hi, b);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    Chunk c;
    c.u = make_uint4(a[k].x, a[k].y, b[k].x, b[k].y);
    s.part[k] = c.h;
  }
  return s;
}

// Eight reduction elements of one column of bf16 values that lie [reduction][column] in LDS: ds_read_b64_tr_b16 hands a lane
// four of them, from the addresses of its group of 16 lanes.
__device__ inline bf16x8_t read_transposed(const unsigned char* first, const unsigned char* second) {
  typedef short s16x4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4_t* lds_ptr;
  const s16x4_t a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)first), b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)second);
  return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// large += x0 y0; small += the seven products next in size
__device__ inline void mma_split(const Split8& x, const Split8& y, f32x16_t& large, f32x16_t& small) {
  small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x.part[1], y.part[2], small, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x.part[2], y.part[1], small, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x.part[0], y.part[2], small, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x.part[2], y.part[0], small, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x.part[1], y.part[1], small, 0, 0, 0);
  large = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x.part[0], y.part[0], large, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x.part[0], y.part[1], small, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x.part[1], y.part[0], small, 0, 0, 0);
}

// large += small; whether any sum of this lane is not finite
template <int TM, int TN>
__device__ inline bool join_split(f32x16_t (&large)[TM][TN], const f32x16_t (&small)[TM][TN]) {
  bool beyond = false;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        large[i][j][e] += small[i][j][e];
        beyond |= !(fabsf(large[i][j][e]) <= FLT_MAX);
      }
  return beyond;
}

template <int TM, int TN>
__device__ inline void clear(f32x16_t (&acc)[TM][TN]) {
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
}

}  // namespace tch
