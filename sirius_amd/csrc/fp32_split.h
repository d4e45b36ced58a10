// fp32 products on the bf16 matrix pipes.
//
// An fp32 value is the exact sum of three bf16 values (8 + 8 + 8 bits of mantissa): x = x0 + x1 + x2 with x0 = the upper half of
// the bits of x, x1 = the upper half of the bits of what is left, x2 = the rest.  Of the nine products of two such sums eight go through
// v_mfma_f32_32x32x16_bf16, which accumulates in fp32: 256 cycles for a 32 x 32 x 16 product instead of the 512 of eight
// v_mfma_f32_32x32x2_f32.  The ninth, x2 y2, is below 2^-30 of the product, 2^-7 of a unit in the last place.
//
// Error: the seven small products have an accumulator of their own, 2^-5 of the size of the other at most, so that the large one is
// rounded once per 16 reduction elements (fp32 MFMA: once per element), and a sum of one product is rounded as fp32 rounds it.  Norm of
// the error against 64 bits over the norm of the result, 128 x 128 tiles, in units of 1e-7, with fp32 MFMA and in parts:
//   normal x normal over 136 / 768 / 4608:   2.1 / 4.9 / 12.2   and 0.7 / 1.6 / 4.2
//   ReLU'd x normal:                         1.5 / 3.5 / 8.6    and 0.5 / 1.2 / 3.5
//   uniform x uniform:                       1.7 / 4.2 / 10.1   and 0.7 / 1.5 / 3.6
// (In one accumulator 4.2 for normal x normal over 768.)
//
// Range: operands are taken apart times 2^24, and the sums multiplied by 2^-48 at the end.  The last bit of the smallest values is then a
// normal bf16 number, so that parts lose no bit of any value.  (Without the factor the last parts of values below 2^-110 are bf16
// denormals and cut off at 2^-134.)  At the other end parts overflow, from operands of 2^104 or sums of 2^80 on; they come out as
// infinity, or as NaN where infinities cancel.  A kernel that finds a sum that is not finite adds all of them up again
// with fp32 MFMA, whose result counts then: what fp32 makes of infinities, NaN and the largest values.
//
// Time: taking a pair of values apart is 13 vector instructions, which are what bounds small products.  Rounded parts (v_cvt_pk_bf16_f32
// instead of v_perm_b32, a shift for one of two masks) took 4 % longer over the forward products of the three models; rests by
// v_dot2_f32_bf16, 9 instructions, as long as those, and weight gradients 6 % longer.
#pragma once

#include "kernels.h"
#include <cfloat>

namespace tch {

constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-48f;

struct Split8 {
  bf16x8_t part[3];
};

// A pair of values, times kSplitScale, into the bits of its parts.
__device__ inline void split_pair(float v0, float v1, uint32_t (&w)[3]) {
  v0 *= kSplitScale;
  v1 *= kSplitScale;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    w[k] = __builtin_amdgcn_perm(__float_as_uint(v1), __float_as_uint(v0), 0x07060302u);
    if (k < 2) {
      v0 -= __uint_as_float(__float_as_uint(v0) & 0xffff0000u);
      v1 -= __uint_as_float(__float_as_uint(v1) & 0xffff0000u);
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

// large = (large + small) * kSplitUnscale; whether any sum of this lane is not finite
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
        large[i][j][e] *= kSplitUnscale;
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
