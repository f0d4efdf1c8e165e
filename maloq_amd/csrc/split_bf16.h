#pragma once
// fp32 products on the bf16 matrix cores.
//
// A float is the sum of three bf16 numbers: its leading 8 bits, the next 8 and
// the rest (the three-way split of Henry, Tang and Heinecke, "Leveraging the
// bfloat16 artificial intelligence datatype for higher-precision computations",
// 2019).  Of the nine products of two such sums the six down to 2^-16 of the
// leading one are formed and added in fp32 by the MFMA, smallest first.  What is
// left out is below 2^-22 of a product (the leading plane is truncated, so the
// others reach 2^-7 and 2^-16 of the number), and 2^-25.5 of it rms.  Sums of 640
// products of normal numbers are off by 3.8e-7 (rms), the fp32 MFMA's by 4.6e-7; of
// 3200 by 8.8e-7 and 1.01e-6.  It is 2.67 times as fast: six
// v_mfma_f32_32x32x16_bf16 of 32 cycles where the fp32 units take eight
// v_mfma_f32_32x32x2_f32 of 64.
//
// Range: the planes are bf16, whose least number is 2^-133, so that a float below
// 2^-109 loses its last bits.  A product beyond the floats is infinite; from 2^144 on
// it may be NaN (its parts are infinite too, and the third plane's may have the other
// sign).  Infinite operands: see fix_inf.
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace maloq {

typedef float split_f2 __attribute__((ext_vector_type(2)));
typedef __bf16 split_b2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  const split_b2 t = __builtin_convertvector(split_f2{a, b}, split_b2);
  return __builtin_bit_cast(uint32_t, t);
}

// The three planes of v, element k in 16-bit lane k of each.  The leading plane
// is truncated, so that no finite value rounds up to infinity.
__device__ __forceinline__ void split8(const float (&v)[8], uint4 (&p)[3]) {
  uint32_t w[3][4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t u0 = __float_as_uint(v[2 * k]), u1 = __float_as_uint(v[2 * k + 1]);
    w[0][k] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
    float r0 = v[2 * k] - __uint_as_float(u0 & 0xffff0000u), r1 = v[2 * k + 1] - __uint_as_float(u1 & 0xffff0000u);
    w[1][k] = pack_bf16(r0, r1);
    r0 -= __uint_as_float(w[1][k] << 16);
    r1 -= __uint_as_float(w[1][k] & 0xffff0000u);
    w[2][k] = pack_bf16(r0, r1);
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) p[i] = make_uint4(w[i][0], w[i][1], w[i][2], w[i][3]);
}

// Infinities.  split8 makes (+-inf, NaN, NaN) of one, which gives NaN where the fp32
// units give infinity.  A kernel whose sums hold one that is not finite therefore forms
// them again with fix_inf after each split (a test of the operands themselves, on the
// vector unit beside the splits, took 1.5 % of the time).
__device__ __forceinline__ float not_finite(float t, float v) { return fmaf(v, 0.f, t); }  // t, or NaN

// Such a lane's 16 bytes of planes in LDS, `plane` bytes apart: (+-1, 0, +-inf).  The
// third plane meets only the other operand's leading one, so that the product with any
// number of 2^-133 or more is infinity, with its sign, and with zero NaN.  (NaNs stay
// NaN, but for signalling ones with none of their upper bits set.)
__device__ __forceinline__ void fix_inf(char* at, int plane) {
#pragma unroll 1
  for (int k = 0; k < 4; ++k) {
    uint32_t* p0 = reinterpret_cast<uint32_t*>(at) + k;
    uint32_t *p1 = p0 + plane / 4, *p2 = p1 + plane / 4;
    const uint32_t a = *p0, sign = a & 0x80008000u;
    const uint32_t m = ((a & 0x7fffu) == 0x7f80u ? 0xffffu : 0u) | ((a & 0x7fff0000u) == 0x7f800000u ? 0xffff0000u : 0u);
    *p0 = (a & ~m) | (m & (sign | 0x3f803f80u));
    *p1 &= ~m;
    *p2 = (*p2 & ~m) | (m & (sign | 0x7f807f80u));
  }
}

// The six products in the order they are added: planes (a, b).
constexpr int SPLIT_PRODUCTS = 6;
__host__ __device__ constexpr int split_a(int k) { constexpr int t[6] = {0, 2, 1, 0, 1, 0}; return t[k]; }
__host__ __device__ constexpr int split_b(int k) { constexpr int t[6] = {2, 0, 1, 1, 0, 0}; return t[k]; }

}  // namespace maloq
