// fp32 contractions on the bf16 matrix cores (gfx950), without giving up fp32
// precision.
//
// An fp32 number is the exact sum of three bf16 numbers: x = h + m + l, where h
// keeps the sign, the exponent and the top 8 significand bits of x (its upper
// 16 bits), m the next 8 and l the last 8 (both differences are exact in fp32,
// and at most 16 and 8 bits wide).  A product x*y is then nine bf16 products,
// each exact in fp32, of which the MFMA sums the six that reach fp32 precision:
//   x y = h h' + (h m' + m h') + (h l' + l h' + m m')  + [m l' + l m' + l l']
// The three left out are below 2^-23 of |x y| together (2^-25 on average); an
// fp32 sum rounds its result by as much.  The six products go to two
// accumulators -- h h' to one, the small five to the other -- added once at the
// end: a small product added to a large accumulator inside the MFMA would lose
// its low bits at every step (measured over K = 2048 products of one sign: one
// accumulator 3.5e-6 relative error, two 2.5e-7, the fp32 MFMA 7.0e-7; K = 64
// of either sign 7.8e-8 against 1.4e-7 of the fp32 MFMA).
//
// Why: v_mfma_f32_32x32x16_bf16 does 32768 flops in 32 cycles, v_mfma_f32_16x16x4
// (fp32) 2048 in 32, so six bf16 products take 0.375 of the fp32 matrix time;
// and a bf16 MFMA leaves the VALU issue slots beside it free (measured: 64 VALU
// operations between 16 32x32x16 MFMAs cost 3%, an fp32 MFMA and a VALU
// operation do not overlap at all).
//
// MFMA operand layout (v_mfma_f32_32x32x16_bf16, wave64, lane group g = l/32):
//   A (32x16): lane l supplies A[m = l%32][k = 8g + j], j = 0..7
//   B (16x32): lane l supplies B[k = 8g + j][n = l%32]
//   D (32x32): lane l holds    D[m = 8(i/4) + 4g + i%4][n = l%32], i = 0..15
// The contraction index k can be mapped to any physical index as long as A and
// B agree.
#pragma once
#include "wha_device.hpp"

namespace wha {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// The three bf16 parts of a pair of floats, each pair packed in one register
// (first float in the low half).
struct SplitPair {
  unsigned h, m, l;
};
__device__ __forceinline__ unsigned pack_hi16(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302);
}
__device__ __forceinline__ float top16(float x) { return __uint_as_float(__float_as_uint(x) & 0xffff0000u); }
__device__ __forceinline__ SplitPair split_pair(float a, float b) {
  SplitPair s;
  s.h = pack_hi16(a, b);
  const float am = a - top16(a), bm = b - top16(b);
  s.m = pack_hi16(am, bm);
  s.l = pack_hi16(am - top16(am), bm - top16(bm));
  return s;
}

// One MFMA operand (8 k values of one row or column) in its three parts.
struct Frag3 {
  bf16x8 h, m, l;
};
__device__ __forceinline__ Frag3 split_frag(const float (&x)[8]) {
  uintx4 h, m, l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const SplitPair s = split_pair(x[2 * i], x[2 * i + 1]);
    h[i] = s.h;
    m[i] = s.m;
    l[i] = s.l;
  }
  return Frag3{__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)};
}

__device__ __forceinline__ floatx16 mfma_bf16(bf16x8 a, bf16x8 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// The five small products, smallest first.
__device__ __forceinline__ floatx16 mfma_small(const Frag3& a, const Frag3& b, floatx16 c) {
  c = mfma_bf16(a.l, b.h, c);
  c = mfma_bf16(a.h, b.l, c);
  c = mfma_bf16(a.m, b.m, c);
  c = mfma_bf16(a.m, b.h, c);
  return mfma_bf16(a.h, b.m, c);
}
__device__ __forceinline__ floatx16 zero16() {
  floatx16 z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.f;
  return z;
}

}  // namespace wha
