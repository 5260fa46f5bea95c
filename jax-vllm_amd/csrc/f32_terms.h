// A float as the sum of three bf16 numbers (of 2^24 times the float, see gemm_f32.hip), and where the products of many rows want a row's terms:
// what a product of these rows would otherwise make in a launch of its own (6.4 us and a second pass over 1,003 x 2,048 floats) is left by the kernel that makes the rows.
#pragma once
#include "common.h"

#define G32_STEP 32            // columns of a step and of v_mfma_f32_16x16x32_bf16
#define G32_SCALE 0x1p24f
#define G32_UNSCALE 0x1p-48f

namespace f32_terms {
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// Pair i of a lane's 8 numbers: its part of the three terms of 2^24 times these.
__device__ __forceinline__ void split_pair(float a, float b, int i, u32x4 (&t)[3]) {
  a *= G32_SCALE, b *= G32_SCALE;
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    t[e][i] = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){a, b}, bf16x2));
    if (e < 2) {
      a -= __uint_as_float(t[e][i] << 16);
      b -= __uint_as_float(t[e][i] & 0xffff0000u);
    }
  }
}
__device__ __forceinline__ void split8(const f32x4 (&v)[2], u32x4 (&t)[3]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) split_pair(v[i / 2][i % 2 * 2], v[i / 2][i % 2 * 2 + 1], i, t);
}
// Columns 8 piece .. + 7 of row m, a multiple of 32 columns in `steps` steps: in the order of the operands of tiles of 128 rows,
// [M / 32][steps][term][16 columns][8 columns][32 rows][8] (fragments), or [M][steps][term][32].
__device__ __forceinline__ void leave_terms(unsigned* X, bool fragments, int steps, long long m, int piece, const f32x4 (&v)[2]) {
  u32x4 t[3];
  split8(v, t);
  const int s = piece >> 2, q = piece & 3;
  u32x4* out = (u32x4*)X + (fragments ? ((m >> 5) * steps + s) * 384 + (q >> 1) * 64 + (q & 1) * 32 + (m & 31) : (m * steps + s) * 12 + q);
#pragma unroll
  for (int e = 0; e < 3; ++e) out[e * (fragments ? 128 : 4)] = t[e];
}
}  // namespace f32_terms
