// What the matrix-core attention of prompts (attention_mfma.hip) and of single tokens (attention_decode.hip) share.
#pragma once

#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

namespace {

constexpr int BS = 64;      // positions per cache block (the only block size that these files take)

__device__ inline bf16x8 as_bf16x8(u32x4 v) {
  union {
    u32x4 u;
    bf16x8 b;
  } c;
  c.u = v;
  return c.b;
}

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// two floats to packed bfloat16, round to nearest even (v_cvt_pk_bf16_f32)
__device__ inline unsigned pack_bf16(float lo, float hi) {
  union {
    bf16x2 b;
    unsigned u;
  } c;
  c.b = __builtin_convertvector((f32x2){lo, hi}, bf16x2);
  return c.u;
}

// Reductions over the four 16-lane rows of a wave (the lanes that share lane % 16) with the row-swap
// instructions of gfx950, which stay in the vector unit (a shuffle goes through LDS and back).
// v_permlane16_swap exchanges the odd rows of its first operand with the even rows of its second;
// with the same value in both, every lane then holds its own and its xor-16 partner's value, the
// lower row's first.  v_permlane32_swap does the same with the wave's halves.
__device__ inline float rows_max(float x) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ inline float rows_sum(float x) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// 2^x for x <= 0 (v_exp_f32; results below the normal range flush to zero, which is what a
// probability that small is worth)
__device__ inline float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// The running maximum that the probabilities are taken against follows the scores' maximum lazily: it moves
// (and what has been summed is rescaled) only when some row of the wave meets a score more than this far
// above it, in the log2 domain.  Probabilities then reach 2^8 at most, which float32 sums and bfloat16
// operands (eight bits of exponent) hold as well as values below 1; the quotient at the end is the same.
// After a row's first keys the branch is taken rarely; with a slack of zero it ran whenever any row's maximum
// moved at all, and its multiplications of every accumulator cost 5 to 8 % of a long prompt's time.
constexpr float RESCALE_SLACK = 8.0f;

}  // namespace
