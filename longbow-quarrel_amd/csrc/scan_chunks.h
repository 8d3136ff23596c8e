// What the scans in chunks of 64 tokens share (delta_chunks.hip, ssd_chunks.hip): products of tiles of 16 x 16 in 32 bits.
#pragma once

#include "device_math.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

// c + A . B by v_mfma_f32_16x16x4_f32: lane l gives A[l % 16][4 (l / 16) .. + 3] and B[4 (l / 16) .. + 3][l % 16] and
// receives D[4 (l / 16) + e][l % 16].
__device__ inline f32x4 step4(const f32x4& a, const f32x4& b, f32x4 c) {
#pragma unroll
  for (int s = 0; s < 4; ++s) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b[s], c, 0, 0, 0);
  return c;
}

// c + A . B for an A that has zeros above its diagonal, where B's rows are tokens: what is no finite number in a token's
// row must not pass a zero to an earlier one's (0 x NaN, 0 x inf).  Such entries stay out of the matrix product, and
// are multiplied for the rows at and below them only; the bits of the others are those of the matrix product.
__device__ inline f32x4 step4_lower(const f32x4& a, const f32x4& b, f32x4 c) {
  f32x4 finite;
#pragma unroll
  for (int s = 0; s < 4; ++s) finite[s] = b[s] * 0.f == 0.f ? b[s] : 0.f;
  c = step4(a, finite, c);
  const int col = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
#pragma unroll 1  // (rarely run: as few registers as can be)
  for (int kg = 0; kg < 4; ++kg)
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float bk = __shfl(b[s], kg * 16 + col, 64);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float ak = __shfl(a[s], kg * 16 + 4 * g + e, 64);
        if (4 * kg + s <= 4 * g + e && bk * 0.f != 0.f) c[e] = fmaf(ak, bk, c[e]);
      }
    }
  return c;
}

// NaN once a tile has had an entry that is no finite number (from 0 on).
__device__ inline float not_finite(const f32x4& b, float so_far) {
  return fmaf(b[0], 0.f, fmaf(b[1], 0.f, fmaf(b[2], 0.f, fmaf(b[3], 0.f, so_far))));
}

}  // namespace
