// What the scans in chunks of 64 tokens share (delta_chunks.hip, ssd_chunks.hip): how chunks are numbered, and products of
// tiles of 16 x 16 in 32 bits.
#pragma once

#include "device_math.h"
#include "sequence_parts.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int CHUNK = 64, SUB = 16, KT = CHUNK / SUB;  // tokens a chunk and a block of it; blocks a chunk
constexpr int FRAG = 256;                              // floats a tile of 16 x 16

// The chunks of a sequence of n tokens: none for one shorter than `least`, which is walked token by token instead.
__device__ inline int chunks_of(int n, int least) { return parts_of(n, CHUNK, least); }

// the number of sequence b's first chunk
__device__ inline int first_chunk(const int* __restrict__ cu_rows, int b, int least) {
  int n = 0;
  for (int i = threadIdx.x & 63; i < b; i += 64) n += chunks_of(cu_rows[i + 1] - cu_rows[i], least);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, 64);
  return __builtin_amdgcn_readfirstlane(n);
}

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

// The most chunks that `rows` tokens of `batch` sequences can have.
inline long long most_chunks(int rows, int batch, int least) {
  return rows / CHUNK + (long long)(rows / least < batch ? rows / least : batch);
}

// A launch's chunks in rounds of equal numbers, each within the scratch.
inline long long chunks_a_round(long long all, long long scratch_floats, long long a_chunk) {
  const long long fit = scratch_floats / a_chunk, rounds = (all + fit - 1) / fit;
  return (all + rounds - 1) / rounds;
}

// The floats that a launch asks for: its chunks', or as many as `bound` floats hold, or one chunk's.
inline long long chunks_scratch(long long all, long long a_chunk, long long bound) {
  const long long most = bound / a_chunk > 1 ? bound / a_chunk : 1;
  return a_chunk * (all < most ? all : most);
}

}  // namespace
