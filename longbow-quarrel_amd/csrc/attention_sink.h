// What the three files of the windowed attention with a sink share: the arguments of its kernels, how a score is shaped on
// its way to the softmax, and how a 32-bit probability is cut into bfloat16 operands.
#pragma once

#include <cfloat>

#include "common.h"

constexpr float LOG2E = 1.44269504088896340736f;
constexpr float NONE = -3.0e38f;  // the running maximum of a row that has seen no key (finite: no inf - inf)

struct ScoreShape {
  float cap;                       // 0: no cap
  const float *temp, *r1, *r2;     // a number a query head each, or null (r1 and r2 together)
  const float* dist;               // [nh][dist_n], or null
  int dist_n;
};

struct SinkArgs {
  int ldq, ldo, ldg, rows, rows_per_tile, heads_per_tile, nh, nkv, KD, VD;
  const int *row_pos, *row_seq, *seq_slot, *block_table;
  int bt_stride, BS;
  float scale;
  int window, keep_first, sink;
  int maps, out_f32;
  const float* sinks;  // null: the sink's score is 0
  ScoreShape shape;
  const float* wide_gate;
  int ldwg;
  int chunk;  // 0: no chunks
};

// the first key of the window (or of the chunk) of a row at position p
__device__ inline int first_key(const SinkArgs& a, int p) {
  const int lo = (a.window > 0 && p >= a.window) ? p - a.window + 1 : 0;
  return a.chunk > 0 ? max(lo, p / a.chunk * a.chunk) : lo;
}

// Where a query head's softmax starts from its sink: the running maximum in powers of two, finite whatever the sink, and
// the sink's part of the sum.  A sink of -inf, or so low that it is in powers of two, adds nothing; one so high that it is
// infinite in powers of two outweighs every key; NaN and +inf make NaN of the sum.
struct SinkStart {
  float m, l;
};
__device__ inline SinkStart start_at(float sink) {
  const float m = sink * LOG2E;
  return {fminf(fmaxf(m, NONE), FLT_MAX), m < NONE ? 0.f : fmaf(sink, 0.f, 1.f)};
}
__device__ inline SinkStart sink_start(const SinkArgs& a, int h) {
  if (a.sinks == nullptr) return {0.f, 1.f};
  return start_at(a.sinks[h]);
}

// What a lane needs of its query head to shape a score.
struct HeadShape {
  float mul, cap, inv_cap, r1, r2;
  const float* dist;
  int last;
  bool log_bias;
};

__device__ inline HeadShape head_shape(const SinkArgs& a, int h) {
  HeadShape s;
  s.mul = a.shape.temp != nullptr ? a.scale * a.shape.temp[h] : a.scale;
  s.cap = a.shape.cap, s.inv_cap = a.shape.cap > 0.f ? 1.f / a.shape.cap : 0.f;
  s.r1 = a.shape.r1 != nullptr ? a.shape.r1[h] : 0.f, s.r2 = a.shape.r1 != nullptr ? a.shape.r2[h] : 0.f;
  s.log_bias = a.shape.r1 != nullptr;
  s.last = a.shape.dist_n - 1;
  s.dist = a.shape.dist != nullptr ? a.shape.dist + (long long)h * a.shape.dist_n : nullptr;
  return s;
}

// The score of a key `d` positions back (d >= 0).  EXACT: the library's tanh and logarithm (32-bit runs); else the
// hardware's exponential and logarithm, whose absolute error is that of a 32-bit rounding of 1.
template <bool EXACT>
__device__ inline float shaped(float dot, int d, const HeadShape& s) {
  float v = dot * s.mul;
  if (s.cap > 0.f) {
    const float y = v * s.inv_cap;
    if constexpr (EXACT) {
      v = s.cap * tanhf(y);
    } else {
      const float e = __expf(-2.f * fabsf(y));
      v = copysignf(s.cap * (1.f - e) * __builtin_amdgcn_rcpf(1.f + e), y);
    }
  }
  if (s.log_bias) {
    if constexpr (EXACT) v -= s.r1 * log1pf(s.r2 * (float)d);
    else v -= s.r1 * __logf(fmaf(s.r2, (float)d, 1.f));
  }
  if (s.dist != nullptr) v += s.dist[min(d, s.last)];
  return v;
}

template <typename T>
__device__ inline void put_out(T* out, long long at, float v, int out_f32) {
  if (out_f32) ((float*)out)[at] = v;
  else out[at] = from_f32<T>(v);
}

// Eight neighbouring entries of a row of q, which starts on 8 bytes.
__device__ inline uint4 load_q8(const bf16_t* p) {
  const uint2 lo = *(const uint2*)p, hi = *(const uint2*)(p + 4);
  return make_uint4(lo.x, lo.y, hi.x, hi.y);
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ inline bf16x8 as_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

// A 32-bit number as the exact sum of three bfloat16 numbers: its upper half, the upper half of what is below that, and the
// rest.  The upper halves of two words, side by side, are two entries of an operand.
__device__ inline unsigned upper2(float lo, float hi) {
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
__device__ inline float below_upper(float x) { return x - __uint_as_float(__float_as_uint(x) & 0xffff0000u); }

inline bool scores_shaped(const ScoreShape& s) {
  return s.cap > 0.f || s.temp != nullptr || s.r1 != nullptr || s.dist != nullptr;
}

// Prompts of a bfloat16 run (attention_sink_rows.hip).  -> 1 launched, 0 not a launch that it takes, -2 an error.
int lq_sink_rows32(const bf16_t* q, void* out, const bf16_t* gate, const bf16_t* kcache, const bf16_t* vcache,
                   const int* cu_rows, const SinkArgs& a, int batch, hipStream_t stream);

// Single tokens of a bfloat16 run (attention_sink_decode.hip); the same answers.
int lq_sink_decode(const bf16_t* q, void* out, const bf16_t* gate, const bf16_t* kcache, const bf16_t* vcache,
                   const SinkArgs& a, int max_len, float* part, long long part_floats, int* tickets, long long tickets_n,
                   hipStream_t stream);
long long lq_sink_decode_workspace(int rows, int nh, int nkv, int KD, int VD, int block_size, int window, int keep_first,
                                   int chunk, int max_len);
