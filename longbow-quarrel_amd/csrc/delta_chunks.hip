// The gated delta rule over long portions of a sequence, in chunks of 64 tokens on the matrix cores.
//
// Token by token (recurrent.hip):  S <- diag(g_t) S;  u_t = beta_t (v_t - S^T k_t);  S <- S + k_t u_t^T;  o_t = S^T q_t,
// a chain of two exchanges over a column's lanes a token, 0.31 to 0.42 microseconds of it and 1.2 where the chip is
// full.  Over a chunk that starts from the state S, with p_t the product of the decays g_1 .. g_t of a key channel and
// f_st that of g_(s+1) .. g_t (all of them products of numbers up to 1, never quotients):
//   A[t][s] = sum_n k_t k_s f_st (s < t),  B[t][s] = sum_n q_t k_s f_st (s <= t)
//   U = T (V - K~ S),  T = (I + diag(beta) A)^-1 diag(beta),  K~_t = p_t k_t
//   O = Q~ S + B U,  Q~_t = p_t q_t;      S <- diag(p_64) S + sum_s (f_s,64 k_s) u_s^T
// T, B, K~, Q~ and the last factor do not depend on the state: a first launch makes them for all chunks and heads side by
// side (`delta_prepare_kernel`), in the order in which the second reads its operands.  The second (`delta_walk_kernel`)
// walks a sequence's chunks in order, a workgroup a head and 16 columns of the values.
//
// Everything is 32-bit (v_mfma_f32_16x16x4_f32: lane l gives A[l % 16][k = l / 16] and B[k = l / 16][l % 16] and
// receives D[4 (l / 16) + e][l % 16]).  Which entry stands for which k is free as long as both operands agree: step s of
// a run of 16 k takes k = 4 (l / 16) + s, so that a result's four registers are the next product's B operands as they
// are, and an A operand is four neighbouring entries of a row.  "Fragments" below: 16 rows by 16 k, lane l's four
// entries (row l % 16, k = 4 (l / 16) .. + 3) at 4 l.
//
// Chunks count from a sequence's first row of the step; a last chunk's missing tokens take part as zeros.
#include <cmath>
#include <type_traits>

#include "scan_chunks.h"

namespace {

constexpr int NMAX = 128, NT = NMAX / 16;  // key channels (fewer: zeros)
// a (chunk, head)'s part of the scratch, in floats
constexpr int AT_KEYS = 0, AT_QUERIES = AT_KEYS + KT * NT * FRAG, AT_UPDATE = AT_QUERIES + KT * NT * FRAG,
              AT_T = AT_UPDATE + NT * KT * FRAG, AT_B = AT_T + KT * KT * FRAG, AT_DECAY = AT_B + KT * KT * FRAG,
              PART = AT_DECAY + NMAX;

struct DeltaArgs {
  const float *q, *k, *v, *beta, *a, *dt_bias, *a_log;
  int ldq, ldk, ldv, ldbeta, lda, ldo;
  float *state, *out, *scratch;
  int heads, kv_heads, N, P, batch, channel_decay;
  const int *seq_slot, *cu_rows;
  int least;        // sequences of fewer tokens are not taken
  int first, last;  // the chunks of this pair of launches: numbers first .. last - 1, the scratch of `first` at its start
  float q_scale, inv_tau;  // of gated linear attention
};

template <int CTRL>
__device__ inline float add_from(float keep, float give) {  // the partner's `give` on top of this lane's `keep`
  return keep + dpp_swap<CTRL>(give);
}

// The sums over a wavefront of up to COUNT (8 or 16) values: lane s (modulo 16) ends up with that of v[s] (modulo COUNT).
// Every exchange halves the values a lane still carries: its partner takes the other half.
template <int COUNT>
__device__ inline float sums_by_lane(float (&v)[SUB]) {
  const int lane = threadIdx.x;
  if constexpr (COUNT == 16) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = add_from<0x140>(lane & 8 ? v[i + 8] : v[i], lane & 8 ? v[i] : v[i + 8]);  // 15 - lane
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = add_from<0x140>(v[i], v[i]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = add_from<0x141>(lane & 4 ? v[i + 4] : v[i], lane & 4 ? v[i] : v[i + 4]);  // 7 - lane
#pragma unroll
  for (int i = 0; i < 2; ++i) v[i] = add_from<0x4E>(lane & 2 ? v[i + 2] : v[i], lane & 2 ? v[i] : v[i + 2]);
  float x = add_from<0xB1>(lane & 1 ? v[1] : v[0], lane & 1 ? v[0] : v[1]);
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}

// exp(rate ln(1 + e^z)).  ln(1 + x) of x = e^-|z| <= 1 as 2 atanh(x / (2 + x)), whose series in s^2 <= 1 / 9 ends below
// 2^-25 of it with s^15: a third of the library function's instructions, which were 4 microseconds of a chunk's 26.
__device__ inline float decay_of(float z, float rate) {
  const float x = expf(-fabsf(z)), d = 2.f + x;
  float r = __builtin_amdgcn_rcpf(d);
  r = fmaf(fmaf(-d, r, 1.f), r, r);
  const float s = x * r, y = s * s;
  float p = 2.f / 15.f;
  p = fmaf(p, y, 2.f / 13.f), p = fmaf(p, y, 2.f / 11.f), p = fmaf(p, y, 2.f / 9.f), p = fmaf(p, y, 2.f / 7.f);
  p = fmaf(p, y, 2.f / 5.f), p = fmaf(p, y, 2.f / 3.f);
  return expf(rate * (fmaxf(z, 0.f) + fmaf(s * y, p, 2.f * s)));
}

constexpr int LD = NMAX + 4;   // floats a row of LDS: neighbouring rows start 4 banks apart
constexpr int LDT = CHUNK + 4;

struct Prepared {
  float k[CHUNK][LD], q[CHUNK][LD], g[CHUNK][LD];  // after the blocks: k and q by the decays from their block's start, k by those to its end
  float block[KT][NMAX];                           // the product of a block's decays
  float m[CHUNK][LDT];                             // A, then T
  float b[CHUNK][LDT];
  float inv[KT][SUB][SUB + 4];                     // the inverses of the blocks on the diagonal
  float beta[CHUNK];
};

// One workgroup of eight wavefronts a (chunk, head).  Wavefronts w and w + 4 first make A and B within block w, channel
// by channel (a lane holds two, and for every earlier token of the block the product of the decays since): no
// factoring of f_st into a row's and a column's part is safe where decays are strong.  Between blocks it is: from the
// row's block's start on, and up to the column's block's end.
// ERASE: the delta rule.  Without it (gated linear attention) U is V: only B, Q~, the update's factor and the decays are made, and a
// channel's decay is sigmoid(z + bias)^inv_tau.
// (What the state is multiplied with from chunk to chunk is there the exponential of a sum of logarithms, rounded once where a
// product of 64 decays is rounded at each: these errors are what adds up along a sequence.)
__device__ inline float log_decay(float z, float inv_tau) { return -softplus_f(-z) * inv_tau; }

template <bool QUADS, bool ERASE>
__global__ __launch_bounds__(512, 2) void delta_prepare_kernel(DeltaArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  Prepared& L = *(Prepared*)smem;
  const Part at = find_part(a.cu_rows, a.batch, CHUNK, a.least, a.first + blockIdx.x);
  if (at.seq < 0) return;
  const int h = blockIdx.y, j = h / (a.heads / a.kv_heads), tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const long long r0 = at.first;
  const int nt = at.rows, N = a.N;
  float* to = a.scratch + ((long long)blockIdx.x * a.heads + h) * PART;
  const float rate = ERASE ? -expf(a.a_log[h]) : 0.f;

  // every load of a thread is asked for before the first is waited for
  if constexpr (QUADS) {
    constexpr int PER = CHUNK * NMAX / 4 / 512;
    f32x4 k[PER], q[PER], z[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = tid + 512 * i, t = e / (NMAX / 4), n = e % (NMAX / 4) * 4;
      k[i] = q[i] = z[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
      if (t < nt && n < N) {
        const long long r = r0 + t;
        k[i] = *(const f32x4*)(a.k + r * a.ldk + j * N + n), q[i] = *(const f32x4*)(a.q + r * a.ldq + j * N + n);
        if constexpr (!ERASE) q[i] *= a.q_scale;
        if (a.channel_decay) z[i] = *(const f32x4*)(a.a + r * a.lda + h * N + n) + *(const f32x4*)(a.dt_bias + h * N + n);
      }
    }
    f32x4 logs = {0.f, 0.f, 0.f, 0.f};  // (a thread's channels are the same in every turn)
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = tid + 512 * i, t = e / (NMAX / 4), n = e % (NMAX / 4) * 4;
      *(f32x4*)&L.k[t][n] = k[i], *(f32x4*)&L.q[t][n] = q[i];
      if (a.channel_decay) {
        f32x4 g = {1.f, 1.f, 1.f, 1.f};
        if (t < nt && n < N)
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            if constexpr (ERASE) {
              g[x] = decay_of(z[i][x], rate);
            } else {
              const float log = log_decay(z[i][x], a.inv_tau);
              logs[x] += log, g[x] = expf(log);
            }
          }
        *(f32x4*)&L.g[t][n] = g;
      }
    }
    if constexpr (!ERASE) *(f32x4*)(&L.m[0][0] + (tid / (NMAX / 4)) * NMAX + tid % (NMAX / 4) * 4) = logs;
  } else {
    float logs = 0.f;
    for (int e = tid; e < CHUNK * NMAX; e += 512) {
      const int t = e / NMAX, n = e % NMAX;
      const bool there = t < nt && n < N;
      const long long r = r0 + t;
      L.k[t][n] = there ? a.k[r * a.ldk + j * N + n] : 0.f;
      L.q[t][n] = there ? a.q[r * a.ldq + j * N + n] * (ERASE ? 1.f : a.q_scale) : 0.f;
      if (a.channel_decay) {
        const float z = there ? a.a[r * a.lda + h * N + n] + a.dt_bias[h * N + n] : 0.f;
        if constexpr (ERASE) {
          L.g[t][n] = there ? decay_of(z, rate) : 1.f;
        } else {
          const float log = there ? log_decay(z, a.inv_tau) : 0.f;
          logs += log, L.g[t][n] = expf(log);
        }
      }
    }
    if constexpr (!ERASE) (&L.m[0][0])[tid] = logs;
  }
  if (ERASE && !a.channel_decay) {  // one decay a head: a thread makes that of its row
    const int t = tid >> 3;
    const float g = t < nt ? decay_of(a.a[(r0 + t) * a.lda + h] + a.dt_bias[h], rate) : 1.f;
    for (int n = tid & 7; n < NMAX; n += 8) L.g[t][n] = g;
  }
  if (ERASE && tid < CHUNK) L.beta[tid] = tid < nt ? sigmoid_f(a.beta[(r0 + tid) * a.ldbeta + h]) : 0.f;
  for (int e = tid; e < CHUNK * LDT; e += 512) {
    if constexpr (ERASE) (&L.m[0][0])[e] = 0.f;  // (else it holds the threads' sums of logarithms)
    (&L.b[0][0])[e] = 0.f;
  }
  __syncthreads();

  {  // within a block of 16 tokens
    const int blk = w & 3;
    const bool of_b = w >= KT;
    float faded[SUB][2], from_start[SUB][2], run[2] = {1.f, 1.f};  // faded: a token's k by the decays since
    auto row_of = [&](auto full, int t) {
      constexpr int COUNT = decltype(full)::value;
      const int row = SUB * blk + t;
      float with[2], sums[SUB];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int n = lane + 64 * c;
        const float g = L.g[row][n];
#pragma unroll
        for (int s = 0; s < COUNT; ++s)
          if (s < t) faded[s][c] *= g;
        faded[t][c] = L.k[row][n];
        with[c] = of_b ? L.q[row][n] : faded[t][c];
        run[c] *= g;
        from_start[t][c] = with[c] * run[c];
      }
      if (!ERASE && !of_b) return;  // (no A)
#pragma unroll
      for (int s = 0; s < COUNT; ++s) sums[s] = s <= t ? fmaf(faded[s][1], with[1], faded[s][0] * with[0]) : 0.f;
      const float sum = sums_by_lane<COUNT>(sums);
      // (stored here: else the rows' loads and sums run into one another and out of registers)
      if (lane < (of_b ? t + 1 : t)) (of_b ? L.b : L.m)[row][SUB * blk + lane] = sum;
      asm volatile("" ::: "memory");
    };
#pragma unroll
    for (int t = 0; t < 8; ++t) row_of(std::integral_constant<int, 8>{}, t);
#pragma unroll
    for (int t = 8; t < SUB; ++t) row_of(std::integral_constant<int, 16>{}, t);
    __syncthreads();  // (the plain rows have been read)
#pragma unroll
    for (int t = 0; t < SUB; ++t)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int row = SUB * blk + t, n = lane + 64 * c;
        (of_b ? L.q : L.k)[row][n] = from_start[t][c];
        if (!of_b) L.g[row][n] = faded[t][c];
      }
    if (!of_b) L.block[blk][lane] = run[0], L.block[blk][lane + 64] = run[1];
  }
  __syncthreads();

  // K~ and Q~ as fragments, rows tokens
#pragma unroll
  for (int e = tid; e < KT * NT * 64; e += 512) {
    const int mt = e / (NT * 64), row = SUB * mt + (e & 15), n = e / 64 % NT * 16 + (e >> 4 & 3) * 4;
    f32x4 f = {1.f, 1.f, 1.f, 1.f};
#pragma unroll
    for (int i = 0; i < KT - 1; ++i)
      if (i < mt) f *= *(const f32x4*)&L.block[i][n];
    if constexpr (ERASE) *(f32x4*)(to + AT_KEYS + e * 4) = *(const f32x4*)&L.k[row][n] * f;
    *(f32x4*)(to + AT_QUERIES + e * 4) = *(const f32x4*)&L.q[row][n] * f;
  }
  // what the state is updated with, rows key channels
#pragma unroll
  for (int e = tid; e < NT * KT * 64; e += 512) {
    const int kb = e / 64 % KT, n = e / (KT * 64) * 16 + (e & 15), t = SUB * kb + (e >> 4 & 3) * 4;
    float f = 1.f;
#pragma unroll
    for (int i = 1; i < KT; ++i)
      if (i > kb) f *= L.block[i][n];
    *(f32x4*)(to + AT_UPDATE + e * 4) = (f32x4){L.g[t][n] * f, L.g[t + 1][n] * f, L.g[t + 2][n] * f, L.g[t + 3][n] * f};
  }
  if (tid < NMAX) {
    float f = 1.f;
    if constexpr (ERASE) {
      for (int i = 0; i < KT; ++i) f *= L.block[i][tid];
    } else {
      f = 0.f;
      for (int i = 0; i < (QUADS ? 512 / (NMAX / 4) : 512 / NMAX); ++i) f += (&L.m[0][0])[i * NMAX + tid];
      f = expf(f);
    }
    to[AT_DECAY + tid] = f;
  }
  // between blocks: six pairs of A and of B
  const int c = lane & 15, g = lane >> 4;
  for (int u = ERASE ? w : 2 * w + 1; u < 12; u += ERASE ? 8 : 16) {
    const int pair = u >> 1, i = pair < 1 ? 1 : pair < 3 ? 2 : 3, jb = pair - i * (i - 1) / 2;
    const float(*rows)[LD] = (u & 1) ? L.q : L.k;
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int nb = 0; nb < NT; ++nb) {
      const int n = 16 * nb + 4 * g;
      f32x4 col = *(const f32x4*)&L.g[SUB * jb + c][n];
      for (int x = jb + 1; x < i; ++x) col *= *(const f32x4*)&L.block[x][n];
      acc[nb & 1] = step4(*(const f32x4*)&rows[SUB * i + c][n], col, acc[nb & 1]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) ((u & 1) ? L.b : L.m)[SUB * i + 4 * g + e][SUB * jb + c] = acc[0][e] + acc[1][e];
  }
  if constexpr (!ERASE) {
    __syncthreads();
    for (int e = tid; e < KT * KT * 64; e += 512)
      *(f32x4*)(to + AT_B + e * 4) = *(const f32x4*)&L.b[SUB * (e / (KT * 64)) + (e & 15)][e / 64 % KT * SUB + (e >> 4 & 3) * 4];
    return;
  }
  // the inverse of I + diag(beta) A: the blocks on the diagonal by substitution, a lane a column
  if (w < KT && lane < SUB) {
    float x[SUB];
#pragma unroll
    for (int t = 0; t < SUB; ++t) {
      float sum = 0.f;
#pragma unroll
      for (int s = 0; s < t; ++s) sum = fmaf(L.m[SUB * w + t][SUB * w + s], x[s], sum);
      x[t] = (t == lane ? 1.f : 0.f) - L.beta[SUB * w + t] * sum;
      L.inv[w][t][lane] = x[t];
    }
  }
  __syncthreads();
  // ... and wavefront w the column of blocks w: X_ww is that inverse, X_iw = -X_ii sum_m (beta A)_im X_mw
  f32x4 X[KT];
#pragma unroll
  for (int i = 0; i < KT; ++i) X[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < KT; ++i) {
    if (w < KT && i == w) {
#pragma unroll
      for (int e = 0; e < 4; ++e) X[i][e] = L.inv[i][4 * g + e][c];
    } else if (i > w) {
      f32x4 Z = {0.f, 0.f, 0.f, 0.f};
      const float bi = L.beta[SUB * i + c];
#pragma unroll
      for (int x = 0; x < i; ++x)
        if (x >= w) Z = step4(*(const f32x4*)&L.m[SUB * i + c][SUB * x + 4 * g] * bi, X[x], Z);
      {
        const float odd = not_finite(Z, 0.f);
        const f32x4 inv = *(const f32x4*)&L.inv[i][c][4 * g] * -1.f;
        X[i] = __any(odd != odd) ? step4_lower(inv, Z, X[i]) : step4(inv, Z, X[i]);
      }
    }
  }
  __syncthreads();  // (A has been read)
  if (w < KT) {
#pragma unroll
    for (int i = 0; i < KT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {  // (a token's beta multiplies none of the zeros above the diagonal: it may be NaN)
        const int row = SUB * i + 4 * g + e, col = SUB * w + c;
        L.m[row][col] = row >= col ? X[i][e] * L.beta[col] : 0.f;
      }
  }
  __syncthreads();
  for (int e = tid; e < KT * KT * 64; e += 512) {
    const int row = SUB * (e / (KT * 64)) + (e & 15), s = e / 64 % KT * SUB + (e >> 4 & 3) * 4;
    *(f32x4*)(to + AT_T + e * 4) = *(const f32x4*)&L.m[row][s];
    *(f32x4*)(to + AT_B + e * 4) = *(const f32x4*)&L.b[row][s];
  }
}

__device__ inline void lds_barrier() {  // this wavefront's LDS accesses are done, its loads from memory need not be
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// What a workgroup walks: sequences from the longest on, in one 16 columns of the values after the other, in these the heads (so
// that with heads in eights a head's workgroups are on one die, whose cache its operands then pass once).  In the order of
// the sequences, the heads before the columns, three prompts of 257, 878 and 1 500 tokens and 16 heads took 133 microseconds, two of
// the longest walks or more to a compute unit; in this order 92.
struct Walk {
  int b, h, p0;
};
__device__ inline Walk walk_of(const DeltaArgs& a) {
  const int columns = (a.P + 15) / 16, a_sequence = a.heads * columns, rank = blockIdx.x / a_sequence, in = blockIdx.x % a_sequence;
  return {sequence_by_length(a.cu_rows, a.batch, rank), in % a.heads, in / a.heads * 16};
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, bytes, 0x00020000);
}
// 16 bytes a lane of the tile `tile` (a constant) behind `at` floats of a part of the scratch
__device__ __forceinline__ f32x4 load_frag(__amdgpu_buffer_rsrc_t from, int lane16, int at, int tile) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(from, lane16 + tile % 4 * FRAG * 4, (at + tile / 4 * 4 * FRAG) * 4, 0));
}

__device__ __forceinline__ f32x4& lane_of(f32x4 (&tile)[64], int lane16) { return *(f32x4*)((char*)tile + lane16); }

template <bool CAREFUL>
__device__ __forceinline__ f32x4 step4_diagonal(const f32x4& a, const f32x4& b, f32x4 c) {
  if constexpr (CAREFUL) return step4_lower(a, b, c);
  else return step4(a, b, c);
}

// One workgroup of eight wavefronts a (sequence, head, 16 columns of the values); wavefront w holds channels 16 w .. + 15
// of the state.  A chunk: wavefronts 0 to 3 make 16 tokens of V - K~ S each and 4 to 7 of Q~ S; then 0 to 3 of U, while
// 4 to 7 add B U of the chunk before to its results; then all update the state.  Tiles cross between wavefronts through
// LDS in lane order.
// What bounds a chunk is this chain: matrix instructions keep a SIMD for 1.5 us of its 2.55, the rest are the three crossings.
// So the loads of the next chunk's operands go out between the products that free their registers, in the shadow of
// the matrix instructions; B U, which no later chunk needs, waits until the wavefronts that make it would be idle; and the two
// wavefronts of a SIMD share the triangles' tiles evenly.  (With the loads and B U each in a place of its own a chunk took 3.4 us.
// A launch of 2 100 tokens, 128 workgroups, 113 us before and 85 now; 1 024 workgroups 159 and 124.  In half the
// registers, two workgroups a compute unit, the latter took 118, but 384 workgroups, of which the longest 256
// had a compute unit each, 87 instead of 71.)
__global__ __launch_bounds__(512, 2) void delta_walk_kernel(DeltaArgs a) {
  __shared__ f32x4 Ss[NT][64], Ws[KT][64], Us[2][KT][64];
  __shared__ int again;
  const Walk at = walk_of(a);
  const int b = at.b, h = at.h, tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4, p = at.p0 + c;
  const bool second = w >= KT;  // Q~, B and the results
  const int mt = second ? NT - 1 - w : w;  // (the two wavefronts of a SIMD have five tiles of T and B together)
  const long long r1 = a.cu_rows[b + 1];
  const int base = first_chunk(a.cu_rows, b, a.least), i0 = max(a.first - base, 0);
  const int chunks = min(chunks_of((int)(r1 - a.cu_rows[b]), a.least), a.last - base) - i0;  // from the sequence's i0th on
  if (chunks <= 0) return;
  const long long r0 = a.cu_rows[b] + (long long)i0 * CHUNK;
  const float* part = a.scratch + ((long long)(base + i0 - a.first) * a.heads + h) * PART;
  const long long step = (long long)a.heads * PART;
  const bool live = p < a.P;
  int lane16 = lane * 16;
  const int row0 = SUB * mt + 4 * g, none = 0x7fffffff;  // (no buffer's offset: such a lane reads 0 and writes nothing)
  const __amdgpu_buffer_rsrc_t state = buffer_of(a.state + ((long long)a.seq_slot[b] * a.heads + h) * a.P * a.N, a.P * a.N * 4);
  const int n0 = 16 * w + 4 * g, at_state = live ? (p * a.N + n0) * 4 : none;
  const int at_v = live ? (row0 * a.ldv + p) * 4 : none, at_out = live ? (row0 * a.ldo + p) * 4 : none;
  f32x4 S, rows[NT], tri[KT - 1], diag, upd[KT], decay, Y = {0.f, 0.f, 0.f, 0.f};
  f32x4 V = {0.f, 0.f, 0.f, 0.f};
  // Every wavefront asks for as many tiles, whatever it needs and whether there is another chunk (a buffer of no bytes gives zeros and
  // moves nothing): the compiler then knows how many loads are behind the one it waits for.
  auto ask_rows = [&](int nb, int i) {
    rows[nb] = load_frag(buffer_of(part + i * step, i < chunks ? PART * 4 : 0), lane16,
                            (second ? AT_QUERIES : AT_KEYS) + mt * NT * FRAG, nb);
  };
  auto ask_tri = [&](int i) {
    const int at_tri = (second ? AT_B : AT_T) + mt * KT * FRAG, bytes = i < chunks ? PART * 4 : 0;
#pragma unroll
    for (int kb = 0; kb < KT - 1; ++kb) tri[kb] = load_frag(buffer_of(part + i * step, kb < mt ? bytes : 0), lane16, at_tri, kb);
    diag = load_frag(buffer_of(part + i * step, bytes), lane16, at_tri + mt * FRAG, 0);
  };
  auto ask_upd = [&](int kb, int i) {
    upd[kb] = load_frag(buffer_of(part + i * step, i < chunks ? PART * 4 : 0), lane16, AT_UPDATE + w * KT * FRAG, kb);
  };
  auto ask_decay = [&](int i) {
    const int bytes = i < chunks ? PART * 4 : 0;
    decay = load_frag(buffer_of(part + i * step, bytes), 16 * g, AT_DECAY + 16 * w, 0);
  };
  // (a matrix's rows of a chunk, from its first row's first column of the head on)
  auto ask_v = [&](int i) {
    const long long c0 = r0 + (long long)i * CHUNK;
    const int n = second || i >= chunks ? 0 : (int)min((long long)CHUNK, r1 - c0);
    const __amdgpu_buffer_rsrc_t from = buffer_of(a.v + c0 * a.ldv + (long long)h * a.P, second || i >= chunks ? 0 : (CHUNK * a.ldv + a.P) * 4);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      V[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(from, row0 < n - e ? at_v : none, e * a.ldv * 4, 0));
  };
  // The triangular products' zeros are no matter until a token brings a NaN or an infinity (U has one): then
  // all is walked again, and none of them reaches an earlier token.  (A test of every chunk's operands ahead of those
  // products lay in the chain and took 0.5 of its 3.3 microseconds; this takes 171 for 168.6 microseconds of a whole launch
  // of 2 048 tokens.)
  if (tid == 0) again = 0;  // (barriers follow)
  auto walk = [&](auto with_care) {
    constexpr bool careful = decltype(with_care)::value;
    float odd = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) S[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(state, n0 < a.N - e ? at_state : none, 4 * e, 0));
    lane_of(Ss[w], lane16) = S;
#pragma unroll
    for (int nb = 0; nb < NT; ++nb) ask_rows(nb, 0);
    __builtin_amdgcn_sched_barrier(0);  // (the loop's first wait is for these: nothing that it need not wait for goes ahead of them)
    ask_tri(0), ask_v(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kb = 0; kb < KT; ++kb) ask_upd(kb, 0);
    ask_decay(0);
    lds_barrier();
    auto finish = [&](int i) {  // B U on top of chunk i's results
      f32x4 all[KT], own = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < KT - 1; ++kb) all[kb] = lane_of(Us[i & 1][kb], lane16);
      all[KT - 1] = lane_of(Us[i & 1][mt], lane16);
#pragma unroll
      for (int kb = 0; kb < KT - 1; ++kb)
        if (kb < mt) own = step4(tri[kb], all[kb], own);
      own = step4_diagonal<careful>(diag, all[KT - 1], own);
      const f32x4 whole = Y + own;
      const long long c0 = r0 + (long long)i * CHUNK;
      const int n = i < 0 ? 0 : (int)min((long long)CHUNK, r1 - c0);
      const __amdgpu_buffer_rsrc_t to = buffer_of(a.out + c0 * a.ldo + (long long)h * a.P, i < 0 ? 0 : (CHUNK * a.ldo + a.P) * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(whole[e]), to, row0 < n - e ? at_out : none, e * a.ldo * 4, 0);
    };
#pragma unroll 1
    for (int i = 0; i < chunks; ++i) {
      const int u = i & 1;
      asm volatile("" : "+v"(lane16));  // (or the loads' offsets, lane16 and a constant each, stay in registers of their own)
      f32x4 acc[4];  // (four chains of products: their roundings are smaller, and none waits for the one before it)
#pragma unroll
      for (int x = 0; x < 4; ++x) acc[x] = (f32x4){0.f, 0.f, 0.f, 0.f};
      f32x4 from[NT];
#pragma unroll
      for (int nb = 0; nb < NT; ++nb) from[nb] = lane_of(Ss[nb], lane16);
#pragma unroll
      for (int nb = 0; nb < NT; ++nb) {
        acc[nb & 3] = step4(rows[nb], from[nb], acc[nb & 3]);
        ask_rows(nb, i + 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      const f32x4 next = (acc[0] + acc[1]) + (acc[2] + acc[3]);
      if (!second) {
        lane_of(Ws[mt], lane16) = V - next;
      }
      lds_barrier();
      if (!second) {
        f32x4 all[KT], U = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < KT - 1; ++kb) all[kb] = lane_of(Ws[kb], lane16);
        all[KT - 1] = lane_of(Ws[mt], lane16);
#pragma unroll
        for (int kb = 0; kb < KT - 1; ++kb)
          if (kb < mt) U = step4(tri[kb], all[kb], U);
        U = step4_diagonal<careful>(diag, all[KT - 1], U);
        lane_of(Us[u][mt], lane16) = U;
        odd = not_finite(U, odd);  // (a token's V - K~ S that is not finite leaves its U so too, whatever stands on T's diagonal)
      } else {
        finish(i - 1);
        Y = next;
      }
      ask_tri(second ? i : i + 1), ask_v(i + 1);
      lds_barrier();
      // (what the chunk adds is summed by itself: one rounding at the state's size a chunk, not one a product)
      f32x4 add[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int kb = 0; kb < KT; ++kb) {
        add[kb & 1] = step4(upd[kb], lane_of(Us[u][kb], lane16), add[kb & 1]);
        ask_upd(kb, i + 1);
      }
      S = S * decay + (add[0] + add[1]);
      ask_decay(i + 1);
      lane_of(Ss[w], lane16) = S;
      lds_barrier();
    }
    if (second) finish(chunks - 1);
    return odd;
  };
  const float odd = walk(std::false_type{});
  if (odd != odd) again = 1;
  lds_barrier();  // (no wait for the results' stores)
  if (__builtin_amdgcn_readfirstlane(again)) walk(std::true_type{});
#pragma unroll
  for (int e = 0; e < 4; ++e) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(S[e]), state, n0 < a.N - e ? at_state : none, 4 * e, 0);
}

// The walk of gated linear attention, U = V:  O = Q~ S + B V;  S <- diag(p_64) S + sum_s (f_s,64 k_s) v_s^T.  One workgroup of eight
// wavefronts a (sequence, head, 16 columns of the values).  Wavefront w holds channels 16 w .. + 15 of the state; for the results
// it takes 16 tokens (w % 4) and half of the sums (w / 4: channels and blocks of tokens).  The state and the values stand in LDS
// twice, so that a chunk has one barrier.
__global__ __launch_bounds__(512, 2) void gla_walk_kernel(DeltaArgs a) {
  __shared__ f32x4 Ss[2][NT][64], Vs[2][KT][64], Ps[2][KT][64];
  const Walk at = walk_of(a);
  const int b = at.b, h = at.h, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int c = lane & 15, g = lane >> 4, p = at.p0 + c, mt = w & 3, half = w >> 2;
  const long long r1 = a.cu_rows[b + 1];
  const int base = first_chunk(a.cu_rows, b, a.least), i0 = max(a.first - base, 0);
  const int chunks = min(chunks_of((int)(r1 - a.cu_rows[b]), a.least), a.last - base) - i0;  // from the sequence's i0th on
  if (chunks <= 0) return;
  const long long r0 = a.cu_rows[b] + (long long)i0 * CHUNK;
  const float* from = a.scratch + ((long long)(base + i0 - a.first) * a.heads + h) * PART;
  const long long step = (long long)a.heads * PART;
  float* sp = a.state + (((long long)a.seq_slot[b] * a.heads + h) * a.P + min(p, a.P - 1)) * a.N;
  const bool live = p < a.P;
  f32x4 S, rows[NT / 2], tri[2], upd[KT], V = {0.f, 0.f, 0.f, 0.f}, decay;
  auto ask = [&](const float* f) {
#pragma unroll
    for (int nb = 0; nb < NT / 2; ++nb) rows[nb] = *(const f32x4*)(f + AT_QUERIES + ((mt * NT + half * (NT / 2) + nb) * 64 + lane) * 4);
#pragma unroll
    for (int x = 0; x < 2; ++x)
      if (2 * half + x <= mt) tri[x] = *(const f32x4*)(f + AT_B + ((mt * KT + 2 * half + x) * 64 + lane) * 4);
#pragma unroll
    for (int kb = 0; kb < KT; ++kb) upd[kb] = *(const f32x4*)(f + AT_UPDATE + ((w * KT + kb) * 64 + lane) * 4);
    decay = *(const f32x4*)(f + AT_DECAY + 16 * w + 4 * g);
  };
  auto ask_v = [&](long long c0) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const long long r = c0 + SUB * mt + 4 * g + e;
      V[e] = live && r < r1 ? a.v[r * a.ldv + (long long)h * a.P + p] : 0.f;
    }
  };
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int n = 16 * w + 4 * g + e;
    S[e] = live && n < a.N ? sp[n] : 0.f;
  }
  ask(from);
  if (half == 0) ask_v(r0);
  Ss[0][w][lane] = S;
  if (half == 0) {
    Vs[0][mt][lane] = V;
    if (chunks > 1) ask_v(r0 + CHUNK);
  }
  lds_barrier();
  for (int i = 0; i < chunks; ++i, from += step) {
    const int cur = i & 1;
    const long long c0 = r0 + (long long)i * CHUNK;
    f32x4 acc[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) acc[x] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int nb = 0; nb < NT / 2; ++nb) acc[nb & 1] = step4(rows[nb], Ss[cur][half * (NT / 2) + nb][lane], acc[nb & 1]);
    f32x4 own = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const int kb = 2 * half + x;
      if (kb > mt) continue;
      const f32x4 v = Vs[cur][kb][lane];
      const float odd = not_finite(v, 0.f);
      // (B's zeros above the diagonal meet no NaN and no infinity of a later token)
      own = kb == mt && __any(odd != odd) ? step4_lower(tri[x], v, own) : step4(tri[x], v, own);
    }
    // (what the chunk adds is summed by itself: one rounding at the state's size a chunk, not one a product)
#pragma unroll
    for (int kb = 0; kb < KT; ++kb) acc[2 + (kb & 1)] = step4(upd[kb], Vs[cur][kb][lane], acc[2 + (kb & 1)]);
    S = S * decay + (acc[2] + acc[3]);
    if (i + 1 < chunks) ask(from + step);
    const f32x4 Y = (acc[0] + acc[1]) + own;
    if (half == 1) Ps[cur][mt][lane] = Y;
    Ss[cur ^ 1][w][lane] = S;
    if (half == 0 && i + 1 < chunks) {
      Vs[cur ^ 1][mt][lane] = V;
      if (i + 2 < chunks) ask_v(c0 + 2 * CHUNK);
    }
    lds_barrier();
    if (half == 0) {
      const f32x4 whole = Y + Ps[cur][mt][lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const long long r = c0 + SUB * mt + 4 * g + e;
        if (live && r < r1) a.out[r * a.ldo + (long long)h * a.P + p] = whole[e];
      }
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int n = 16 * w + 4 * g + e;
    if (live && n < a.N) sp[n] = S[e];
  }
}

}  // namespace

// Float32 scratch with which a launch runs in chunks (0: token by token).  Microseconds a launch, token by token and in
// chunks, 16 heads of 128 x 128 over 8 q/k heads, a decay every channel (the unit vectors' launch in both): 48 tokens
// 32 / 34, 64 tokens 39 / 34, 256 tokens 124 / 49, 2 048 tokens 902 / 148 (one decay a head 654 / 146), eight of 64 93 / 62, eight of 512
// 586 / 230.  Of 2 048 tokens' 148 the preparation is 50 (21 for a workgroup by itself, a compute unit's LDS holds one), the walk 85
// (2.55 a chunk, of which the matrix instructions of a SIMD are 1.5: half the chip is idle with 128 workgroups).
// Relative error against 64 bits at 2 048 tokens: 3.3e-7 both ways with a decay every channel, 4.9e-7 and 5.1e-7
// with one a head; of the state at their end 3.4e-7 and 3.3e-7, 4.5e-7 both.
constexpr int LQ_DELTA_MIN = 56;
// A step's sequences of fewer tokens than this walk, beside the longer ones in chunks: a chunk of one token costs as much
// as one of 64 wherever all chunks together are more than the chip takes at once.  Microseconds, 16 heads of 128 x 128, a
// decay a channel, token by token / all in chunks / the long ones only: 512 tokens beside 16 of 1 308 / 131 / 106, 2 000
// beside 70 of 1 1 225 / 460 / 358; a decay a head, 2 000 beside eight of 20 632 / 209 / 187.
int lq_delta_least_rows(int rows, int batch, int heads, int channel_decay) {
  return most_chunks(rows, batch, 1) * heads <= lq_compute_units() ? 1 : channel_decay ? 24 : 48;
}
extern "C" long long lq_delta_scan_least(int heads);
// A launch of more chunks than the scratch holds goes in rounds of equal numbers of them, each from the state that the
// last one left: a prompt's scratch is bounded (131.6 KB a chunk and head: 4.3 GB for 65 536 rows of 16 heads).  Rounds
// cost where the sequences of one leave the chip idle: 32 heads, four of 2 048 tokens 1 007 us in one round (556 MB), 1 002
// with 256 MB, 1 065 with 128, 1 093 with 64; 8 192 tokens of one sequence 928, 982, 965, 999; 16 heads, eight of 512 240
// in one round (152 MB), 279 with 128 MB, 287 with 64.
constexpr long long LQ_DELTA_SCRATCH = 64ll << 20;  // floats
extern "C" long long lq_delta_scan_workspace(int rows, int batch, int heads, int Dk, int P, int max_rows) {
  if (rows <= 0 || batch <= 0 || heads <= 0 || P <= 0 || Dk <= 0 || Dk > NMAX || max_rows < LQ_DELTA_MIN) return 0;
  if (heads > 65535 || lq_ceil_div(P, 16) > 65535) return 0;
  return chunks_scratch(most_chunks(rows, batch, lq_delta_least_rows(rows, batch, heads, 1)), lq_delta_scan_least(heads), LQ_DELTA_SCRATCH);
}
extern "C" long long lq_delta_scan_least(int heads) { return (long long)heads * PART; }  // of one chunk

// Whether a launch is faster in chunks (given scratch) than token by token, by what both take.  A chunk costs the same
// whatever the sizes (their zeros are multiplied too) and however few tokens it has; a walk's token costs little where
// states are small or one decay serves a head, as soon as there are workgroups for the whole chip.  Microseconds, walk /
// chunks, 16 heads of 128 x 128: a decay a head, one of 64 tokens 30 / 32, of 256 89 / 44, 16 of 100 124 / 134, of 200 231 / 222, eight of
// 512 284 / 212, 200 beside 16 of 1 87 / 64; a decay a channel, 16 of 64 173 / 117, 70 of 64 681 / 443; of 64 x 64, 200 beside 16 of 1 73 / 49,
// with a decay a channel eight of 130 64 / 78, 16 of 512 261 / 368.  Over 1 800 launches (nine sizes, both decays, 1 to 128 sequences, alike or one beside
// shorter ones) the way that is named takes 0.4 % more than the better of the two, and in 49 of them 5 % and more.  (Priced as when a
// chunk of the walk took 3.4 microseconds, and with a tenth in the chunks' favour: 1.0 %, and 95.)
extern "C" int lq_delta_scan_in_chunks(int rows, int batch, int heads, int Dk, int P, int max_rows, int channel_decay) {
  if (lq_delta_scan_workspace(rows, batch, heads, Dk, P, max_rows) == 0) return 0;
  const double size = P / 128.0 * (Dk > 64 ? Dk / 128.0 : 0.4), cols = (P + 15) / 16;
  const double latency = channel_decay ? 0.42 : 0.31, token = (channel_decay ? 8.5e-3 : 3.7e-3) * size * heads;
  const double state = (channel_decay ? 0.12 : 0.045) * size * heads;  // a sequence's state, read and written
  auto walk = [&](double n, double longest, double sequences) {
    return 10 + sqrt(token * n * token * n + latency * longest * latency * longest) + state * sequences;
  };
  // the sequences beside the longest, by their mean, go in chunks as it does or all token by token
  const double rest = rows - max_rows, least = lq_delta_least_rows(rows, batch, heads, channel_decay);
  const bool alike = batch == 1 || rest >= least * (batch - 1);
  const double in_chunks = alike ? batch : 1, of_chunks = (alike ? rows : max_rows) / 64.0 + in_chunks / 2;
  const double products = 0.0113 * cols * heads * of_chunks, chain = 2.55 * (max_rows / 64 + 1);
  double chunks = 25 + 0.085 * heads * of_chunks + (products > chain ? products : chain) + 0.15 * P / 128 * heads * in_chunks;
  if (!alike) chunks += walk(rest, least, batch - 1);
  return chunks < walk(rows, max_rows, batch);
}

// q and k hold unit vectors already.  `scratch`: at least a chunk's floats for every head.  -> 0, or -2
int lq_delta_chunks(const float* q, int ldq, const float* k, int ldk, const float* v, int ldv, const float* beta,
                    int ldbeta, const float* a, int lda, const float* dt_bias, const float* a_log, float* state, float* out,
                    int ldo, int heads, int kv_heads, int Dk, int P, const int* seq_slot, const int* cu_rows, int batch,
                    int rows, int channel_decay, float* scratch, long long scratch_floats, hipStream_t stream) {
  DeltaArgs d = {q, k, v, beta, a, dt_bias, a_log, ldq, ldk, ldv, ldbeta, lda, ldo, state, out, scratch,
                 heads, kv_heads, Dk, P, batch, channel_decay, seq_slot, cu_rows, lq_delta_least_rows(rows, batch, heads, channel_decay), 0, 0, 0.f, 0.f};
  const bool quads = Dk % 4 == 0 && ldq % 4 == 0 && ldk % 4 == 0 && (!channel_decay || lda % 4 == 0) &&
                     (((uintptr_t)q | (uintptr_t)k | (channel_decay ? (uintptr_t)a | (uintptr_t)dt_bias : 0)) & 15) == 0;
  const auto prepare = quads ? delta_prepare_kernel<true, true> : delta_prepare_kernel<false, true>;
  static bool configured[2] = {false, false};
  if (!configured[quads]) {
    const hipError_t e = hipFuncSetAttribute((const void*)prepare, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(Prepared));
    if (e != hipSuccess) {
      lq_set_error("delta_scan: cannot reserve %d bytes of LDS: %s", (int)sizeof(Prepared), hipGetErrorString(e));
      return -2;
    }
    configured[quads] = true;
  }
  const long long all = most_chunks(rows, batch, d.least), room = chunks_a_round(all, scratch_floats, lq_delta_scan_least(heads));
  for (long long first = 0; first < all; first += room) {
    d.first = (int)first, d.last = (int)(first + room < all ? first + room : all);
    prepare<<<dim3(d.last - d.first, heads), 512, sizeof(Prepared), stream>>>(d);
    LQ_CHECK_LAUNCH("delta_scan(chunks)");
    delta_walk_kernel<<<(unsigned)((long long)batch * heads * lq_ceil_div(P, 16)), 512, 0, stream>>>(d);
    LQ_CHECK_LAUNCH("delta_scan(walk over chunks)");
  }
  return 0;
}

// ---- gated linear attention
// Float32 scratch for a launch in chunks (0: sizes that are not taken: key heads of more than 128, portions below 48 tokens, 96 of
// states of up to 4 096 entries).  Microseconds, token by token (in segments where it has them) and
// in chunks, heads of 128 x 256: 8 heads, 48 tokens 28 / 25, 128 tokens 59 / 30, 512 159 / 44, 3 000 781 / 144, eight sequences
// of 200 to 700 710 / 135, 24 of 120 400 / 119; 16 heads, 2 048 994 / 119; 4 heads of 64 x
// 64, 300 tokens 99 / 35.  Error against 64 bits, 2 048 tokens of 128 x 256: 2.8e-6 and 5.0e-7, of the state they leave
// 4.3e-6 and 3.1e-7; 64 tokens 2.2e-7 and 2.3e-7.
extern "C" long long lq_gla_chunks_workspace(int rows, int batch, int heads, int Dk, int P, int max_rows) {
  if (rows <= 0 || batch <= 0 || heads <= 0 || P <= 0 || Dk <= 0 || Dk > NMAX || max_rows < (Dk * P > 4096 ? 48 : 96)) return 0;
  if (heads > 65535 || lq_ceil_div(P, 16) > 65535) return 0;
  return chunks_scratch(most_chunks(rows, batch, 1), lq_delta_scan_least(heads), LQ_DELTA_SCRATCH);
}

// Whether a launch is faster in chunks than token by token, by what both take.  A chunk costs the same however few tokens it has, so
// that one prompt beside many single tokens, or many short portions, may be sooner walked.  Microseconds, walk / chunks, 16 heads of 64 x
// 128: 300 tokens alone 99 / 37, beside 31 single ones 127 / 115, beside 128 160 / 405; 48 beside 128 77 / 387; 24 portions of 64 74 / 92, 96
// of 64 261 / 357; 16 heads of 128 x 256, 64 tokens beside 128 554 / 740, 512 beside 128 818 / 775.  Over 1 116 launches (see lq_gla_walk_us; this
// estimate is off by 13 %) the way that is named takes 0.5 % more than the better of the two, and in five of them 5 % and more above the walk
// (64 heads of 64 x 64, two sequences of 1 000 beside 30 of 5: 344 / 567; 16 of 64 x 128, eight of 512 beside 56 of 1: 273 / 340).
double lq_gla_walk_us(int rows, int batch, int heads, int N, int P, int max_rows);
extern "C" int lq_gla_scan_in_chunks(int rows, int batch, int heads, int Dk, int P, int max_rows) {
  if (lq_gla_chunks_workspace(rows, batch, heads, Dk, P, max_rows) == 0) return 0;
  const double longest = lq_ceil_div(max_rows, CHUNK), others = batch - 1, mean = others > 0 ? (rows - max_rows) / others / CHUNK + 0.5 : 0;
  const double chunks = heads * (longest + others * (mean > 1 ? mean : 1));
  const double products = 0.005 * lq_ceil_div(P, 16) * chunks, chain = 2.5 * longest, state = (double)batch * heads * P * Dk / (128 * 128);
  const double us = 20 + (Dk % 4 == 0 ? 0.09 : 0.1) * chunks + (products > chain ? products : chain) + 0.076 * state;
  return us < lq_gla_walk_us(rows, batch, heads, Dk, P, max_rows);
}

int lq_gla_chunks(const float* q, int ldq, const float* k, int ldk, const float* v, int ldv, const float* z, int ldz, const float* bias,
                  float* state, float* out, int ldo, int heads, int Dk, int P, float q_scale, float inv_tau, const int* seq_slot,
                  const int* cu_rows, int batch, int rows, float* scratch, long long scratch_floats, hipStream_t stream) {
  DeltaArgs d = {q, k, v, nullptr, z, bias, nullptr, ldq, ldk, ldv, 0, ldz, ldo, state, out, scratch, heads, heads, Dk, P, batch, 1,
                 seq_slot, cu_rows, 1, 0, 0, q_scale, inv_tau};
  const bool quads = Dk % 4 == 0 && ldq % 4 == 0 && ldk % 4 == 0 && ldz % 4 == 0 &&
                     (((uintptr_t)q | (uintptr_t)k | (uintptr_t)z | (uintptr_t)bias) & 15) == 0;
  const auto prepare = quads ? delta_prepare_kernel<true, false> : delta_prepare_kernel<false, false>;
  static bool configured[2] = {false, false};
  if (!configured[quads]) {
    const hipError_t e = hipFuncSetAttribute((const void*)prepare, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(Prepared));
    if (e != hipSuccess) {
      lq_set_error("gla_scan: cannot reserve %d bytes of LDS: %s", (int)sizeof(Prepared), hipGetErrorString(e));
      return -2;
    }
    configured[quads] = true;
  }
  const long long all = most_chunks(rows, batch, 1), room = chunks_a_round(all, scratch_floats, lq_delta_scan_least(heads));
  for (long long first = 0; first < all; first += room) {
    d.first = (int)first, d.last = (int)(first + room < all ? first + room : all);
    prepare<<<dim3(d.last - d.first, heads), 512, sizeof(Prepared), stream>>>(d);
    LQ_CHECK_LAUNCH("gla_scan(chunks)");
    gla_walk_kernel<<<(unsigned)((long long)batch * heads * lq_ceil_div(P, 16)), 512, 0, stream>>>(d);
    LQ_CHECK_LAUNCH("gla_scan(walk over chunks)");
  }
  return 0;
}
