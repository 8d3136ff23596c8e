// The state-space scan over long portions of a sequence, in chunks of 64 tokens on the matrix cores.
//
// Token by token (recurrent.hip):  S <- d_t S + s_t B_t x_t^T,  y_t = S^T C_t + D x_t, one decay d_t and step s_t a token
// and head.  Over a chunk that starts from the state S, with p_t = d_1 .. d_t and f_st = d_(s+1) .. d_t (products of numbers
// up to 1, never quotients):
//   y_t = p_t S^T C_t + sum_(s <= t) f_st s_s (C_t . B_s) x_s + D x_t,      S <- p_64 S + sum_s f_s,64 s_s B_s x_s^T
// Three launches: what every chunk adds to the state; the chunks' starts, one after the other, entry by entry; the results
// from a chunk's start and its own tokens.  Only the second has a chain along the sequence.  (The walk in eight segments
// that this replaces ran every segment's chain of exchanges over lanes twice, on 8 x 4 x 32 workgroups of the 2 048
// tokens and 32 heads below.)
//
// Everything is 32-bit (v_mfma_f32_16x16x4_f32; the order of k and the fragments as in delta_chunks.hip).  A state in the
// scratch lies in tiles of 16 channels n by 16 columns p in a result's order, lane l's four entries (n = 4 (l / 16) .. + 3,
// p = l % 16) at 4 l, which is also the order in which the third launch takes it as an operand.
// Chunks count from a sequence's first row of the step; a last chunk's missing tokens take part as zeros.
#include <cmath>
#include <type_traits>

#include "scan_chunks.h"

namespace {

constexpr int HALF = 128, NT = HALF / 16;  // channels that a workgroup holds in LDS at a time
constexpr int COLS = 64;                   // columns of the values a workgroup

struct SsdArgs {
  const float *x, *B, *C, *dt, *dt_bias, *a_log, *d_skip, *decay;
  int ldx, ldb, ldc, lddt, lddecay, ldy;
  float *state, *y, *scratch, *ends;  // scratch: [chunk][head][state]; ends: [chunk][head], p_64
  int heads, groups, N, P, ones, batch;
  const int *seq_slot, *cu_rows;
  int least;        // sequences of fewer tokens are not taken
  int first, last;  // the chunks of these three launches: numbers first .. last - 1, the scratch of `first` at its start
};

__host__ __device__ inline int n_tiles(int N) { return (N + HALF - 1) / HALF * NT; }
__host__ __device__ inline int p_tiles(int P) { return (P + 15) / 16; }
__host__ __device__ inline long long part_floats(int N, int P) { return (long long)n_tiles(N) * p_tiles(P) * FRAG; }

// A token's decay and step (one thread a token; past the portion's end: nothing decays and nothing is added).
__device__ inline void token_scalars(const SsdArgs& a, long long row, bool there, int h, float& decay, float& step) {
  decay = 1.f, step = 0.f;
  if (!there) return;
  const float z = a.dt[row * a.lddt + h];
  if (a.decay != nullptr) {
    decay = a.decay[row * a.lddecay + h], step = z;
  } else {
    step = softplus_f(z + a.dt_bias[h]);
    decay = expf(-expf(a.a_log[h]) * step);
  }
}

// A thread's share of ROWS = 64 rows of W columns, as whole vectors or entry by entry; every load is asked for before
// the first is stored.
template <int W, int TH, bool QUADS>
struct Slab {
  static constexpr int PER = CHUNK * W / 4 / TH;
  f32x4 v[PER];
  __device__ void fetch(const float* from, long long ld, int rows, int cols) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = threadIdx.x + TH * i, t = e / (W / 4), n = e % (W / 4) * 4;
      v[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
      if (t < rows) {
        const float* p = from + t * ld + n;
        if constexpr (QUADS) {
          if (n + 3 < cols) v[i] = *(const f32x4*)p;
          else
            for (int x = 0; x < 4; ++x) v[i][x] = n + x < cols ? p[x] : 0.f;
        } else {
#pragma unroll
          for (int x = 0; x < 4; ++x) v[i][x] = n + x < cols ? p[x] : 0.f;
        }
      }
    }
  }
  __device__ void stash(float* to, int ld) const {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = threadIdx.x + TH * i, t = e / (W / 4), n = e % (W / 4) * 4;
      *(f32x4*)(to + t * ld + n) = v[i];
    }
  }
};

constexpr int LDN = HALF + 4, LDX = COLS + 4;  // floats a row of LDS: rows four apart start 16 banks apart

// What a chunk adds to the state.  One workgroup of four wavefronts a (chunk, head, 64 columns).
template <bool QUADS>
__global__ __launch_bounds__(256) void ssd_chunk_state_kernel(SsdArgs a) {
  __shared__ __attribute__((aligned(16))) float Bs[CHUNK][LDN], Xs[CHUNK][LDX];
  __shared__ float weight[CHUNK];
  const Part at = find_part(a.cu_rows, a.batch, CHUNK, a.least, a.first + blockIdx.x);
  if (at.seq < 0) return;
  const int h = blockIdx.y, grp = h / (a.heads / a.groups), p0 = blockIdx.z * COLS, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int c = lane & 15, g = lane >> 4, Px = a.P - a.ones;
  const long long r0 = at.first, place = (long long)blockIdx.x * a.heads + h;
  const int nt = at.rows;
  Slab<COLS, 256, QUADS> xs;
  Slab<HALF, 256, QUADS> bs;
  xs.fetch(a.x + r0 * a.ldx + (long long)h * Px + p0, a.ldx, nt, Px - p0);
  bs.fetch(a.B + r0 * a.ldb + (long long)grp * a.N, a.ldb, nt, a.N);
  if (w == 0) {
    float d, s;
    token_scalars(a, r0 + lane, lane < nt, h, d, s);
    float upto = d;  // d_lane .. d_63
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float later = __shfl_down(upto, off, 64);
      if (lane + off < 64) upto *= later;
    }
    const float after = __shfl_down(upto, 1, 64);
    weight[lane] = s * (lane < 63 ? after : 1.f);
    if (lane == 0 && blockIdx.z == 0) a.ends[place] = upto;
  }
  xs.stash(&Xs[0][0], LDX);
  __syncthreads();
  // the tokens' weights go onto x (and onto the column of ones)
  for (int e = tid; e < CHUNK * COLS; e += 256) {
    const int t = e / COLS, p = e % COLS;
    Xs[t][p] = (a.ones && p0 + p == Px && t < nt ? 1.f : Xs[t][p]) * weight[t];
  }
  const int tiles_p = p_tiles(a.P), pt0 = p0 / 16, pts = min(COLS / 16, tiles_p - pt0);
  for (int n0 = 0; n0 < a.N; n0 += HALF) {
    if (n0 > 0) {
      __syncthreads();
      bs.fetch(a.B + r0 * a.ldb + (long long)grp * a.N + n0, a.ldb, nt, a.N - n0);
    }
    bs.stash(&Bs[0][0], LDN);
    __syncthreads();
    f32x4 acc[2][COLS / 16];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < COLS / 16; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < KT; ++kb) {
      const int t = SUB * kb + 4 * g;
      f32x4 n_[2], x_[COLS / 16];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int s = 0; s < 4; ++s) n_[i][s] = Bs[t + s][16 * (w + 4 * i) + c];
#pragma unroll
      for (int j = 0; j < COLS / 16; ++j)
#pragma unroll
        for (int s = 0; s < 4; ++s) x_[j][s] = Xs[t + s][16 * j + c];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < COLS / 16; ++j) acc[i][j] = step4(n_[i], x_[j], acc[i][j]);
    }
    float* to = a.scratch + place * part_floats(a.N, a.P);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < COLS / 16; ++j)
        if (j < pts) *(f32x4*)(to + (((long long)(n0 / 16 + w + 4 * i) * tiles_p + pt0 + j) * 64 + lane) * 4) = acc[i][j];
  }
}

// In every chunk's place the state that it starts from, and the last one's end into the cache.  A thread four entries of
// a (sequence, head)'s state; four chunks' loads are asked for together.
__global__ __launch_bounds__(256) void ssd_chunk_chain_kernel(SsdArgs a) {
  const int b = blockIdx.x / a.heads, h = blockIdx.x % a.heads, tiles_p = p_tiles(a.P);
  const int base = first_chunk(a.cu_rows, b, a.least), i0 = max(a.first - base, 0);
  const int chunks = min(chunks_of(a.cu_rows[b + 1] - a.cu_rows[b], a.least), a.last - base) - i0;  // from the sequence's i0th on
  const long long part = part_floats(a.N, a.P), place = (long long)(base + i0 - a.first) * a.heads + h;
  const long long quad = (long long)blockIdx.y * 256 + threadIdx.x;
  if (chunks <= 0 || quad * 4 >= part) return;
  const int tile = (int)(quad / 64), lane = (int)(quad % 64);
  const int n = tile / tiles_p * 16 + 4 * (lane >> 4), p = tile % tiles_p * 16 + (lane & 15);
  float* sp = a.state + (((long long)a.seq_slot[b] * a.heads + h) * a.P + min(p, a.P - 1)) * a.N;
  f32x4 S;
#pragma unroll
  for (int e = 0; e < 4; ++e) S[e] = p < a.P && n + e < a.N ? sp[n + e] : 0.f;
  const long long step = (long long)a.heads * part;
  float* at = a.scratch + place * part + quad * 4;
  const float* ends = a.ends + place;
  for (int done = 0; done < chunks; done += 4) {
    f32x4 add[4];
    float d[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = min(done + j, chunks - 1);
      add[j] = *(const f32x4*)(at + i * step), d[j] = ends[(long long)i * a.heads];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (done + j < chunks) {
        *(f32x4*)(at + (done + j) * step) = S;
        S = S * d[j] + add[j];
      }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (p < a.P && n + e < a.N) sp[n + e] = S[e];
}

// (64 channels at a time: 70 KB of LDS, two workgroups a compute unit, whose loads, decays and products overlap)
constexpr int RUN = 64, RT = RUN / 16, LDR = RUN + 4;

struct OutLds {
  float C[CHUNK][LDR], B[CHUNK][LDR], x[CHUNK][LDX];
  float G[CHUNK][LDX];  // first f_st s_s, then that times C_t . B_s
  float decay[CHUNK], step[CHUNK], from_start[CHUNK];
  int odd;  // x or B has an entry that is no finite number
};

// A chunk's results.  One workgroup of eight wavefronts a (chunk, head, 64 columns): wavefronts w and w + 4 take 16
// columns, the first its first 32 tokens and the second its last.  A workgroup is a chain of trips to memory, the decays' products
// and 4 microseconds of matrix instructions; one a compute unit (128 channels at a time), with the decays' products of 64 tokens in
// one wavefront's row, took 17.  32 heads of 128 x 64, 2 048 tokens: 68
// -> 46 us.
template <bool QUADS>
__global__ __launch_bounds__(512, 4) void ssd_chunk_out_kernel(SsdArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  OutLds& L = *(OutLds*)smem;
  const Part at = find_part(a.cu_rows, a.batch, CHUNK, a.least, a.first + blockIdx.x);
  if (at.seq < 0) return;
  const int h = blockIdx.y, grp = h / (a.heads / a.groups), p0 = blockIdx.z * COLS, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int c = lane & 15, g = lane >> 4, Px = a.P - a.ones, pt = w & 3, m0 = w >> 2 << 1;  // token tiles m0 and m0 + 1
  const long long r0 = at.first, place = (long long)blockIdx.x * a.heads + h;
  const int nt = at.rows, tiles_p = p_tiles(a.P);
  const float* start = a.scratch + place * part_floats(a.N, a.P);
  const int my_pt = min(p0 / 16 + pt, tiles_p - 1);
  Slab<COLS, 512, QUADS> xs;
  Slab<RUN, 512, QUADS> cs, bs;
  auto ask = [&](int n0) {
    cs.fetch(a.C + r0 * a.ldc + (long long)grp * a.N + n0, a.ldc, nt, a.N - n0);
    bs.fetch(a.B + r0 * a.ldb + (long long)grp * a.N + n0, a.ldb, nt, a.N - n0);
  };
  ask(0);
  xs.fetch(a.x + r0 * a.ldx + (long long)h * Px + p0, a.ldx, nt, Px - p0);
  if (tid == 0) L.odd = 0;
  if (tid < CHUNK) token_scalars(a, r0 + tid, tid < nt, h, L.decay[tid], L.step[tid]);
  xs.stash(&L.x[0][0], LDX);
  float nan_if = 0.f;
#pragma unroll
  for (int i = 0; i < xs.PER; ++i) nan_if = not_finite(xs.v[i], nan_if);
  __syncthreads();
  if (a.ones && tid < nt && Px >= p0 && Px < p0 + COLS) L.x[tid][Px - p0] = 1.f;
  if (w >= KT) {  // f_st s_s, lane s: wavefront KT + j the 16 tokens t of block j
    const int j = w - KT, blk = lane >> 4;
    float v = L.decay[lane];  // the products of a block's decays from a token to the block's end
#pragma unroll
    for (int off = 1; off < SUB; off <<= 1) {
      const float later = __shfl_down(v, off, 64);
      if ((lane & 15) + off < SUB) v *= later;
    }
    const float after = __shfl_down(v, 1, 64);
    float f = L.step[lane];
    if (blk < j) {  // what lies between the token and block j
      if ((lane & 15) < SUB - 1) f *= after;
    } else if (blk > j) {
      f = 0.f;
    }
#pragma unroll
    for (int i = 1; i < KT - 1; ++i) {
      const float whole = __shfl(v, SUB * i, 64);
      if (blk < i && i < j) f *= whole;
    }
#pragma unroll
    for (int i = 0; i < SUB; ++i) {
      const int t = SUB * j + i;
      if (t > lane) f *= L.decay[t];
      L.G[t][lane] = t >= lane ? f : 0.f;
    }
  } else if (w == 0) {  // p_t
    float p = L.decay[lane];
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float before = __shfl_up(p, off, 64);
      if (lane >= off) p *= before;
    }
    L.from_start[lane] = p;
  }
  // C_t . B_s: ten tiles at and below the diagonal, wavefront w the tiles w and w + 8
  f32x4 inter[2][4], G[2];  // (four chains of products: their roundings are smaller, and none waits for the one before it)
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    G[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) inter[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }
  auto tile_of = [](int u, int& mt, int& st) { mt = u < 1 ? 0 : u < 3 ? 1 : u < 6 ? 2 : 3, st = u - mt * (mt + 1) / 2; };
  for (int n0 = 0; n0 < a.N; n0 += RUN) {
    f32x4 S[RT];  // (used last)
#pragma unroll
    for (int nb = 0; nb < RT; ++nb) S[nb] = *(const f32x4*)(start + (((long long)(n0 / 16 + nb) * tiles_p + my_pt) * 64 + lane) * 4);
    cs.stash(&L.C[0][0], LDR), bs.stash(&L.B[0][0], LDR);
#pragma unroll
    for (int i = 0; i < bs.PER; ++i) nan_if = not_finite(bs.v[i], nan_if);
    if (nan_if != nan_if) L.odd = 1;  // (read behind the barriers below)
    __syncthreads();
    if (n0 + RUN < a.N) ask(n0 + RUN);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int u = w + 8 * i;
      if (u < 10) {
        int mt, st;
        tile_of(u, mt, st);
        f32x4 acc[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) acc[x] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int nb = 0; nb < RT; ++nb)
          acc[nb & 3] = step4(*(const f32x4*)&L.C[SUB * mt + c][16 * nb + 4 * g], *(const f32x4*)&L.B[SUB * st + c][16 * nb + 4 * g],
                              acc[nb & 3]);
        G[i] += (acc[0] + acc[1]) + (acc[2] + acc[3]);
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int nb = 0; nb < RT; ++nb)
        inter[i][nb & 3] = step4(*(const f32x4*)&L.C[SUB * (m0 + i) + c][16 * nb + 4 * g], S[nb], inter[i][nb & 3]);
    __syncthreads();
  }
  f32x4 own[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) own[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  // `careful`: what is no finite number reaches no earlier token
  auto scaled = [&](auto careful) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int u = w + 8 * i;
      if (u < 10) {
        int mt, st;
        tile_of(u, mt, st);
#pragma unroll
        for (int e = 0; e < 4; ++e)  // (above the diagonal zeros, which a NaN in a later token's B must leave as they are)
          if (!careful || mt > st || 4 * g + e >= c) L.G[SUB * mt + 4 * g + e][SUB * st + c] *= G[i][e];
      }
    }
    __syncthreads();
  };
  auto own_tokens = [&](auto careful) {
#pragma unroll
    for (int kb = 0; kb < KT; ++kb) {
      if (kb > m0 + 1) continue;
      f32x4 x_;
#pragma unroll
      for (int s = 0; s < 4; ++s) x_[s] = L.x[SUB * kb + 4 * g + s][16 * pt + c];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (kb <= m0 + i) {
          const f32x4 G_ = *(const f32x4*)&L.G[SUB * (m0 + i) + c][SUB * kb + 4 * g];
          own[i] = careful && kb == m0 + i ? step4_lower(G_, x_, own[i]) : step4(G_, x_, own[i]);
        }
    }
  };
  if (__builtin_amdgcn_readfirstlane(L.odd)) scaled(std::true_type{}), own_tokens(std::true_type{});
  else scaled(std::false_type{}), own_tokens(std::false_type{});
  const int p = p0 + 16 * pt + c;
  const float D = a.decay == nullptr ? a.d_skip[h] : 0.f;
  if (p >= a.P) return;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = SUB * (m0 + i) + 4 * g + e;
      if (t < nt)
        a.y[(r0 + t) * a.ldy + (long long)h * a.P + p] =
            fmaf(D, L.x[t][16 * pt + c], fmaf(L.from_start[t], (inter[i][0][e] + inter[i][1][e]) + (inter[i][2][e] + inter[i][3][e]), own[i][e]));
    }
}

}  // namespace

// From 128 rows of the longest sequence on, states of up to 256 channels (two rounds through LDS).  Microseconds a launch,
// token by token (long sequences in segments) and in chunks: 32 heads of 128 x 64 over 8 groups, 130 tokens 42 / 26, 512
// tokens 83 / 41, 2 048 tokens 263 / 88, eight of 130 72 / 65, eight of 512 233 / 142; a matrix memory of 4 heads of 256 x
// 512, two sequences of 1 000 and 1 100 tokens 635 / 134.  Relative error
// against 64 bits: 5.9e-8 and 4.7e-8 at 2 048 tokens (of the state 4.8e-7 and 4.4e-7), 1.4e-7 and 1.7e-7 of the memory's
// results (of its state 1.2e-7 and 1.1e-7).
constexpr int LQ_SSD_MIN = 128;
// A step's sequences of fewer tokens than this walk, beside the longer ones in chunks: a chunk of one token costs as much
// as one of 64 wherever all chunks together are more than the chip takes at once.  Microseconds, 32 heads of 128 x 64, token by token / all in
// chunks / the long ones only: 512 tokens beside 16 of 1 164 / 94 / 69, 2 000 beside eight of 20 544 / 134 / 129, a memory
// of 256 x 513, 2 000 beside eight of 1 925 / 207 / 195.
int lq_ssd_least_rows(int rows, int batch, int heads) { return most_chunks(rows, batch, 1) * heads <= lq_compute_units() ? 1 : 48; }

// A launch of more chunks than the scratch holds goes in rounds of equal numbers of them, each from the state that the
// last one left: a prompt's scratch is bounded (a matrix memory of 4 heads of 256 x 513 takes 2.2 MB a chunk).
// Microseconds in one round and with 256, 128 and 64 MB: 32 heads of 128 x 64, 32 768 tokens (538 MB) 1 476, 1 577,
// 1 537, 1 690; the memory, 8 192 tokens (279 MB) 610, 615, 643, 675, sixteen sequences of 512 (311 MB) 626, 664, 671, 811.
constexpr long long LQ_SSD_SCRATCH = 64ll << 20;  // floats

long long lq_ssd_chunks_least(int heads, int P, int N) { return heads * (part_floats(N, P) + 1); }  // of one chunk

long long lq_ssd_chunks_floats(int rows, int batch, int heads, int P, int N, int max_rows) {
  if (rows <= 0 || N > 2 * HALF || max_rows < LQ_SSD_MIN || heads > 65535 || lq_ceil_div(P, COLS) > 65535) return 0;
  return chunks_scratch(most_chunks(rows, batch, lq_ssd_least_rows(rows, batch, heads)), lq_ssd_chunks_least(heads, P, N), LQ_SSD_SCRATCH);
}

// Whether a launch is faster in chunks (given scratch) than token by token (`segments`: in segments), by what both take.
// A chunk of up to 128 channels costs the same however few they are and however few tokens it has; a walk's token costs little
// where states are small, as soon as there are workgroups for the whole chip.  Microseconds, walk / chunks, 32 heads: of
// 128 x 64, one sequence of 130 tokens 42 / 26, eight of 512 233 / 142, 32 of 256 461 / 318; of 64 x 64, eight of 256 90 / 76,
// 32 of 256 227 / 245, one of 2 048 181 / 75; of 16 x 64, four of 1 000 137 / 121, eight of 512 144 / 121; of 64 x 16, eight
// of 1 000 159 / 192.
bool lq_ssd_chunks_faster(int batch, int heads, int P, int N, int max_rows, int rows, bool segments) {
  if (lq_ssd_chunks_floats(rows, batch, heads, P, N, max_rows) == 0) return false;
  const double token = 1.75e-3 * P / 64 * (N > 128 ? N / 80.0 : N > 32 ? N / 128.0 : 0.25) * heads, state = 0.02 * P / 64 * N / 128 * heads;
  auto walk = [&](double n, double longest, double sequences, bool segments) {
    const double chain = segments ? 20 + 0.12 * longest : (N > 32 ? 0.3 : 0.45) * longest, all = (segments ? 2 : 1) * token * n;
    return 5 + (segments ? fmax(chain, all) : sqrt(chain * chain + all * all)) + state * sequences;
  };
  // the sequences beside the longest, by their mean, go in chunks as it does or all token by token
  const double rest = rows - max_rows, least = lq_ssd_least_rows(rows, batch, heads);
  const bool alike = batch == 1 || rest >= least * (batch - 1);
  const double of_chunks = alike ? rows / 64.0 + batch / 2.0 : max_rows / 64.0 + 0.5;
  double chunks = 24 + (N > HALF ? 0.1 : 0.061) * lq_ceil_div(P, COLS) * heads * of_chunks;
  if (!alike) chunks += 10 + walk(rest, least, batch - 1, false);
  return 0.9 * chunks < walk(rows, max_rows, batch, segments);
}

// -> 0, or -2.  `scratch`: lq_ssd_chunks_floats(...) floats, or fewer, down to lq_ssd_chunks_least(...)
int lq_ssd_chunks(const float* x, int ldx, const float* B, int ldb, const float* C, int ldc, const float* dt, int lddt,
                  const float* dt_bias, const float* a_log, const float* d_skip, float* state, float* y, int ldy, int heads,
                  int P, int N, int groups, const int* seq_slot, const int* cu_rows, int batch, int rows, float* scratch,
                  long long scratch_floats, const float* decay, int lddecay, int ones, hipStream_t stream) {
  const int least = lq_ssd_least_rows(rows, batch, heads);
  const long long all = most_chunks(rows, batch, least);
  const long long room = chunks_a_round(all, scratch_floats, lq_ssd_chunks_least(heads, P, N));
  SsdArgs a = {x, B, C, dt, dt_bias, a_log, d_skip, decay, ldx, ldb, ldc, lddt, lddecay, ldy, state, y, scratch,
               scratch + room * heads * part_floats(N, P), heads, groups, N, P, ones, batch, seq_slot, cu_rows, least, 0, 0};
  const bool quads = N % 4 == 0 && (P - ones) % 4 == 0 && ldx % 4 == 0 && ldb % 4 == 0 && ldc % 4 == 0 &&
                     (((uintptr_t)x | (uintptr_t)B | (uintptr_t)C) & 15) == 0;
  const auto state_kernel = quads ? ssd_chunk_state_kernel<true> : ssd_chunk_state_kernel<false>;
  const auto out_kernel = quads ? ssd_chunk_out_kernel<true> : ssd_chunk_out_kernel<false>;
  static bool configured[2] = {false, false};
  if (!configured[quads]) {
    const hipError_t e = hipFuncSetAttribute((const void*)out_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(OutLds));
    if (e != hipSuccess) {
      lq_set_error("ssd_scan: cannot reserve %d bytes of LDS: %s", (int)sizeof(OutLds), hipGetErrorString(e));
      return -2;
    }
    configured[quads] = true;
  }
  for (long long first = 0; first < all; first += room) {
    a.first = (int)first, a.last = (int)(first + room < all ? first + room : all);
    const dim3 grid(a.last - a.first, heads, lq_ceil_div(P, COLS));
    state_kernel<<<grid, 256, 0, stream>>>(a);
    LQ_CHECK_LAUNCH("ssd_scan(chunks' states)");
    ssd_chunk_chain_kernel<<<dim3((unsigned)batch * heads, (unsigned)lq_ceil_div64(part_floats(N, P), 1024)), 256, 0, stream>>>(a);
    LQ_CHECK_LAUNCH("ssd_scan(chunks in a chain)");
    out_kernel<<<grid, 512, sizeof(OutLds), stream>>>(a);
    LQ_CHECK_LAUNCH("ssd_scan(chunks' results)");
  }
  return 0;
}
