// y[M, N] = x[M, K] . W[N, K]^T  -- weights are [out, in], K contiguous in both
// (internal/device/kernels.metal:105-132: "y[b,row] = sum_k W[row,k] x[b,k]").
//
// This file holds the size-agnostic product: the whole of the float32 path and the fallback of the
// bfloat16 path for shapes that the bfloat16 matrix-core kernels refuse.  Operands are widened to
// float32 (never narrowed) and multiplied on the matrix cores in their true 32-bit mode,
// v_mfma_f32_16x16x4_f32: float32 in, float32 accumulate, no reduced-precision step anywhere.
//
// One summation tree for every output, whatever kernel, tile or batch it is computed in, so that a
// row's result does not depend on how many other rows the launch holds (bit for bit):
//   * K is cut into chunks of CHUNK = 256 consecutive k, counted from k = 0;
//   * a chunk's sum starts from zero and runs through the chunk in slabs of 16 k, a slab being four
//     matrix instructions: instruction j of a slab multiplies k0 + 4 g + j for g = 0..3 (the four k that
//     one instruction takes are spread over the slab so that a lane can fetch its four k of a slab as
//     16 consecutive bytes);
//   * the chunks' sums are added one after the other in ascending order, in float32.
// k past K count as zeros, which change no sum.  The rounding error of a long row grows with
// K / 256 + 64 additions instead of K.
//
// Three kernels: an LDS-tiled one (block tiles of 64 x 64 or 128 x 128, any size and alignment); a pipelined one of
// 32 to 128 x 128 tiles for float32 operands in whole pieces with K in 32s, from 17 rows of a wide weight on; and one for up to 64 rows
// that streams the weights straight from memory, a block of waves a tile of 16 columns, its waves taking chunks in turn and
// adding their sums up in order through LDS (up to 16 rows of float32 with K in 32s the weights come through LDS as well).
#include "common.h"

#include <type_traits>

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int CHUNK = 256, SLAB = 16;

// v_mfma_f32_16x16x4_f32: lane l gives A[row l % 16][k l / 16] and B[k l / 16][column l % 16] and holds
// D[4 (l / 16) + e][l % 16], e < 4.
__device__ inline f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// ---- tiled: 4 waves (2 x 2), a wave TM x TN tiles of 16 x 16 ---------------------------------------------
template <typename T, typename TO, int TM, int TN>
__global__ __launch_bounds__(256) void gemm_f32_tiled_kernel(const T* __restrict__ A, int lda, const T* __restrict__ W,
                                                             int ldw, TO* __restrict__ C, int ldc, int M, int N, int K) {
  constexpr int BM = 2 * TM * 16, BN = 2 * TN * 16;
  // k-major tiles; rows of BM + 4 floats put the four k that an instruction reads on different banks
  __shared__ float As[SLAB][BM + 4];
  __shared__ float Ws[SLAB][BN + 4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r16 = lane & 15, g = lane >> 4;
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  // loader: a thread takes 4 consecutive k of one row, 64 rows a pass
  const int lrow = tid >> 2, lk = (tid & 3) * 4;
  constexpr int PA = BM / 64, PW = BN / 64;

  f32x4 total[TM][TN], chunk[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      total[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
      chunk[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }

  float ra[PA][4], rw[PW][4];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int p = 0; p < PA; ++p) {
      const int m = m0 + p * 64 + lrow;
      const T* src = A + (long long)min(m, M - 1) * lda + k0 + lk;
#pragma unroll
      for (int u = 0; u < 4; ++u) ra[p][u] = (m < M && k0 + lk + u < K) ? to_f32(src[u]) : 0.f;
    }
#pragma unroll
    for (int p = 0; p < PW; ++p) {
      const int n = n0 + p * 64 + lrow;
      const T* src = W + (long long)min(n, N - 1) * ldw + k0 + lk;
#pragma unroll
      for (int u = 0; u < 4; ++u) rw[p][u] = (n < N && k0 + lk + u < K) ? to_f32(src[u]) : 0.f;
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int p = 0; p < PA; ++p)
#pragma unroll
      for (int u = 0; u < 4; ++u) As[lk + u][p * 64 + lrow] = ra[p][u];
#pragma unroll
    for (int p = 0; p < PW; ++p)
#pragma unroll
      for (int u = 0; u < 4; ++u) Ws[lk + u][p * 64 + lrow] = rw[p][u];
  };

  fetch(0);
  for (int k0 = 0; k0 < K; k0 += SLAB) {
    stage();
    __syncthreads();
    if (k0 + SLAB < K) fetch(k0 + SLAB);  // the next slab is on its way while this one is multiplied
#pragma unroll
    for (int j4 = 0; j4 < 4; ++j4) {
      float a[TM], b[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) a[i] = As[4 * g + j4][(wm * TM + i) * 16 + r16];
#pragma unroll
      for (int j = 0; j < TN; ++j) b[j] = Ws[4 * g + j4][(wn * TN + j) * 16 + r16];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) chunk[i][j] = mfma4(a[i], b[j], chunk[i][j]);
    }
    if ((k0 + SLAB) % CHUNK == 0 || k0 + SLAB >= K) {
      // a chunk is complete: it joins the running sum, and the next starts from zero
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          total[i][j] += chunk[i][j];
          chunk[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
        }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + (wn * TN + j) * 16 + r16;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + (wm * TM + i) * 16 + 4 * g + e;
        if (m < M && n < N) C[(long long)m * ldc + n] = from_f32<TO>(total[i][j][e]);
      }
    }
}

// ---- pipelined: the same tiles, operands in whole pieces ---------------------------------------------------
// 32 TM x 128 a block (TM 1 to 4), 4 waves of 16 TM x 64.  Stages of 32 k (two slabs) go from memory straight into LDS (16 bytes a lane, no
// registers): the next one's transfers fly while this one is multiplied, 32 TM matrix instructions a wave, behind one barrier a
// stage.  A lane's four k of a slab are one 16-byte read.  An LDS row is 32 k, 128 bytes; its
// piece u lies at u ^ (row / 2 % 8), so that the 16 rows of a fragment lie in different banks.  Two blocks a compute
// unit, so that one multiplies while the other waits at its barrier.  The tiles go to the dies in runs, row tiles first:
// a die's blocks share their weights.
// What bounded the kernel above: its LDS accesses, four bytes at a time, two barriers a slab.  What bounds this one: the matrix units, busy
// 95 % of the time at whole rounds, and the last round where it is not whole.  Reads (of the slab after) and transfers are dealt out among a slab's
// products, one in every four to eight: asked for together, 8 of 1 KiB a wave, they fill the queues before memory and LDS, and
// the wave stands with them in front of its products; the matrix units were then busy 83 % of the time, whether one block was on a
// compute unit or two, whether the data were zeros or not, and whether the reads were asked for a slab ahead (each by itself nothing).
// Microseconds, above, all at a stage's start and dealt out (the same bits): 865 x 28 672 x 4 096 3 181 / 1 775 / 1 517 (64 / 114 / 134 of
// 157 TFLOP/s), 865 x 4 096 x 14 336 2 214 / 932 / 844, 333 x 28 672 x 4 096 725 / 619, 2 048 x 28 672 x 4 096 6 438 / 3 644 / 3 243 (148 TFLOP/s).
// One tile of 32 rows a compute unit keeps three stages: a slab's products are then too short for a transfer (90 us with two stages, 81
// with three, K 4 096).  Several such tiles run four a compute unit with two stages (three tiles 193 us, with three stages 206); with 64
// and 96 rows a third stage gave nothing or took 6 %.
constexpr int STAGE_K = 32, TILE = 128;

// 16 bytes a lane from `base`, which holds `range` bytes, to LDS: lane l's from base + offset + skip to `lds` + 16 l.
__device__ __forceinline__ void piece_to_lds(const float* base, int range, int offset, int skip, unsigned char* lds) {
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, range, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)lds, 16, offset, skip, 0, 0);
}

// 32 TM rows a block.  FAR: a tile's rows lie beyond the reach of 32-bit offsets, and its transfers go by pointers.
template <typename TO, int TM, int STAGES = 2, bool FAR = false>
__global__ __launch_bounds__(256, 2) void gemm_f32_pipelined_kernel(const float* __restrict__ A, int lda,
                                                                    const float* __restrict__ W, int ldw,
                                                                    TO* __restrict__ C, int ldc, int M, int N, int K,
                                                                    int tiles_m, int tiles_n) {
  constexpr int BM = 32 * TM, PER = (BM + TILE) / 32;  // transfers of 8 rows that a wave asks for a stage
  static_assert((STAGES - 1) * PER < 16, "a wait counts at most 15 transfers");
  __shared__ __attribute__((aligned(1024))) unsigned char stage[STAGES][(BM + TILE) * STAGE_K * 4];  // A's rows, then W's
  const int run = ((int)gridDim.x + 7) / 8, tile = (int)blockIdx.x % 8 * run + (int)blockIdx.x / 8;
  if (tile >= tiles_m * tiles_n) return;  // (the whole block: the grid is eight runs)
  const int m0 = tile % tiles_m * BM, n0 = tile / tiles_m * TILE;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4, wm = wave >> 1, wn = wave & 1;

  // a wave's transfers of a stage: 8 rows each, lane l the piece at place l % 8 of row l / 8
  using Offset = std::conditional_t<FAR, long long, int>;
  Offset from[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int row = (wave * PER + j) * 8 + (lane >> 3), piece = (lane & 7) ^ (row >> 1 & 7);
    from[j] = (row < BM ? min(row, M - 1 - m0) * (Offset)lda : min(row - BM, N - 1 - n0) * (Offset)ldw) * 4 + piece * 16;
  }
  auto ask = [&](int j, int s, int k0) {  // (from stage K on nothing is in range)
    const float* base = (wave * PER + j) * 8 < BM ? A + (long long)m0 * lda : W + (long long)n0 * ldw;
    if constexpr (FAR)  // (there the last stage comes again, to where nothing reads it)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)((const char*)(base + min(k0, K - STAGE_K)) + from[j]),
                                       (__attribute__((address_space(3))) void*)(stage[s] + (wave * PER + j) * 1024), 16, 0, 0);
    else piece_to_lds(base, k0 < K ? 0x7fffffff : 0, from[j], k0 * 4, stage[s] + (wave * PER + j) * 1024);
  };
  f32x4 total[TM][4], chunk[TM][4];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) total[i][j] = chunk[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const int swizzle = r16 >> 1;  // (tiles of 16 rows start at whole periods of it)

  f32x4 frag[2][PER];  // the fragments of a stage's two slabs: A's TM, then W's four
  auto fetch = [&](int j, int sl, int s) {
    const int at = ((sl * 4 + g) ^ swizzle) * 16;
    frag[sl][j] = j < TM ? *(const f32x4*)(stage[s] + (wm * 16 * TM + r16) * 128 + at + j * 2048)
                         : *(const f32x4*)(stage[s] + (BM + wn * 64 + r16) * 128 + at + (j - TM) * 2048);
  };
  // a slab's products, with `ops` accesses dealt out among them
  constexpr std::integral_constant<int, PER> reads;
  constexpr std::integral_constant<int, 2 * PER> both;
  auto multiply = [&](int sl, auto ops, auto&& op) {
#pragma unroll
    for (int q = 0; q < 4 * TM; ++q) {
#pragma unroll
      for (int n = q * ops / (4 * TM); n < (q + 1) * ops / (4 * TM); ++n) op(n);
      __builtin_amdgcn_sched_barrier(0);
      const int i = q % TM, j4 = q / TM;
#pragma unroll
      for (int j = 0; j < 4; ++j) chunk[i][j] = mfma4(frag[sl][i][j4], frag[sl][TM + j][j4], chunk[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto reads_done = [&]() {
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
  };

#pragma unroll
  for (int s = 0; s < STAGES; ++s)
#pragma unroll
    for (int j = 0; j < PER; ++j) ask(j, s, s * STAGE_K);
  __builtin_amdgcn_s_waitcnt(0x0F70 | (STAGES - 1) * PER);  // vmcnt: this wave's transfers of the first stage have landed,
  asm volatile("s_barrier" ::: "memory");  // and everyone's
#pragma unroll
  for (int j = 0; j < PER; ++j) fetch(j, 0, 0);
  for (int k0 = 0, s = 0; k0 < K; k0 += STAGE_K) {
    const int next = s + 1 < STAGES ? s + 1 : 0;
    reads_done();
    multiply(0, reads, [&](int n) { fetch(n, 1, s); });
    reads_done();
    __builtin_amdgcn_s_waitcnt(0x0F70 | (STAGES - 2) * PER);  // vmcnt: this wave's transfers of the next stage have landed,
    asm volatile("s_barrier" ::: "memory");  // and everyone's; and everyone is done reading this one
    multiply(1, both, [&](int n) {  // (behind the last stage the reads are of no use)
      if (n % 2 == 0) ask(n / 2, s, k0 + STAGES * STAGE_K);
      else fetch(n / 2, 0, next);
    });
    s = next;
    if ((k0 + STAGE_K) % CHUNK == 0 || k0 + STAGE_K >= K) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          total[i][j] += chunk[i][j];
          chunk[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
        }
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // (no transfer may land behind the workgroup's end)
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + (wn * 4 + j) * 16 + r16;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + (wm * TM + i) * 16 + 4 * g + e;
        if (m < M && n < N) C[(long long)m * ldc + n] = from_f32<TO>(total[i][j][e]);
      }
    }
}

// ---- at most 64 rows: the weights streamed from memory ---------------------------------------------------
// Four k of a row as float32: 16 bytes of float32 or 8 bytes of bfloat16.
__device__ inline f32x4 load4(const float* p) { return *(const f32x4*)p; }
__device__ inline f32x4 load4(const bf16_t* p) {
  const uint2 v = *(const uint2*)p;
  f32x4 r;
  r.x = __uint_as_float(v.x << 16);
  r.y = __uint_as_float(v.x & 0xffff0000u);
  r.z = __uint_as_float(v.y << 16);
  r.w = __uint_as_float(v.y & 0xffff0000u);
  return r;
}

// Up to 16 MT rows: MT row tiles share a wave's weights.  NW waves a block take chunks in turn.  The weights of a whole
// chunk are asked for together (16 loads of 1 KiB a wave), x four slabs at a time: within 128 registers a compute unit
// holds 16 waves, as two blocks of 8, of which one streams while the other's meet, or as one of 16 where there are no
// more blocks than compute units.
template <typename T, typename TO, int MT, int ROWS_WAVES>
__global__ __launch_bounds__(ROWS_WAVES * 64, MT <= 2 ? 4 : 2) void gemm_f32_rows_kernel(const T* __restrict__ X, int ldx,
                                                                                        const T* __restrict__ W, int ldw,
                                                                                        TO* __restrict__ C, int ldc, int M, int N,
                                                                                        int K) {
  __shared__ float sums[2][ROWS_WAVES][MT * 256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c16 = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const T* wp = W + (long long)min(n0 + c16, N - 1) * ldw + 4 * g;
  const T* xp[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) xp[i] = X + (long long)min(16 * i + c16, M - 1) * ldx + 4 * g;
  const int chunks = (K + CHUNK - 1) / CHUNK;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 total = zero;  // of row tile `wave`
  for (int round = 0; round * ROWS_WAVES < chunks; ++round) {
    const int ch = round * ROWS_WAVES + wave;
    f32x4 sum[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) sum[i] = zero;
    if (ch < chunks) {
      const int k_begin = ch * CHUNK;
      f32x4 wv[CHUNK / SLAB];
#pragma unroll
      for (int s = 0; s < CHUNK / SLAB; ++s) {
        const int k = k_begin + s * SLAB;  // this lane's four k: k + 4 g .. k + 4 g + 3 (K is a multiple of 4)
        wv[s] = k + 4 * g < K ? load4(wp + k) : zero;
      }
#pragma unroll
      for (int s0 = 0; s0 < CHUNK / SLAB; s0 += 4) {
        f32x4 xv[MT][4];
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            const int k = k_begin + (s0 + s) * SLAB;
            xv[i][s] = k + 4 * g < K ? load4(xp[i] + k) : zero;
          }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int j4 = 0; j4 < 4; ++j4)
#pragma unroll
            for (int i = 0; i < MT; ++i) sum[i] = mfma4(xv[i][s][j4], wv[s0 + s][j4], sum[i]);
      }
    }
    // the round's chunks join the running sum in ascending order (wave i adds row tile i)
    float(*buf)[MT * 256] = sums[round & 1];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) buf[wave][i * 256 + e * 64 + lane] = sum[i][e];
    __syncthreads();  // (two buffers: the one written two rounds ago has been read by then)
    const int n_round = min(ROWS_WAVES, chunks - round * ROWS_WAVES);
    if (wave < MT)
      for (int w = 0; w < n_round; ++w)
#pragma unroll
        for (int e = 0; e < 4; ++e) total[e] += buf[w][wave * 256 + e * 64 + lane];
  }
  if (wave < MT) {
    const int n = n0 + c16;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int m = 16 * wave + 4 * g + e;
      if (m < M && n < N) C[(long long)m * ldc + n] = from_f32<TO>(total[e]);
    }
  }
}

// At most 16 rows of float32 with K in 32s: the same chunks, waves and sums, the weights through LDS.  In the kernel above a load is 64
// bytes from each of 16 rows, half lines, and a wave waits for all of a chunk before it asks for the next.  Here a wave's transfers into
// LDS read 128 bytes of 8 rows, neighbouring lanes a row, marked as a stream (nt), into four slots of its own of 16 rows by 32 k: a
// slot is waited for, read, and asked for anew, with its x, across chunks.  Microseconds before and now, the same bits: 4 rows of 28 672 x
// 4 096 108 -> 80 (5.9 TB/s), of 125 000 x 4 096 412 -> 320 (6.4), of 4 096 x 14 336 54 -> 39, of 4 096 x 4 096 19.1 -> 15.9, of 6 144 x 4 096
// 32 -> 23, of 2 048 x 2 048 10.6 -> 7.2; 16 rows of 28 672 x 4 096 125 -> 92; 1 row of 30 x 512 4.8 -> 4.5.
constexpr int NOWHERE = (int)0x80000000u;  // an offset beyond every buffer: nothing is read, zeros come

template <typename TO, int WAVES>
__global__ __launch_bounds__(WAVES * 64, 4) void gemm_f32_stream_kernel(const float* __restrict__ X, int ldx,
                                                                                        const float* __restrict__ W, int ldw,
                                                                                        TO* __restrict__ C, int ldc, int M, int N, int K) {
  constexpr int SLOTS = 4, PER = CHUNK / 32;  // slots of 32 k; of them in a chunk
  static_assert(PER % SLOTS == 0, "a chunk begins with the first slot");
  extern __shared__ __attribute__((aligned(1024))) unsigned char ring[];  // [WAVES][SLOTS][2048], then two rounds' sums
  float(*sums)[WAVES][256] = (float(*)[WAVES][256])(ring + WAVES * SLOTS * 2048);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int c16 = lane & 15, g = lane >> 4, n0 = blockIdx.x * 16;
  const int chunks = (K + CHUNK - 1) / CHUNK, slabs = K / 32;
  const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)X, 0, (int)(((long long)(M - 1) * ldx + K) * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t w_rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)(W + (long long)n0 * ldw), 0, (int)(((long long)(min(16, N - n0) - 1) * ldw + K) * 4), 0x00020000);
  const int x_off = c16 < M ? (c16 * ldx + 4 * g) * 4 : NOWHERE;
  int w_off[2];  // this lane in a transfer: row lane / 8, the chunk of four k that lies at position lane % 8
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int row = 8 * q + (lane >> 3);
    w_off[q] = n0 + row < N ? row * ldw * 4 + ((lane & 7) ^ (row >> 1)) * 16 : NOWHERE;
  }
  unsigned char* mine = ring + wave * (SLOTS * 2048);
  f32x4 xv[SLOTS][2];
  int ask_chunk = wave, ask_slab = 0;  // the next to ask for: slab `ask_slab` of chunk `ask_chunk`
  auto ask = [&](int slot) {
    const int at = (ask_chunk * PER + ask_slab) * 128;
#pragma unroll
    for (int q = 0; q < 2; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, (__attribute__((address_space(3))) void*)(mine + slot * 2048 + q * 1024), 16, w_off[q], at, 0, 2);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      xv[slot][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, x_off, at + h * 64, 0));
    if (++ask_slab == min(PER, slabs - ask_chunk * PER)) ask_slab = 0, ask_chunk += WAVES;
    __builtin_amdgcn_sched_barrier(0);  // (the waits count a slot's requests, x's among them: none may change its place with another slot's)
  };
  // this wave's slabs: whole chunks, but for the last of all
  const int my_chunks = wave < chunks ? (chunks - wave + WAVES - 1) / WAVES : 0;
  int left = my_chunks * PER;
  if (my_chunks > 0 && wave + (my_chunks - 1) * WAVES == chunks - 1) left -= chunks * PER - slabs;
#pragma unroll
  for (int i = 0; i < SLOTS; ++i)
    if (i < left) ask(i);
  int frag[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) frag[h] = c16 * 128 + (((4 * h + g) ^ (c16 >> 1)) & 7) * 16;

  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 total = zero, sum;
  // A chunk of n slabs.  FULL: more than the slots' worth comes behind it, so that every slot is asked for anew without a question and
  // the wait for x leaves what was asked for since flying.
  auto chunk = [&](int n, auto full) {
    constexpr bool FULL = decltype(full)::value;
    sum = zero;
#pragma unroll
    for (int s = 0; s < PER; ++s) {
      const int slot = s % SLOTS;
      if (FULL || s < n) {
        if (FULL || left > 3) __builtin_amdgcn_s_waitcnt(0x0F70 | 12);  // vmcnt: four a slot
        else if (left == 3) __builtin_amdgcn_s_waitcnt(0x0F70 | 8);
        else if (left == 2) __builtin_amdgcn_s_waitcnt(0x0F70 | 4);
        else __builtin_amdgcn_s_waitcnt(0x0F70);
        __builtin_amdgcn_sched_barrier(0);
        f32x4 b[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) b[h] = *(const f32x4*)(mine + slot * 2048 + frag[h]);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the slot has been read
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int j = 0; j < 4; ++j) sum = mfma4(xv[slot][h][j], b[h][j], sum);
        if (FULL || left > SLOTS) ask(slot);
        --left;
      }
    }
  };
  for (int round = 0; round * WAVES < chunks; ++round) {
    const int ch = round * WAVES + wave;
    if (left >= PER + SLOTS) chunk(PER, std::true_type());
    else if (ch < chunks) chunk(min(PER, slabs - ch * PER), std::false_type());
    else sum = zero;
    // the round's chunks join the running sum in ascending order
#pragma unroll
    for (int e = 0; e < 4; ++e) sums[round & 1][wave][e * 64 + lane] = sum[e];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (transfers fly on; of two buffers, the one written two rounds ago has been read)
    const int n_round = min(WAVES, chunks - round * WAVES);
    if (wave == 0)
      for (int w = 0; w < n_round; ++w)
#pragma unroll
        for (int e = 0; e < 4; ++e) total[e] += sums[round & 1][w][e * 64 + lane];
  }
  if (wave == 0) {
    const int n = n0 + c16;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int m = 4 * g + e;
      if (m < M && n < N) C[(long long)m * ldc + n] = from_f32<TO>(total[e]);
    }
  }
}

template <typename TO, int WAVES>
int launch_f32_stream(const void* x, const void* w, void* out, int M, int N, int K, int lda, int ldw, int ldc, hipStream_t stream) {
  constexpr int lds = WAVES * (4 * 2048 + 2 * 256 * 4);
  const auto kernel = gemm_f32_stream_kernel<TO, WAVES>;
  static bool configured = false;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
      lq_set_error("linear: cannot reserve %d bytes of LDS: %s", lds, hipGetErrorString(e));
      return -2;
    }
    configured = true;
  }
  kernel<<<lq_ceil_div(N, 16), WAVES * 64, lds, stream>>>((const float*)x, lda, (const float*)w, ldw, (TO*)out, ldc, M, N, K);
  LQ_CHECK_LAUNCH("linear(float32 stream)");
  return 0;
}

// Tiles of 32, 64, 96 or 128 rows by 128 columns: what a product takes goes by the tiles of the fullest compute unit, and a narrow
// tile fills the chip better while a wide one multiplies faster.  Microseconds for K 4 096: one tile a compute unit, and each of
// several (measured over 2 048 to 28 672 columns of K 2 048 to 14 336 at 65 to 1 200 rows, 98 products: the shape that this names is within
// 1.7 % of the best of the four, 0.07 % on average).  With 128 rows alone -> this: 100 rows of 4 096 x 14 336 831 -> 261,
// 333 of 6 144 x 4 096 241 -> 187, 600 of 4 096 x 14 336 832 -> 637, 433 of 28 672 x 4 096 934 -> 788.
float pipelined_us(int tm, int M, int tiles_n, int K) {
  constexpr float one[4] = {81.f, 135.f, 188.f, 244.f}, each[4] = {62.f, 119.f, 175.f, 233.f};
  const long long n = lq_ceil_div64((long long)lq_ceil_div(M, 32 * tm) * tiles_n, lq_compute_units());
  return (n <= 1 ? one[tm - 1] : 4.f + each[tm - 1] * n) * K / 4096.f;
}

template <typename T, typename TO>
int launch(const void* x, const void* w, void* out, int M, int N, int K, int lda, int ldw, int ldc, hipStream_t stream) {
  const int el = (int)sizeof(T);
  // rows of four k each, fetched as one piece: K, the strides and the addresses must allow it
  const bool pieces = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && ((uintptr_t)x % (4 * el)) == 0 &&
                      ((uintptr_t)w % (4 * el)) == 0;
  const bool tiles = sizeof(T) == 4 && pieces && K % STAGE_K == 0, far = (long long)(lda > ldw ? lda : ldw) * TILE * 4 >= (1ll << 31);
  // Few rows of a wide weight: pipelined tiles once their 128 columns fill enough of the chip, 7 sixteenths for 17 to 32 rows (17 rows by
  // the rows' kernel / here: 12 288 x 4 096 71 / 77 us, 14 336 x 4 096 90 / 78, 28 672 x 4 096 151 / 103; 32 rows of it 180 / 105)
  // and a quarter for 33 to 64 (33 rows of 4 096 x 4 096 45 / 75, 8 192 x 4 096 86 / 76, 14 336 x 4 096 158 / 79).
  const bool wide = tiles && M > 16 && 16 * lq_ceil_div(N, TILE) >= (M > 32 ? 4 : 7) * lq_compute_units();
  if (M <= 64 && pieces && !wide) {
    // Microseconds before (up to 16 rows: 8 waves, all of x at once; beyond: the tiled kernel) and now, float32: 4 rows of
    // 28 672 x 4 096 124 -> 109, of 128 256 x 4 096 507 -> 431, of 4 096 x 14 336 55 -> 50, of 4 096 x 4 096 23 -> 19; 17 rows of
    // 28 672 x 4 096 300 -> 160, 40 rows of 4 096 x 4 096 239 -> 46.
    const bool sixteen = M <= 32 && lq_ceil_div(N, 16) <= lq_compute_units() && K > 8 * CHUNK;
    if constexpr (sizeof(T) == 4)
      if (M <= 16 && K % 32 == 0 && (long long)ldw * 64 < (1ll << 31) && (long long)lda * 64 < (1ll << 31))
        return sixteen ? launch_f32_stream<TO, 16>(x, w, out, M, N, K, lda, ldw, ldc, stream)
                       : launch_f32_stream<TO, 8>(x, w, out, M, N, K, lda, ldw, ldc, stream);
    const auto kernel = M > 32 ? gemm_f32_rows_kernel<T, TO, 4, 8>
                        : M > 16 ? (sixteen ? gemm_f32_rows_kernel<T, TO, 2, 16> : gemm_f32_rows_kernel<T, TO, 2, 8>)
                                 : (sixteen ? gemm_f32_rows_kernel<T, TO, 1, 16> : gemm_f32_rows_kernel<T, TO, 1, 8>);
    kernel<<<lq_ceil_div(N, 16), sixteen ? 1024 : 512, 0, stream>>>((const T*)x, lda, (const T*)w, ldw, (TO*)out, ldc, M, N, K);
    LQ_CHECK_LAUNCH("linear(float32 rows)");
    return 0;
  }
  if constexpr (sizeof(T) == 4) {
    if (wide || (tiles && M > 64 && N > 64)) {
      const int tiles_n = lq_ceil_div(N, TILE);
      LQ_REQUIRE((long long)lq_ceil_div(M, 32) * tiles_n < (1ll << 30), "linear: too many tiles");
      int tm = 4;
      for (int t = 3; t >= 1; --t)
        if (pipelined_us(t, M, tiles_n, K) < pipelined_us(tm, M, tiles_n, K)) tm = t;
      const long long blocks = (long long)lq_ceil_div(M, 32 * tm) * tiles_n;
      const auto kernel = far ? (tm == 1   ? gemm_f32_pipelined_kernel<TO, 1, 2, true>
                                 : tm == 2 ? gemm_f32_pipelined_kernel<TO, 2, 2, true>
                                 : tm == 3 ? gemm_f32_pipelined_kernel<TO, 3, 2, true>
                                           : gemm_f32_pipelined_kernel<TO, 4, 2, true>)
                          : tm == 1 ? (blocks <= lq_compute_units() ? gemm_f32_pipelined_kernel<TO, 1, 3> : gemm_f32_pipelined_kernel<TO, 1>)
                          : tm == 2 ? gemm_f32_pipelined_kernel<TO, 2>
                          : tm == 3 ? gemm_f32_pipelined_kernel<TO, 3>
                                    : gemm_f32_pipelined_kernel<TO, 4>;
      kernel<<<(int)((blocks + 7) / 8 * 8), 256, 0, stream>>>((const float*)x, lda, (const float*)w, ldw, (TO*)out, ldc, M, N, K,
                                                            (int)(blocks / tiles_n), tiles_n);
      LQ_CHECK_LAUNCH("linear(float32 pipelined)");
      return 0;
    }
  }
  if (M > 64 && N > 64) {
    dim3 grid(lq_ceil_div(N, 128), lq_ceil_div(M, 128));
    LQ_REQUIRE(grid.y <= 65535, "linear: %d rows are too many for one launch", M);
    gemm_f32_tiled_kernel<T, TO, 4, 4><<<grid, 256, 0, stream>>>((const T*)x, lda, (const T*)w, ldw, (TO*)out, ldc, M, N, K);
  } else {
    dim3 grid(lq_ceil_div(N, 64), lq_ceil_div(M, 64));
    LQ_REQUIRE(grid.y <= 65535, "linear: %d rows are too many for one launch", M);
    gemm_f32_tiled_kernel<T, TO, 2, 2><<<grid, 256, 0, stream>>>((const T*)x, lda, (const T*)w, ldw, (TO*)out, ldc, M, N, K);
  }
  LQ_CHECK_LAUNCH("linear(float32 tiled)");
  return 0;
}

}  // namespace

int lq_gemm_generic(const void* x, const void* w, void* out, int in_dtype, int out_dtype, int M,
                    int N, int K, int lda, int ldw, int ldc, hipStream_t stream) {
  if (in_dtype == LQ_F32 && out_dtype == LQ_F32) return launch<float, float>(x, w, out, M, N, K, lda, ldw, ldc, stream);
  if (in_dtype == LQ_BF16 && out_dtype == LQ_BF16) return launch<bf16_t, bf16_t>(x, w, out, M, N, K, lda, ldw, ldc, stream);
  if (in_dtype == LQ_BF16 && out_dtype == LQ_F32) return launch<bf16_t, float>(x, w, out, M, N, K, lda, ldw, ldc, stream);
  if (in_dtype == LQ_F32 && out_dtype == LQ_BF16) return launch<float, bf16_t>(x, w, out, M, N, K, lda, ldw, ldc, stream);
  lq_set_error("linear: unsupported dtypes %d -> %d", in_dtype, out_dtype);
  return -1;
}
