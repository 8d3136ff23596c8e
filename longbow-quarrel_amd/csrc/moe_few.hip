// A mixture of experts over at most 16 rows (decoding steps, the shortest prompts): two launches that read the weights of the
// experts that some row chose and no others.
//
// Such a step is bound by the bytes of its weights.  Every row used to go through all experts' columns, the activations of the
// unchosen ones set to zero by a launch between the products: one row that chooses 2 of 8 experts read four times what it needs,
// 8 rows that choose at random 11 % more.  Here every wavefront finds the chosen experts from the routing table itself (a load of
// a column of it for each lane, asked for beside the first rows of x), and the columns, then the k, of these experts alone are
// dealt out.
//
// Microseconds for a mixture's two products and the activation, every row through all experts -> this; 8 experts of 3 584 and width
// 2 048, two of them a row: 1 row 77 -> 21, 4 rows (7 experts chosen) 76 -> 62, 8 rows 80 -> 66, 16 rows 152 -> 76; of 7 168 and
// width 4 096: 1 row 239 -> 70, 8 rows 248 -> 225, 16 rows 370 -> 272; of 1 792 and width 1 024: 33 -> 12, 38 -> 22, 44 -> 27.  The
// products stream their weights at 5.7 to 6 TB/s from 4 rows on (the second at 4.0 to 4.8 when these times were taken).
//
// What a row's result is made of does not depend on the other rows' choices: an expert's columns are sums over the same shares
// of K whichever block takes them, a wavefront of the second product takes chunk i of the whole matrix's k where i % 16 is its
// number, and a chunk of an expert that only other rows chose adds zeros.
//
//   v_mfma_f32_16x16x32_bf16: lane (c = l % 16, g = l / 16) gives A[c][8 g .. + 8] and B[c][the same k] and receives
//   D[4 g + e][c].  A is x (rows beyond the last are whatever lies there, and nothing is kept of them), B 16 rows of the weight.
#include "device_math.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int KW = 16, THREADS = KW * 64;  // wavefronts of a workgroup: they share K
constexpr int ROWS = 16, EXPERTS = 64;

__device__ inline f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// A weight is read once a launch, in whole lines through LDS, and marked as a stream (nt), so that the caches keep the activations, the
// code and what the products around these read instead: 33 tokens of eight sequences of Vupelorn 40.7 -> 39.7 ms, 17 of Sofinex 24.8 -> 24.2.

struct Experts {
  const float* route;  // [rows][n]: an expert's weight, or -1
  int rows, n;
  int ff;      // columns of an expert
  int shared;  // columns of one more expert behind them that every row uses (0: none)
};

// The experts that some row chose, a bit each; the same in every lane.
__device__ inline unsigned long long chosen_experts(const Experts& ex) {
  const int lane = threadIdx.x & 63;
  float top = -1.f;
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
    top = fmaxf(top, ex.route[min(r, ex.rows - 1) * ex.n + min(lane, ex.n - 1)]);
  const unsigned long long bits = __ballot(lane < ex.n && top >= 0.f);
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)bits), hi = __builtin_amdgcn_readfirstlane((unsigned)(bits >> 32));
  return ((unsigned long long)hi << 32) | lo;
}

__device__ inline int nth_bit(unsigned long long bits, int n) {
  for (int i = 0; i < n; ++i) bits &= bits - 1;
  return __ffsll(bits) - 1;
}

// ---- the first product and the activation ---------------------------------------------------------------------------------
enum { UNIT_CLAMPED_SWISH = 0, UNIT_SILU = 1, UNIT_RELU2 = 2 };

struct FirstArgs {
  Experts ex;
  const float* shared_gate;  // [rows], `ld_gate` apart: the logit of a gate on the shared expert, or null
  int ld_gate;
  int unit, on_input;        // on_input: an expert's weight multiplies what it reads
  float limit;
};

// act[row][column] of every chosen expert's columns and the shared one's (others are left as they are), bfloat16; W's rows are
// expert by expert the gate's ff and the up matrix's ff (`GATED`), or the up matrix's alone.
// A unit is a tile of 16 weight rows: 16 columns of an expert, or with a gate 8, their gate rows and their up rows.  The units
// are dealt out evenly over the workgroups, the 16 wavefronts of which own a share of K each and keep their rows of x in
// registers.  The weights come through LDS as in the second product: a wavefront has three slots of its own, 16 rows of 64 k,
// filled by two transfers of whole lines; a slot is waited for, read, and asked for anew, across tiles and units, so that two
// and more are always on their way (64 KiB a compute unit).  After every two tiles the wavefronts' partial sums meet in LDS,
// where eight of them, in turn, finish a fourth of a unit each while the rest go on: the barrier behind lies ahead of the next
// two tiles' sums.
// What bounds it: the memory, and the round trip to the routing table ahead of the first weight.  8 rows that choose 7 of 8 experts of
// 3 584, width 2 048 (205 MB) 35.8 us, 5.7 TB/s; with units of 16 columns of a gated expert, 6 or 7 a workgroup instead of 12 or
// 13, 36.4; with fragments loaded into registers, half lines of 16 rows, two tiles ahead, and all wavefronts waiting for the end of
// every eight tiles, 40.9.
// SLABS: 64s of k that a wavefront owns at most.
constexpr int SLOTS1 = 3, SLOT = 2048;

__device__ __forceinline__ void lds_meet() { asm volatile("s_waitcnt lgkmcnt(0)\ns_barrier" ::: "memory"); }  // (transfers go on)

template <int SLABS, bool GATED>
__global__ __launch_bounds__(THREADS) void moe_few_first_kernel(const bf16_t* __restrict__ x, int ldx, const bf16_t* __restrict__ W,
                                                                int ldw, int packed, bf16_t* __restrict__ act, int ldo, int K,
                                                                int slabs_per_wave, FirstArgs a) {
  constexpr int PARTS = GATED ? 2 : 1, COLS = 16 / PARTS, TILES = 2;  // columns a unit; units between two meetings
  extern __shared__ __attribute__((aligned(1024))) unsigned char ring[];  // [KW][SLOTS1][SLOT]
  __shared__ float red[TILES][KW][256], route_sh[ROWS * EXPERTS], gate_sh[ROWS];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, c16 = lane & 15;
  const Experts& ex = a.ex;

  const int s0 = wave * slabs_per_wave, slabs = max(0, min(K / 64, s0 + slabs_per_wave) - s0);
  const u32x4 zero = {0u, 0u, 0u, 0u};
  u32x4 xv[SLABS][2];
#pragma unroll
  for (int s = 0; s < SLABS; ++s)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      xv[s][h] = s < slabs ? *(const u32x4*)(x + (long long)min(c16, ex.rows - 1) * ldx + (s0 + s) * 64 + 32 * h + 8 * g) : zero;
  if (tid < ex.rows * ex.n) route_sh[tid] = ex.route[tid];  // (rows * experts <= 1024 = the threads)
  if (a.shared_gate != nullptr && tid < ex.rows) gate_sh[tid] = sigmoid_f(a.shared_gate[(long long)tid * a.ld_gate]);

  const unsigned long long bits = chosen_experts(ex);
  const int per = ex.ff / COLS, of_experts = __popcll(bits) * per;
  const long long units = of_experts + ex.shared / COLS;
  const int u0 = (int)(units * blockIdx.x / gridDim.x), u1 = (int)(units * (blockIdx.x + 1) / gridDim.x), tiles = u1 - u0;
  if (tiles == 0) return;  // (the whole workgroup)

  // a unit's first row of W, the distance to its second eight rows, and its first column of act
  auto place = [&](int u, int& row, int& apart, int& col) {
    if (u < of_experts) {
      const int e = nth_bit(bits, u / per), j = u % per * COLS;
      row = e * PARTS * ex.ff + j, apart = ex.ff, col = e * ex.ff + j;
    } else {
      const int j = (u - of_experts) * COLS;
      row = ex.n * PARTS * ex.ff + j, apart = ex.shared, col = ex.n * ex.ff + j;
    }
    if constexpr (!GATED) apart = 8;
  };
  const bf16_t* lane_at[2];  // this lane in a transfer of 8 rows: row lane / 8, the chunk that lies at position lane % 8
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int row = lane >> 3, chunk = (lane & 7) ^ (4 * q + (row >> 1));
    lane_at[q] = W + (packed ? row * 64 + (long long)s0 * 512 : (long long)row * ldw + s0 * 64) + chunk * 8;
  }
  unsigned char* mine = ring + wave * (SLOTS1 * SLOT);
  int ask_tile = 0, ask_slab = 0;
  long long ask_from = 0, ask_apart = 0;  // where the tile that is asked for begins, and its second eight rows behind that
  auto ask = [&](int slot) {
    if (ask_slab == 0) {
      int row, apart, col;
      place(u0 + ask_tile, row, apart, col);
      ask_from = (long long)__builtin_amdgcn_readfirstlane(row) * ldw, ask_apart = (long long)apart * ldw;
    }
    const long long from = ask_from + ask_slab * (packed ? 512 : 64);
#pragma unroll
    for (int q = 0; q < 2; ++q)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(lane_at[q] + from + q * ask_apart),
                                       (__attribute__((address_space(3))) void*)(mine + slot * SLOT + q * 1024), 16, 0, 2);
    if (++ask_slab == slabs) ask_slab = 0, ++ask_tile;
  };
  // a unit's values of four rows: the wavefronts' shares in their order, and the activation
  auto finish = [&](int u, int e, int t) {
    int row, apart, col;
    place(u, row, apart, col);
    float s[2] = {0.f, 0.f};
#pragma unroll
    for (int w = 0; w < KW; ++w) s[0] += red[t][w][e * 64 + lane];
    if constexpr (GATED) s[1] = dpp_swap<0x128>(s[0]);  // (the up row's, eight lanes on)
    if (c16 >= COLS) return;
    const int r = 4 * g + e;
    if (r >= ex.rows) return;
    float y = 0.f;
    if (u >= of_experts) {  // the shared expert
      if constexpr (GATED) y = silu_f(s[0]) * (a.shared_gate != nullptr ? s[1] * gate_sh[r] : s[1]);
      else y = activate(s[0], ACT_RELU2);
    } else {
      const float w = route_sh[r * ex.n + col / ex.ff];
      if (w >= 0.f) {
        if constexpr (!GATED) {
          y = activate(s[0], ACT_RELU2) * w;
        } else {
          const float in = a.on_input ? w : 1.f;
          float gate = s[0] * in, up = s[1] * in;
          if (a.unit == UNIT_SILU) {
            y = silu_f(gate) * up;
          } else {
            gate = fminf(gate, a.limit), up = fminf(fmaxf(up, -a.limit), a.limit);
            y = gate / (1.f + expf(-1.702f * gate)) * (up + 1.f);
          }
          if (!a.on_input) y *= w;
        }
      }
    }
    act[(long long)r * ldo + col + c16] = f32_to_bf16(y);
  };

  int left = slabs * tiles, slot = 0;  // slots' worth of weights that are not read yet
#pragma unroll
  for (int i = 0; i < SLOTS1; ++i)
    if (i < left) ask(i);
  int frag[2];  // this lane's 16 bytes of a slot's 32-k halves
#pragma unroll
  for (int h = 0; h < 2; ++h) frag[h] = c16 * 128 + (((4 * h + g) ^ (c16 >> 1)) & 7) * 16;
  for (int b0 = 0; b0 < tiles; b0 += TILES) {
    f32x4 acc[TILES];
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
      acc[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
      if (b0 + i < tiles)
#pragma unroll
        for (int s = 0; s < SLABS; ++s)
          if (s < slabs) {
            // the oldest slot's transfers have landed: the two of each slot asked for after it may still fly (what a unit's end stored
            // since makes the wait longer, never shorter)
            if (left >= SLOTS1) __builtin_amdgcn_s_waitcnt(0x0F70 | 2 * (SLOTS1 - 1));
            else if (left == 2) __builtin_amdgcn_s_waitcnt(0x0F72);
            else __builtin_amdgcn_s_waitcnt(0x0F70);
            __builtin_amdgcn_sched_barrier(0);
            u32x4 wv[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) wv[h] = *(const u32x4*)(mine + slot * SLOT + frag[h]);
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the slot has been read
            __builtin_amdgcn_sched_barrier(0);
            if (left > SLOTS1) ask(slot);
            --left;
            slot = slot == SLOTS1 - 1 ? 0 : slot + 1;
#pragma unroll
            for (int h = 0; h < 2; ++h) acc[i] = mfma(xv[s][h], wv[h], acc[i]);
          }
    }
    if (b0 > 0) lds_meet();  // the sums before have been read
#pragma unroll
    for (int i = 0; i < TILES; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) red[i][wave][e * 64 + lane] = acc[i][e];
    lds_meet();
    const int j = (wave - 4 * b0) & (KW - 1);
    if (j < 4 * TILES && b0 + (j >> 2) < tiles) finish(u0 + b0 + (j >> 2), j & 3, j >> 2);
  }
}

// ---- the second product ---------------------------------------------------------------------------------------------------
// out[row][n] = sum over the chosen experts' columns (and the shared one's) of act[row][k] W[n][k], and, with identity experts,
// the row of h times the sum of their weights.  A workgroup takes 16 rows of W, and gridDim.y workgroups share their k (each leaves
// a piece of the result): rows of x are then read once for 16 rows of W, which at 8 rows are half of what a compute unit reads.
// The wavefronts take chunks of CHUNK k in turn.  The weights come through LDS: a wavefront has four slots of its own, 16 rows of
// 64 k (2 KiB), filled by two transfers of whole lines that are marked as a stream, with the slot's x beside them; a slot is waited for, read,
// and asked for anew, so that three are always on their way.  (Fragments loaded into registers, 64 bytes from each of 16 rows,
// three chunks ahead: 2 048 x 28 672 at 8 rows that choose 7 of 8 experts 23.6 us, this way 17.4, 6 TB/s.)
// At most 8 rows take chunks of 128 k and keep the sums of a chunk's halves of 64 k apart to the end (twice as many sums, half as long);
// more rows, and experts that are not in 128s, take chunks of 64.
// Position of 16-byte chunk c of a slot's row r: c ^ r / 2.  Behind a wavefront's last chunk transfers go on, out of the buffer's range,
// until all slots are done: a wait then always counts the same number of them; such a slot takes part in no sum.
constexpr int SLOTS = 4, NOWHERE = (int)0x80000000u;  // (NOWHERE: an offset beyond every buffer)

//
// FAR: rows of the activations or of W beyond the reach of 32-bit offsets.  Everything goes by pointers then, rows that there are not
// by those of the last one, and a slot is waited for with all that was asked for: nothing is counted.
template <int CHUNK, bool FAR>
__global__ __launch_bounds__(THREADS) void moe_few_second_kernel(const bf16_t* __restrict__ act, int lda, const bf16_t* __restrict__ W,
                                                                 int ldw, int packed, float* __restrict__ out, int ldo, long long piece,
                                                                 int N, Experts ex, const bf16_t* __restrict__ h, int ldh,
                                                                 const float* __restrict__ passed, int n_passed) {
  constexpr int SUMS = CHUNK / 64;
  static_assert(SLOTS % SUMS == 0, "a slot's part of its chunk is the slot's number modulo the parts");
  extern __shared__ __attribute__((aligned(1024))) unsigned char ring[];  // [KW][SLOTS][SLOT]; a wavefront's sums at its part's start
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, c16 = lane & 15;
  const int n0 = blockIdx.x * 16, rows = min(16, N - n0);
  const __amdgpu_buffer_rsrc_t w_rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)(W + (long long)n0 * ldw), 0, FAR ? 0 : rows * ldw * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t x_rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)act, 0, FAR ? 0 : ((ex.rows - 1) * lda + ex.n * ex.ff + ex.shared) * 2, 0x00020000);
  int w_off[2];  // this lane in a transfer: row lane / 8, the chunk that lies at position lane % 8
  const bf16_t* w_ptr[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int row = 8 * q + (lane >> 3), chunk = (lane & 7) ^ (row >> 1);
    w_off[q] = row >= rows ? NOWHERE : (packed ? q * 16 * ldw + (lane >> 3) * 128 : row * ldw * 2) + chunk * 16;
    const int n = n0 + min(row, rows - 1);
    w_ptr[q] = W + (packed ? (long long)(n >> 3) * 8 * ldw + (n & 7) * 64 : (long long)n * ldw) + chunk * 8;
  }
  const int x_off = c16 < ex.rows ? c16 * lda * 2 + g * 16 : NOWHERE;
  const bf16_t* x_ptr = act + (long long)min(c16, ex.rows - 1) * lda + g * 8;
  unsigned long long bits = chosen_experts(ex);

  // this wavefront's chunks of the expert that it is at: `left` more of them, the next at k
  const int chunks = ex.ff / CHUNK, turns = KW * gridDim.y, turn = blockIdx.y * KW + wave;  // (turns: a power of two)
  int k = 0, left = 0, part = 0;
  bool shared = ex.shared > 0;
  auto next = [&]() -> int {  // the next 64 k's first, or -1
    if (part == 0)
      while (left == 0) {
        int first, n;
        if (bits != 0) {
          const int e = __ffsll(bits) - 1;
          bits &= bits - 1;
          first = e * chunks, n = chunks;
        } else if (shared) {
          shared = false;
          first = ex.n * chunks, n = ex.shared / CHUNK;
        } else {
          return -1;
        }
        const int skip = (turn - first) & (turns - 1);
        left = n > skip ? (n - skip + turns - 1) / turns : 0;
        k = (first + skip) * CHUNK;
      }
    const int at = k + part * 64;
    if (++part == CHUNK / 64) {
      part = 0;
      --left;
      k += turns * CHUNK;
    }
    return at;
  };
  unsigned char* mine = ring + wave * (SLOTS * SLOT);
  u32x4 xv[SLOTS][2];
  bool there[SLOTS];
  auto ask = [&](int slot) {
    const int at = next();
    there[slot] = at >= 0;
    if constexpr (FAR) {
      const long long from = max(at, 0);
#pragma unroll
      for (int q = 0; q < 2; ++q)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(w_ptr[q] + from * (packed ? 8 : 1)),
                                         (__attribute__((address_space(3))) void*)(mine + slot * SLOT + q * 1024), 16, 0, 0);
#pragma unroll
      for (int i = 0; i < 2; ++i) xv[slot][i] = *(const u32x4*)(x_ptr + from + 32 * i);
      return;
    }
#pragma unroll
    for (int q = 0; q < 2; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, (__attribute__((address_space(3))) void*)(mine + slot * SLOT + q * 1024), 16,
                                               at >= 0 ? w_off[q] : NOWHERE, at >= 0 ? at * (packed ? 16 : 2) : 0, 0, 2);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      xv[slot][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, at >= 0 ? x_off + 64 * i : NOWHERE, at >= 0 ? at * 2 : 0, 0));
    __builtin_amdgcn_sched_barrier(0);  // (the waits count a slot's requests: none may change its place with another slot's)
  };
#pragma unroll
  for (int d = 0; d < SLOTS; ++d) ask(d);
  int frag[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) frag[i] = c16 * 128 + (((4 * i + g) ^ (c16 >> 1)) & 7) * 16;
  f32x4 acc[SUMS];
#pragma unroll
  for (int j = 0; j < SUMS; ++j) acc[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto use = [&](int d) {  // (its transfers have landed)
    __builtin_amdgcn_sched_barrier(0);
    u32x4 wv[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) wv[i] = *(const u32x4*)(mine + d * SLOT + frag[i]);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the slot has been read
    __builtin_amdgcn_sched_barrier(0);
    if (there[d])
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[d % SUMS] = mfma(xv[d][i], wv[i], acc[d % SUMS]);
  };
  while (there[SLOTS - 1]) {  // (slots are filled in their order: the last one asked for stands for all)
#pragma unroll
    for (int d = 0; d < SLOTS; ++d) {
      __builtin_amdgcn_s_waitcnt(0x0F70 | (FAR ? 0 : 12));  // vmcnt: four a slot, three slots behind
      use(d);
      ask(d);
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);
#pragma unroll
  for (int d = 0; d < SLOTS; ++d) use(d);
  float* red = (float*)mine;
#pragma unroll
  for (int j = 0; j < SUMS; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) red[j * 256 + e * 64 + lane] = acc[j][e];
  // four wavefronts finish the entries of 16 columns: wavefront e those of acc[..][e]
  const int r = 4 * g + wave, n = n0 + c16;
  const bool ends = wave < 4 && r < ex.rows && n < N;
  float add = 0.f;
  if (ends && passed != nullptr && blockIdx.y == 0) {
    float w = 0.f;
    for (int i = 0; i < n_passed; ++i) w += fmaxf(passed[r * n_passed + i], 0.f);  // (-1: not chosen)
    if (w != 0.f) add = w * to_f32(h[(long long)r * ldh + n]);
  }
  __syncthreads();
  if (!ends) return;
  float s = 0.f;
#pragma unroll
  for (int w = 0; w < KW; ++w)
#pragma unroll
    for (int j = 0; j < SUMS; ++j) s += ((const float*)(ring + w * (SLOTS * SLOT)))[j * 256 + wave * 64 + lane];
  out[blockIdx.y * piece + (long long)r * ldo + n] = s + add;
}

int slabs_per_wave(int K) { return lq_ceil_div(K / 64, KW); }

template <int SLABS, bool GATED>
int launch_first(const bf16_t* x, int ldx, const bf16_t* w, int ldw, int packed, bf16_t* act, int ldo, int K, const FirstArgs& a, int grid,
                 hipStream_t stream) {
  const auto kernel = moe_few_first_kernel<SLABS, GATED>;
  constexpr int lds = KW * SLOTS1 * SLOT;
  static bool configured = false;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
      lq_set_error("moe_few: cannot reserve %d bytes of LDS: %s", lds, hipGetErrorString(e));
      return -2;
    }
    configured = true;
  }
  kernel<<<grid, THREADS, lds, stream>>>(x, ldx, w, ldw, packed, act, ldo, K, slabs_per_wave(K), a);
  LQ_CHECK_LAUNCH("moe_few(first product)");
  return 0;
}

}  // namespace

// Whether lq_moe_few_first and lq_moe_few_second take a mixture: at most 16 rows and 64 experts of `ff` columns, one more of
// `shared` (0: none), rows of `width` entries.
extern "C" int lq_moe_few_supported(int dtype, int rows, int experts, int ff, int shared, int width) {
  return dtype == LQ_BF16 && rows >= 1 && rows <= ROWS && experts >= 1 && experts <= EXPERTS && ff >= 64 && ff % 64 == 0 &&
         shared >= 0 && shared % 64 == 0 && width >= 512 && width % 64 == 0 && width <= KW * 8 * 32 &&
         2ll * experts * ff + 2ll * shared <= 0x7fffffff;
}

// act[row][e ff + c] (bfloat16) = the activation of expert e's column c for the experts that some row chose: the unit's value for
// rows that chose e, 0 for the others; columns of experts that no row chose are not written.  x [rows, width]; w [experts * parts
// * ff + parts * shared, width], parts 2 (gate rows, then up rows, of an expert) or 1 with unit 2, dense or packed
// (lq_pack_weight).  unit 0: y = g sigmoid(1.702 g) (u + 1) with g = min(gate, limit), u = clamp(up, -limit, limit);
// 1: silu(gate) up; 2: relu(up)^2.  The shared expert has weight one, times the sigmoid of shared_gate[row * ld_gate].
extern "C" int lq_moe_few_first(const void* x, int ldx, const void* w, int ldw, int w_packed, const float* route, void* act, int ldo,
                                int rows, int experts, int ff, int shared, int width, int unit, float limit, int on_input,
                                const float* shared_gate, int ld_gate, hipStream_t stream) {
  LQ_REQUIRE(lq_moe_few_supported(LQ_BF16, rows, experts, ff, shared, width), "moe_few: %d rows, %d experts of %d columns (shared %d), width %d",
             rows, experts, ff, shared, width);
  LQ_REQUIRE(x && w && route && act, "moe_few: null pointer");
  LQ_REQUIRE(unit >= UNIT_CLAMPED_SWISH && unit <= UNIT_RELU2 && (shared == 0 || unit != UNIT_CLAMPED_SWISH), "moe_few: unit %d", unit);
  LQ_REQUIRE(ldx >= width && ldw >= width && ldo >= experts * ff + shared, "moe_few: a row stride is smaller than its row");
  LQ_REQUIRE(ldx % 8 == 0 && ldw % 8 == 0 && ((uintptr_t)x | (uintptr_t)w) % 16 == 0 && (!w_packed || ldw == width),
             "moe_few: operands are not aligned");
  LQ_REQUIRE(shared_gate == nullptr || (shared > 0 && unit == UNIT_SILU && ld_gate >= 1), "moe_few: the shared expert's gate");
  const FirstArgs a = {{route, rows, experts, ff, shared}, shared_gate, ld_gate, unit, on_input, limit};
  const int gated = unit != UNIT_RELU2;
  const long long units = ((long long)experts * ff + shared) / (gated ? 8 : 16);
  const int grid = units < lq_compute_units() ? (int)units : lq_compute_units();
#define LQ_FIRST(SLABS, GATED) \
  launch_first<SLABS, GATED>((const bf16_t*)x, ldx, (const bf16_t*)w, ldw, w_packed, (bf16_t*)act, ldo, width, a, grid, stream)
  if (slabs_per_wave(width) <= 2) return gated ? LQ_FIRST(2, true) : LQ_FIRST(2, false);
  return gated ? LQ_FIRST(4, true) : LQ_FIRST(4, false);
#undef LQ_FIRST
}

// In how many pieces (1, 2 or 4) lq_moe_few_second likes to leave its result: with fewer workgroups of 16 columns than three
// quarters of the compute units, as many as fill them.
extern "C" int lq_moe_few_pieces(int width) {
  int pieces = 1;
  while (pieces < 4 && lq_ceil_div(width, 16) * pieces < 3 * lq_compute_units() / 4) pieces *= 2;
  return pieces;
}

// The sum of out's pieces [rows, width] (32-bit, piece_stride apart) = act . w^T over the columns that lq_moe_few_first wrote; w
// [width, experts * ff + shared], dense or packed.  With passed [rows, n_passed] (identity experts' weights, or -1) also the rows of
// h times their sums.
extern "C" int lq_moe_few_second(const void* act, int lda, const void* w, int ldw, int w_packed, const float* route, float* out, int ldo,
                                 int pieces, long long piece_stride, int rows, int experts, int ff, int shared, int width, const void* h,
                                 int ldh, const float* passed, int n_passed, hipStream_t stream) {
  LQ_REQUIRE(lq_moe_few_supported(LQ_BF16, rows, experts, ff, shared, width), "moe_few: %d rows, %d experts of %d columns (shared %d), width %d",
             rows, experts, ff, shared, width);
  LQ_REQUIRE(act && w && route && out, "moe_few: null pointer");
  LQ_REQUIRE(lda >= experts * ff + shared && ldw >= experts * ff + shared && ldo >= width, "moe_few: a row stride is smaller than its row");
  LQ_REQUIRE((pieces == 1 || pieces == 2 || pieces == 4) && (pieces == 1 || piece_stride >= (long long)rows * ldo), "moe_few: %d pieces", pieces);
  LQ_REQUIRE(lda % 8 == 0 && ldw % 8 == 0 && ((uintptr_t)act | (uintptr_t)w) % 16 == 0 && (!w_packed || (ldw % 64 == 0 && width % 8 == 0)),
             "moe_few: operands are not aligned");
  LQ_REQUIRE(passed == nullptr || (h != nullptr && ldh >= width && n_passed >= 1), "moe_few: identity experts come with the rows");
  const bool long_chunks = rows <= 8 && ff % 128 == 0 && shared % 128 == 0;
  const bool far = (long long)ldw * 32 >= (1ll << 31) || (long long)rows * lda * 2 >= (1ll << 31);
  const auto kernel = far ? (long_chunks ? moe_few_second_kernel<128, true> : moe_few_second_kernel<64, true>)
                          : (long_chunks ? moe_few_second_kernel<128, false> : moe_few_second_kernel<64, false>);
  constexpr int lds = KW * SLOTS * SLOT;
  static bool configured[2][2] = {};
  if (!configured[far][long_chunks]) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
      lq_set_error("moe_few: cannot reserve %d bytes of LDS: %s", lds, hipGetErrorString(e));
      return -2;
    }
    configured[far][long_chunks] = true;
  }
  kernel<<<dim3(lq_ceil_div(width, 16), pieces), THREADS, lds, stream>>>((const bf16_t*)act, lda, (const bf16_t*)w, ldw, w_packed, out, ldo,
                                                                         piece_stride, width, Experts{route, rows, experts, ff, shared},
                                                                         (const bf16_t*)h, ldh, passed, n_passed);
  LQ_CHECK_LAUNCH("moe_few(second product)");
  return 0;
}
