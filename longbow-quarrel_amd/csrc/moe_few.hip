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
// first product streams its weights at 5.0 to 6.3 TB/s from 4 rows on, the second at 6 (at 4.0 to 4.8 when these times were taken).
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

// A weight is read once a launch.  Packed ones are marked as a stream (nt), so that the caches keep the activations, the code and
// what the products around these read instead: 33 tokens of eight sequences of Vupelorn 40.7 -> 39.7 ms, 17 of Sofinex 24.8 -> 24.2 (the
// first product's mark alone 41.2 and 24.7, the second's 41.0 and 24.8).  A dense row's two halves of a line are asked for further
// apart, and marked they would come twice.
template <bool PACKED>
__device__ inline u32x4 load_weight(const bf16_t* p) {
  if constexpr (PACKED) return __builtin_nontemporal_load((const u32x4*)p);
  else return *(const u32x4*)p;
}

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
// A unit is 16 columns of an expert: a tile of 16 weight rows, with a gate two.  The units are dealt out evenly over the
// workgroups, the 16 wavefronts of which own a share of K each and keep their rows of x in registers; the weights of the tile
// after are asked for before a tile is multiplied, across the barriers at which up to 8 tiles' partial sums meet in LDS.
// XS: steps of 32 k that a wavefront owns at most.
template <int XS, bool GATED, bool PACKED>
__global__ __launch_bounds__(THREADS) void moe_few_first_kernel(const bf16_t* __restrict__ x, int ldx, const bf16_t* __restrict__ W,
                                                                int ldw, bf16_t* __restrict__ act, int ldo, int K, int ks_per_wave,
                                                                FirstArgs a) {
  constexpr int PARTS = GATED ? 2 : 1, TILES = 8, UNITS = TILES / PARTS;  // tiles and units between two barriers
  constexpr int GT = 8 / XS;                                             // tiles asked for together
  extern __shared__ __attribute__((aligned(16))) float red[];            // [TILES][KW][256]
  __shared__ float route_sh[ROWS * EXPERTS], gate_sh[ROWS];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, c16 = lane & 15;
  const Experts& ex = a.ex;

  const int k0 = wave * ks_per_wave * 32, k1 = min(K, k0 + ks_per_wave * 32);
  const u32x4 zero = {0u, 0u, 0u, 0u};
  u32x4 xv[XS];
#pragma unroll
  for (int s = 0; s < XS; ++s) {
    const int k = k0 + 32 * s + 8 * g;
    xv[s] = k < k1 ? *(const u32x4*)(x + (long long)min(c16, ex.rows - 1) * ldx + k) : zero;
  }
  if (tid < ex.rows * ex.n) route_sh[tid] = ex.route[tid];  // (rows * experts <= 1024 = the threads)
  if (a.shared_gate != nullptr && tid < ex.rows) gate_sh[tid] = sigmoid_f(a.shared_gate[(long long)tid * a.ld_gate]);

  const unsigned long long bits = chosen_experts(ex);
  const int per = ex.ff / 16, of_experts = __popcll(bits) * per;
  const long long units = of_experts + ex.shared / 16;
  const int u0 = (int)(units * blockIdx.x / gridDim.x), u1 = (int)(units * (blockIdx.x + 1) / gridDim.x);
  const int tiles = (u1 - u0) * PARTS;
  if (tiles == 0) return;  // (the whole workgroup)

  // a unit's first row of W (of its first part), the distance to its second part's, and its first column of act
  auto place = [&](int u, int& row, int& apart, int& col) {
    if (u < of_experts) {
      const int e = nth_bit(bits, u / per), j = u % per * 16;
      row = e * PARTS * ex.ff + j, apart = ex.ff, col = e * ex.ff + j;
    } else {
      const int j = (u - of_experts) * 16;
      row = ex.n * PARTS * ex.ff + j, apart = ex.shared, col = ex.n * ex.ff + j;
    }
  };
  u32x4 wv[2][GT][XS];
  auto ask = [&](int buf, int t0) {
#pragma unroll
    for (int i = 0; i < GT; ++i) {
      int row, apart, col;
      const int t = min(t0 + i, tiles - 1);
      place(u0 + t / PARTS, row, apart, col);
      const int n = row + (t % PARTS) * apart + c16;
      const bf16_t* wp = PACKED ? W + (long long)(n >> 3) * 8 * ldw + (n & 7) * 64 + (long long)(k0 >> 6) * 512 + g * 8
                                : W + (long long)n * ldw + k0 + g * 8;
#pragma unroll
      for (int s = 0; s < XS; ++s)
        wv[buf][i][s] = k0 + 32 * s + 8 * g < k1 ? load_weight<PACKED>(wp + (PACKED ? (s >> 1) * 512 + (s & 1) * 32 : s * 32)) : zero;
    }
  };
  auto multiply = [&](int buf, int t0) {  // tiles t0 .. of the batch that starts at tile t0 / TILES * TILES
#pragma unroll
    for (int i = 0; i < GT; ++i) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < XS; ++s) acc = mfma(xv[s], wv[buf][i][s], acc);
      float* to = red + ((t0 + i) % TILES * KW + wave) * 256 + lane;
#pragma unroll
      for (int e = 0; e < 4; ++e) to[e * 64] = acc[e];
    }
  };
  // a unit's values of four rows and 16 columns: the wavefronts' shares in their order, and the activation
  auto finish = [&](int u, int e, int t) {
    int row, apart, col;
    place(u, row, apart, col);
    float s[PARTS];
#pragma unroll
    for (int p = 0; p < PARTS; ++p) {
      s[p] = 0.f;
#pragma unroll
      for (int w = 0; w < KW; ++w) s[p] += red[((t + p) * KW + w) * 256 + e * 64 + lane];
    }
    const int r = 4 * g + e;
    if (r >= ex.rows) return;
    float y = 0.f;
    if (u >= of_experts) {  // the shared expert
      if constexpr (GATED) y = silu_f(s[0]) * (a.shared_gate != nullptr ? s[PARTS - 1] * gate_sh[r] : s[PARTS - 1]);
      else y = activate(s[0], ACT_RELU2);
    } else {
      const float w = route_sh[r * ex.n + col / ex.ff];
      if (w >= 0.f) {
        if constexpr (!GATED) {
          y = activate(s[0], ACT_RELU2) * w;
        } else {
          const float in = a.on_input ? w : 1.f;
          float gate = s[0] * in, up = s[PARTS - 1] * in;
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

  ask(0, 0);
  for (int b0 = 0; b0 < tiles; b0 += TILES) {  // a batch; TILES / GT is even, so a batch starts with buffer 0
#pragma unroll
    for (int i = 0; i < TILES / GT; ++i) {
      const int t = b0 + i * GT;
      if (t < tiles) {
        if (t + GT < tiles) ask((i + 1) & 1, t + GT);
        __builtin_amdgcn_sched_barrier(0);  // (the next tiles' weights are asked for ahead of these products)
        multiply(i & 1, t);
      }
    }
    __syncthreads();
    for (int j = wave; j < 4 * UNITS; j += KW)
      if (b0 + (j >> 2) * PARTS < tiles) finish(u0 + b0 / PARTS + (j >> 2), j & 3, (j >> 2) * PARTS);
    __syncthreads();
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
constexpr int SLOTS = 4, SLOT = 2048, NOWHERE = (int)0x80000000u;  // (NOWHERE: an offset beyond every buffer)

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

int steps_per_wave(int K) { return (lq_ceil_div(lq_ceil_div(K, 32), KW) + 1) / 2 * 2; }

template <int XS, bool GATED, bool PACKED>
int launch_first(const bf16_t* x, int ldx, const bf16_t* w, int ldw, bf16_t* act, int ldo, int K, const FirstArgs& a, int grid,
                 hipStream_t stream) {
  const auto kernel = moe_few_first_kernel<XS, GATED, PACKED>;
  constexpr int lds = 8 * KW * 256 * (int)sizeof(float);
  static bool configured = false;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
      lq_set_error("moe_few: cannot reserve %d bytes of LDS: %s", lds, hipGetErrorString(e));
      return -2;
    }
    configured = true;
  }
  kernel<<<grid, THREADS, lds, stream>>>(x, ldx, w, ldw, act, ldo, K, steps_per_wave(K), a);
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
  const long long units = ((long long)experts * ff + shared) / 16;
  const int grid = units < lq_compute_units() ? (int)units : lq_compute_units(), gated = unit != UNIT_RELU2;
#define LQ_FIRST(XS, GATED, PACKED) \
  launch_first<XS, GATED, PACKED>((const bf16_t*)x, ldx, (const bf16_t*)w, ldw, (bf16_t*)act, ldo, width, a, grid, stream)
  if (steps_per_wave(width) <= 4)
    return gated ? (w_packed ? LQ_FIRST(4, true, true) : LQ_FIRST(4, true, false))
                 : (w_packed ? LQ_FIRST(4, false, true) : LQ_FIRST(4, false, false));
  return gated ? (w_packed ? LQ_FIRST(8, true, true) : LQ_FIRST(8, true, false))
               : (w_packed ? LQ_FIRST(8, false, true) : LQ_FIRST(8, false, false));
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
