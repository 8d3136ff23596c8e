// Decoding steps (one row a sequence) of causal grouped-query attention over the paged bfloat16 cache, on the matrix cores.
//
// A workgroup of four wavefronts takes a share of one sequence's keys for the query heads of one kv head (up to 16, the columns
// of its products) and walks it a cache block (64 positions) at a time.  All four work on the same block:
//   S^T[key][head] = K . Q^T by v_mfma_f32_16x16x32_bf16: wavefront w's 16 keys 16 w .. + 15 (lane l gives A[row l%16][k (l/16)*8 ..
//   + 8] and B[col l%16][the same k], and receives D[(l/16)*4 + e][l%16]); the scores of all 64 keys meet in LDS, from where every
//   wavefront takes its columns' 64 (eight consecutive keys a lane, as the second product wants them) and works out the same
//   probabilities;
//   O^T[d][head] += V^T . P^T for the tiles of 16 value entries w, w + 4, ...: no two wavefronts hold parts of one sum, so nothing is
//   merged at the end of a share.
// The cache stores V transposed per block for exactly this read: V[block][kv head][d][offset].  Softmax statistics, scores and the
// output accumulator are 32-bit; probabilities are rounded to bfloat16 only as MFMA operands (their sum is taken before rounding).
//
// What bounds a step of short contexts is the rate at which one compute unit draws its keys (32 KB a block of head size 128, about
// 1.1 us at 29 GB/s), the round trips around it (position, block table, keys; and for a row in several shares the partial
// results' way out, a ticket and their way back: 1.5 us) and the code itself: a launch finds none of it in the instruction cache, and every
// kilobyte on the way costs some 0.1 us (the same kernel with its walk laid out twice, 25 KB for 10, took 1 us longer at every
// length).  So a row's blocks are dealt out evenly over as many workgroups as do not get into each other's way
// (`blocks_a_share`), by its true length; the keys are asked for before the query is rotated; there is one copy of the walk, with the next
// block asked for ahead of this one's products, so that long contexts stream.  A row in several shares is finished by whichever of its
// workgroups comes last (a ticket counter per row and kv head), which adds the partial results up in ascending order, up to 16
// shares' asked for at once: no second kernel, and the result does not depend on which workgroup that was.
//
// Microseconds a launch, 32 heads over 8, a wavefront with a cache block of its own (merged through LDS, splits of at least 256
// positions, partial results four splits at a time) -> this: head size 128, one sequence of 100 keys 6.4 -> 5.4, 300 10.8 -> 6.8, 1 500 12.3 ->
// 9.0, 7 010 21.7 -> 15.4, 30 000 38.9 -> 34.9 (3.5 TB/s); 8 of 530 12.2 -> 10.6, 8 of 2 070 23.7 -> 20.2, 8 of 8 020 54.7 -> 53.0 (5.0 TB/s);
// 64 of 560 from pieces 41.6 -> 34.3 (4.3 TB/s); 16 of 128 to 7 628 by units 64 -> 57.  Head size 64: one of 120 4.8 -> 4.2, of 3 000 9.7 ->
// 9.1; 16 of 80 to 1 516 by units from pieces 15.5 -> 13.8; 24 of 160 6.5 -> 6.1.
// Found slower (of 1 202 launches of 1 to 96 rows) by more than 5 %: 16 heads of 64 over as many, 56 rows of 60 keys 6.9 -> 7.5, 96 9.1 -> 9.6; 12 of 96, 8 rows of 200 6.4 -> 7.0,
// 16 of 1 000 17.8 -> 18.8, 56 of 4 000 177 -> 187.
#include "attention_mfma.h"

namespace {

constexpr int NW = 4;                   // wavefronts a workgroup
constexpr int MAX_DECODE_BLOCKS = 512;  // workgroups that share the keys of unequal sequences out
// Partial results that cross from one workgroup of a launch to another.  The L2 caches of the chip's
// dies are not coherent with each other for ordinary accesses, and the fences that make them so
// write back and invalidate a whole L2 for everybody.  Device-scope atomic stores and loads go
// past those caches instead: the writer waits until its stores have completed before it takes its
// ticket, the reader reads after it has seen the last ticket.  Two neighbours go as 8 bytes.
__device__ inline void publish2(float* p, float x, float y) {
  const unsigned long long v = (unsigned long long)__float_as_uint(y) << 32 | __float_as_uint(x);
  __hip_atomic_store((unsigned long long*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline float2 published2(const float* p) {
  const unsigned long long v = __hip_atomic_load((unsigned long long*)const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return make_float2(__uint_as_float((unsigned)v), __uint_as_float((unsigned)(v >> 32)));
}

struct DecodeArgs {
  const bf16_t* q;
  int ldq;
  bf16_t* out;
  int ldo;
  int nh, nkv, group;  // group: query heads a kv head
  const int* row_pos;
  const int* seq_slot;
  const int* block_table;
  int bt_stride;
  const bf16_t* kcache;
  const bf16_t* vcache;
  float scale_log2;  // scale * log2(e)
  int window;
  int batch;
  float* part_o;     // [rows][nh][nsplit][HD], or [nkv][units][heads of the group][HD]
  float* part_ml;    // the same with 2: maximum and sum
  int nsplit;        // workgroups a row and kv head
  int narrow_splits; // the same without a second workgroup on any compute unit
  int long_from;     // > 0: a row goes in nsplit shares from this many blocks on, else whole (many_rows)
  int units;         // > 0: workgroups a kv head, which share the sequences' keys out among themselves
  int* tickets;      // [rows][nkv], zero between launches: how many shares of the row have finished
  // with the rotation and the cache write folded in (all null otherwise): the step's
  // unrotated keys and values, and cos/sin of every row's angles [rows][HD/2][2]
  const bf16_t* k_new;
  const bf16_t* v_new;
  int ldk, ldv;
  const float* cs;
  // > 1 (folded launches only): q, k_new and v_new are float32, the partial sums that a product whose K was
  // shared over blocks left, `pieces` of them `piece_stride` floats apart; ldq, ldk and ldv count floats.
  // The kernel adds them up in order and rounds the sums as the whole product would have.
  int pieces;
  long long piece_stride;
};

// Which split of which sequence unit u of a kv head takes, when the units share the work out themselves
// (a few sequences, no window).  Every sequence's keys are cut into splits of one length: the smallest
// multiple of 256 with which the splits that hold keys number no more than the launch has units for a kv
// head.  Those splits are numbered through (the whole ones first, sequence after sequence, then every
// sequence's last, part-filled one), and unit u takes number u.  With sequences of unequal lengths a launch
// whose grid is (sequence, split) leaves the splits of the short ones empty and makes the long ones' as large
// as if all were long; here a unit has work or ends at once, and the units with work follow one another, so
// that the compute units (which take workgroups in turn) get equal numbers of them.  Lane l holds sequence l;
// every wave of the workgroup works out the same answer.
struct DecodeItem {
  int row, pos, slot, split_len, split;
  int first_unit, n_full, last_unit;  // the row's whole splits sit in units first_unit .., its last, part-filled one in last_unit
};

// Inclusive prefix sums over the wave's 64 lanes with data-parallel-primitive moves (no trip through LDS):
// within rows of 16 lanes by shifts of 1, 2, 4 and 8 (lanes shifted in from outside a row read zero), then
// lane 15 of a row into the odd rows and lane 31 into the upper half.
__device__ inline int wave_prefix_sums(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);   // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);   // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);   // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return v;
}

// Splits of length 256 k that hold keys of a sequence whose newest position is `pos` (position p lies in block
// p / 256; blocks of 256 positions and their quotients are small integers, which a float division gives exactly).
// One function for the kernel's search and for the host's check of it.
__host__ __device__ inline int splits_with_keys(int pos, int k) {
  return (int)(((float)(pos >> 8) + 0.5f) / (float)k) + 1;
}
constexpr int UNIT_SEARCH_TRIES = 1024;

// -> 1: unit u has work (in `it`); 0: it has none; -1: no split length was found within the tries, which the
// host's choice of the units rules out (decode_units) as long as the lengths lie within the launch's bound.
__device__ inline int balanced_item(const DecodeArgs& a, int u, DecodeItem& it) {
  const int lane = threadIdx.x & 63;
  const bool mine = lane < a.batch;
  const int pl = mine ? a.row_pos[lane] : -1;  // lane l looks after sequence l (at most 64 of them)
  const int sl = mine ? a.seq_slot[lane] : 0;
  const int total = __builtin_amdgcn_readlane(wave_prefix_sums(pl + 1), 63);
  // the smallest multiple of 256 with which the splits that hold keys are no more than the units; blocks of
  // 256 positions and their quotients are small integers, which a float division gives exactly
  int k = max(1, (total + 256 * a.units - 1) / (256 * a.units)), cnt = 0;
  for (int tries = 0; tries < UNIT_SEARCH_TRIES; ++tries, ++k) {
    cnt = mine ? splits_with_keys(pl, k) : 0;  // splits of this lane's sequence that hold keys
    if (__builtin_amdgcn_readlane(wave_prefix_sums(cnt), 63) <= a.units) break;
  }
  const int SL = 256 * k;
  // whole splits first, sequence after sequence, then the last splits (the part-filled ones): the two
  // workgroups that share a compute unit, c and c + 32 of a die's run, then differ as little as may be
  const int part = mine && (pl + 1) % SL != 0 ? 1 : 0, full = cnt - part;
  const int full_incl = wave_prefix_sums(full), part_incl = wave_prefix_sums(part);
  const int n_full = __builtin_amdgcn_readlane(full_incl, 63), n_part = __builtin_amdgcn_readlane(part_incl, 63);
  if (n_full + n_part > a.units) return -1;
  if (u >= n_full + n_part) return 0;
  const bool whole = u < n_full;
  const int row = whole ? __popcll(__ballot(mine && full_incl <= u))
                        : __popcll(__ballot(mine && part_incl <= u - n_full));
  it.row = row;
  it.pos = __builtin_amdgcn_readlane(pl, row);
  it.slot = __builtin_amdgcn_readlane(sl, row);
  it.split_len = SL;
  it.n_full = __builtin_amdgcn_readlane(full, row);
  it.first_unit = __builtin_amdgcn_readlane(full_incl - full, row);
  it.last_unit = n_full + __builtin_amdgcn_readlane(part_incl - part, row);
  it.split = whole ? u - it.first_unit : it.n_full;
  return 1;
}

// What a wavefront holds of the cache blocks that are taken together: of each its 16 keys (row lane % 16, entries 32 kk + 8 (lane /
// 16) ..), and of its tiles of value entries row lane % 16, positions 32 j + 8 (lane / 16) .. .  Both halves of a line are asked for
// by instructions next to each other, which the L1 turns into one request of 128 bytes.  Head sizes up to 64 take two blocks together:
// 32 KB on their way for a barrier, as with one block of 128 (or one, where more workgroups a unit serve better: `launch`).
template <int HD, int TOGETHER>
struct Share {
  static constexpr int KS = HD / 32, VT = HD / 16, VW = (VT + NW - 1) / NW, GB = TOGETHER;
  u32x4 k[GB][KS];
  u32x4 v[GB][VW][2];
};

// Asks for a block, or, with the same instructions, for nothing at all (`there`: a descriptor of no bytes, every access of which
// is out of bounds and yields zero): a share's last blocks need no branch, behind which the compiler would have to wait for
// whatever may have been asked for.  Tiles of value entries beyond the head's are out of bounds too.
template <int HD, int GB>
__device__ inline void ask_block(const DecodeArgs& a, int kvh, int blk, bool there, int wave, int c16, int g, int u, Share<HD, GB>& s) {
  using S = Share<HD, GB>;
  const long long base = ((long long)blk * a.nkv + kvh) * (BS * HD);
  const int bytes = there ? BS * HD * 2 : 0;
  const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc((void*)(a.kcache + base), 0, bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc((void*)(a.vcache + base), 0, bytes, 0x00020000);
  const int k_at = ((16 * wave + c16) * HD + g * 8) * 2, v_at = ((16 * wave + c16) * BS + g * 8) * 2;
#pragma unroll
  for (int kk = 0; kk < S::KS; ++kk) s.k[u][kk] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(kr, k_at + kk * 64, 0, 0));
#pragma unroll
  for (int x = 0; x < S::VW; ++x)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      s.v[u][x][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(vr, v_at + x * (NW * 16 * BS * 2) + 64 * j, 0, 0));
}

// ceil(n / d) of positive whole numbers below 2^20: half a unit of the numerator is more than the reciprocal's error.
__device__ inline int ceil_quotient(int n, int d) {
  return __builtin_amdgcn_readfirstlane((int)(((float)(n - 1) + 0.5f) * __builtin_amdgcn_rcpf((float)d)) + 1);
}

typedef u32x4 u32x4_anywhere __attribute__((aligned(2)));  // (an unaligned load of 16 bytes)
typedef f32x4 f32x4_anywhere __attribute__((aligned(4)));

// A head's row on its way to a product's operand (a lane's fragment kk: entries 32 kk + 8 (lane / 16) .. + 7).  Asking for it and using
// it are apart, so that the keys are asked for between the two.  From bfloat16 every wavefront takes the whole row; float32 pieces
// are added up (in ascending order, their sum is rounded) by one wavefront a fragment, through which the others get it in LDS:
// `put` ahead of a barrier, `get` behind it.
template <int HD, bool PIECES>
struct RowOf {
  static constexpr int KS = HD / 32, KW = (KS + NW - 1) / NW, AHEAD = HD <= 128 ? 4 : 2;
  int first;  // (whose wavefront adds up fragment 0)
  u32x4 x[PIECES ? 1 : KS];
  f32x4 t[PIECES ? AHEAD : 1][KW][2];
  const bf16_t* row;

  __device__ inline const f32x4_anywhere* piece(const DecodeArgs& a, int j, int g, int kk) const {
    return (const f32x4_anywhere*)((const float*)row + j * a.piece_stride + g * 8 + kk * 32);
  }
  __device__ inline void ask(const DecodeArgs& a, const bf16_t* row_, int first_, int wave, int g) {
    row = row_, first = first_;
    if constexpr (PIECES) {
#pragma unroll
      for (int y = 0; y < KW; ++y) {
        const int kk = wave - first + NW * y;
        if (kk >= 0 && kk < KS)
#pragma unroll
          for (int j = 0; j < AHEAD; ++j) {
            const f32x4_anywhere* p = piece(a, min(j, a.pieces - 1), g, kk);
            t[j][y][0] = p[0], t[j][y][1] = p[1];
          }
      }
    } else {
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) x[kk] = *(const u32x4_anywhere*)(row + g * 8 + kk * 32);
    }
  }
  __device__ inline void put(const DecodeArgs& a, u32x4 (*lds)[64], int wave, int g) {
    if constexpr (PIECES) {
#pragma unroll
      for (int y = 0; y < KW; ++y) {
        const int kk = wave - first + NW * y;
        if (kk < 0 || kk >= KS) continue;
        f32x4 sum[2] = {t[0][y][0], t[0][y][1]};
#pragma unroll
        for (int j = 1; j < AHEAD; ++j)
          if (j < a.pieces) sum[0] += t[j][y][0], sum[1] += t[j][y][1];
        for (int j = AHEAD; j < a.pieces; ++j) {
          const f32x4_anywhere* p = piece(a, j, g, kk);
          sum[0] += p[0], sum[1] += p[1];
        }
        u32x4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = pack_bf16(sum[e >> 1][2 * (e & 1)], sum[e >> 1][2 * (e & 1) + 1]);
        lds[kk][threadIdx.x & 63] = w;
      }
    }
  }
  __device__ inline void get(const u32x4 (*lds)[64], u32x4 (&to)[KS]) const {
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      if constexpr (PIECES) to[kk] = lds[kk][threadIdx.x & 63];
      else to[kk] = x[kk];
    }
  }
};

// The cosines and sines of a row's angles [HD/2][2] that a lane's entries take: pair (i, i + HD/2), its fragment kk holding
// i = kk*32 + (lane/16)*8 + j and its fragment kk + HD/64 the partners.
template <int HD>
struct Turn {
  f32x4 c[HD / 64 > 0 ? HD / 64 : 1][4];  // cos, sin of two neighbours
};
template <int HD>
__device__ inline void turn_row(const Turn<HD>& by, u32x4 (&x)[HD / 32]) {
#pragma unroll
  for (int kk = 0; kk < HD / 64; ++kk)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4 c2 = by.c[kk][j];
      const unsigned lo = x[kk][j], hi = x[kk + HD / 64][j];
      const float x0a = __uint_as_float(lo << 16), x0b = __uint_as_float(lo & 0xffff0000u);
      const float x1a = __uint_as_float(hi << 16), x1b = __uint_as_float(hi & 0xffff0000u);
      x[kk][j] = pack_bf16(x0a * c2[0] - x1a * c2[1], x0b * c2[2] - x1b * c2[3]);
      x[kk + HD / 64][j] = pack_bf16(x0a * c2[1] + x1a * c2[0], x0b * c2[3] + x1b * c2[2]);
    }
}

// Blocks a share of a row that has n, where rows leave at least half of the compute units free (else: many_rows).  In units of 32 KB of keys and values (a block of head size 128, two of 64), which take a compute
// unit 1.1 us: a row of up to three stays whole (a second share costs 1.5 us: partial results out, ticket, and back).  Each share
// more costs its ticket and its results' way into the last workgroup 0.13 us, which is worth it down to sqrt(n / 8) of them a share
// (one sequence of 1 500 keys 10.1 us with one each, 9.1 with two; of 7 010: 15.4 with four).  Where up to three a share do without a second
// workgroup on any compute unit, they do: 12 rows of 330 keys over 8 kv heads 12.4 -> 10.6 us, 8 of 530 10.9 -> 10.5; beyond that two a
// unit hide each other's round trips (8 of 2 070 keys 21.6 -> 20.4).
template <int HD>
__device__ inline int blocks_a_share(const DecodeArgs& a, int n) {
  constexpr int UNIT = HD <= 64 ? 2 : 1;
  if (n <= 3 * UNIT || n < a.long_from) return n;
  if (a.long_from > 0) return ceil_quotient(n, a.nsplit);
  const int narrow = ceil_quotient(n, a.narrow_splits);
  const int even = narrow <= 3 * UNIT ? narrow : ceil_quotient(n, a.nsplit);
  const int apart = __builtin_amdgcn_readfirstlane((int)(__builtin_amdgcn_sqrtf((float)n * (HD <= 64 ? 0.2f : 0.125f)) + 0.99f));
  return max(even, apart);
}

// GB: blocks taken together; HELD: workgroups that a compute unit holds at least.
template <int HD, bool PIECES, int GB, int HELD>
__global__ __launch_bounds__(NW * 64, HELD) void attn_decode_kernel(DecodeArgs a) {
  using S = Share<HD, GB>;
  __shared__ __attribute__((aligned(16))) float scores[2][16][S::GB * BS + 4];  // (apart so that neighbouring heads' lie in other banks)
  __shared__ __attribute__((aligned(16))) float tops[2][16][NW];  // (what wavefronts' probabilities were taken against)
  __shared__ u32x4 rows[PIECES ? 2 * S::KS : 1][64];
  __shared__ int last_workgroup;
  const int G = a.group;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c16 = lane & 15, g = lane >> 4;
  // grid (sequence, kv head, share), or (kv head, unit) when the units share the keys out themselves
  int r = blockIdx.x, kvh = blockIdx.y, split = blockIdx.z, p, slot, per_unit = 0;
  int first_unit = 0, n_full = 0, last_unit = 0;
  if (a.units > 0) {
    DecodeItem it;
    kvh = blockIdx.x;
    const int found = balanced_item(a, blockIdx.y, it);
    if (found < 0) {
      // Nobody would write the output: make that loud instead of leaving what the buffer held.  Units 0 ..
      // batch - 1 (there are at least two a sequence) fill their row's heads of this kv head with NaN.
      if ((int)blockIdx.y < a.batch) {
        bf16_t nan;
        nan.bits = 0x7FC0;
        bf16_t* o = a.out + (long long)blockIdx.y * a.ldo + (long long)kvh * G * HD;
        for (int i = tid; i < G * HD; i += NW * 64) o[i] = nan;
      }
      return;
    }
    if (found == 0) return;  // the whole workgroup: more units than splits with keys
    r = it.row;  // (a decoding step has one row a sequence, in the order of the sequences)
    p = it.pos;
    slot = it.slot;
    per_unit = it.split_len / BS;
    split = it.split;
    first_unit = it.first_unit;
    n_full = it.n_full;
    last_unit = it.last_unit;
  } else {
    p = a.row_pos[r];
    slot = a.seq_slot[r];
  }
  // The query and its angles are asked for before the position is known (or, with units, together with the block table): a
  // share's time is a chain of memory round trips (position, block table, keys), and these join the first of them.  They are
  // used only when the keys are on their way.
  const int h = kvh * G + min(c16, G - 1);  // (columns beyond the group's heads repeat the last one's; nobody stores them)
  const bool folded = HD % 64 == 0 && a.cs != nullptr;
  constexpr int P = PIECES ? 2 : 1;  // (pointers to rows count 2-byte entries)
  RowOf<HD, PIECES> q_row, k_row;
  q_row.ask(a, a.q + P * ((long long)r * a.ldq + h * HD), 0, wave, g);
  // the row's own key and value, for the share that holds their place
  constexpr int VA = PIECES ? 4 : 1;
  float v_raw[VA][S::VW], v_own[S::VW];
  const long long v_at = (long long)r * a.ldv + kvh * HD + c16;
  if (folded) {
    k_row.ask(a, a.k_new + P * ((long long)r * a.ldk + kvh * HD), S::KS < NW ? NW - S::KS : 0, wave, g);
#pragma unroll
    for (int x = 0; x < S::VW; ++x) {
      const long long at = v_at + min(wave + NW * x, S::VT - 1) * 16;
#pragma unroll
      for (int j = 0; j < VA; ++j) {
        if constexpr (PIECES) v_raw[j][x] = ((const float*)a.v_new + min(j, a.pieces - 1) * a.piece_stride)[at];
        else v_raw[j][x] = bf16_to_f32(a.v_new[at]);
      }
    }
  }
  Turn<HD> turn;
  if (folded) {
    const float* cs = a.cs + (long long)r * HD + g * 16;
#pragma unroll
    for (int kk = 0; kk < HD / 64; ++kk)
#pragma unroll
      for (int j = 0; j < 4; ++j) turn.c[kk][j] = *(const f32x4*)(cs + (kk * 32 + 2 * j) * 2);
  }
  __builtin_amdgcn_sched_barrier(0);
  // the share: blocks b0 .. b1 of the row's first .. last
  const int lo = (a.window > 0 && p >= a.window) ? p - a.window + 1 : 0, first = lo / BS, last = p / BS, n = last - first + 1;
  const int per = a.units > 0 ? per_unit : blocks_a_share<HD>(a, n), shares = ceil_quotient(n, per);
  if (split >= shares) return;  // the whole workgroup
  const int b0 = first + split * per, b1 = min(b0 + per - 1, last);
  const int* table = a.block_table + (long long)slot * a.bt_stride;
  const bool own = folded && b1 == last;  // whether this share holds the row's own position
  u32x4 q[S::KS], k_own[S::KS];
  S cur;
  // The first blocks' numbers come by scalar loads, those of the blocks behind them 64 at a time, lane l that of block b0 + l.  (Each
  // looked up on its own, a block ahead, the walk waited for its way through memory, and where two blocks go together for the
  // keys that were asked for between the two lookups: one sequence of 160 keys, head size 64, 5.5 -> 5.0 us, 24 of 160 6.8 -> 6.1, 16 of 530 from
  // pieces 11.8 -> 9.8; head size 128, a whole row a unit of 24 sequences of 3 000 keys 64.9 -> 58.6.)
  int numbers = table[min(b0 + lane, b1)];
#pragma unroll
  for (int u = 0; u < S::GB; ++u) ask_block<HD, GB>(a, kvh, table[min(b0 + u, b1)], b0 + u <= b1, wave, c16, g, u, cur);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (PIECES) {
    q_row.put(a, rows, wave, g);
    if (own) k_row.put(a, rows + S::KS, wave, g);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
  q_row.get(rows, q);
  if (folded) turn_row<HD>(turn, q);
  const int hi = min(p, b1 * BS + BS - 1);  // the share's last key
#pragma unroll
  for (int x = 0; x < S::VW; ++x) v_own[x] = 0.f;
  if (own) {
    k_row.get(rows + S::KS, k_own);
    turn_row<HD>(turn, k_own);
#pragma unroll
    for (int x = 0; x < S::VW; ++x) {
      v_own[x] = v_raw[0][x];
#pragma unroll
      for (int j = 1; j < VA; ++j)
        if (j < a.pieces) v_own[x] += v_raw[j][x];
      if constexpr (PIECES)
        for (int j = VA; j < a.pieces; ++j)
          v_own[x] += ((const float*)a.v_new + j * a.piece_stride)[v_at + min(wave + NW * x, S::VT - 1) * 16];
    }
  }

  f32x4 o[S::VW];  // o[x][e]: value entry 16 (wave + NW x) + 4 g + e of head c16
  float m = -INFINITY, l = 0.f;
#pragma unroll
  for (int x = 0; x < S::VW; ++x) o[x] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // Blocks b .. b + GB - 1 of the share, as far as it reaches; `turn_of`: whose turn it is of the two buffers.  A wavefront takes its
  // keys' probabilities against their own maximum; whoever reads them multiplies them up to the row's.
  auto take = [&](int b, int turn_of, S& s) {
    f32x4 st[S::GB];  // keys 64 (b + u) + 16 wave + 4 g + e
    float own_top = -INFINITY;
#pragma unroll
    for (int u = 0; u < S::GB; ++u) {
      const int t0 = (b + u) * BS;
      if (b + u == last) {
        // The row's own key and value are put in where the cache's would be: whoever reads this block need not wait for
        // their way through memory.  Values of keys that were never written must not reach the product (0 times what lies
        // there may be NaN).
        const int off = p & (BS - 1), end = off + (own ? 0 : 1) - 8 * g;  // (entries of the lane's from `end` on are not the cache's)
        if (own && 16 * wave + c16 == off)
#pragma unroll
          for (int kk = 0; kk < S::KS; ++kk) s.k[u][kk] = k_own[kk];
        unsigned word[S::VW];  // the word that the row's own value shares with nothing or with its older neighbour
#pragma unroll
        for (int x = 0; x < S::VW; ++x) word[x] = (pack_bf16(v_own[x], 0.f) & 0xffffu) << (end & 1 ? 16 : 0);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int t = 32 * j + 2 * e;
            const unsigned keep = end > t + 1 ? 0xffffffffu : end > t ? 0xffffu : 0u;
#pragma unroll
            for (int x = 0; x < S::VW; ++x) s.v[u][x][j][e] = (s.v[u][x][j][e] & keep) | (end >> 1 == t >> 1 ? word[x] : 0u);
          }
      }
      st[u] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < S::KS; ++kk) st[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(s.k[u][kk]), as_bf16x8(q[kk]), st[u], 0, 0, 0);
      if (t0 + BS - 1 > hi || t0 < lo)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int t = t0 + 16 * wave + 4 * g + e;
          if (t > hi || t < lo) st[u][e] = -INFINITY;
        }
      own_top = fmaxf(own_top, fmaxf(fmaxf(st[u][0], st[u][1]), fmaxf(st[u][2], st[u][3])));
    }
    own_top = rows_max(own_top) * a.scale_log2;  // (scale > 0: it commutes with the maximum)
    const float own_safe = own_top == -INFINITY ? 0.f : own_top;
#pragma unroll
    for (int u = 0; u < S::GB; ++u) {
#pragma unroll
      for (int e = 0; e < 4; ++e) st[u][e] = fast_exp2(fmaf(st[u][e], a.scale_log2, -own_safe));
      *(f32x4*)&scores[turn_of][c16][u * BS + 16 * wave + 4 * g] = st[u];
    }
    if (g == 0) tops[turn_of][c16][wave] = own_top;
    // (loads fly on; the other buffer's readers have passed this barrier once more than its writers)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const f32x4 tw = *(const f32x4*)&tops[turn_of][c16][0];
    f32x4 sv[S::GB][4];  // keys 64 (b + u) + 32 (i / 2) + 8 g + 4 (i % 2) .. + 3
#pragma unroll
    for (int u = 0; u < S::GB; ++u) {
#pragma unroll
      for (int i = 0; i < 4; ++i) sv[u][i] = *(const f32x4*)&scores[turn_of][c16][u * BS + 32 * (i >> 1) + 8 * g + 4 * (i & 1)];
    }
    const float top = fmaxf(fmaxf(tw[0], tw[1]), fmaxf(tw[2], tw[3]));
    if (__any(top > m + RESCALE_SLACK)) {
      const float m_new = fmaxf(m, top), alpha = fast_exp2(m - (m_new == -INFINITY ? 0.f : m_new));
      l *= alpha;
      m = m_new;
#pragma unroll
      for (int x = 0; x < S::VW; ++x) o[x] *= alpha;
    }
    const float m_safe = m == -INFINITY ? 0.f : m;  // (a head all of whose scores so far are -inf)
    const float up[2] = {fast_exp2((g < 2 ? tw[0] : tw[1]) - m_safe), fast_exp2((g < 2 ? tw[2] : tw[3]) - m_safe)};
#pragma unroll
    for (int u = 0; u < S::GB; ++u) {
      f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sv[u][i] *= up[i >> 1];
        sum += sv[u][i];
      }
      l += (sum[0] + sum[1]) + (sum[2] + sum[3]);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        u32x4 pw;
#pragma unroll
        for (int e = 0; e < 4; ++e) pw[e] = pack_bf16(sv[u][2 * j + (e >> 1)][2 * (e & 1)], sv[u][2 * j + (e >> 1)][2 * (e & 1) + 1]);
#pragma unroll
        for (int x = 0; x < S::VW; ++x)
          o[x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(s.v[u][x][j]), as_bf16x8(pw), o[x], 0, 0, 0);
      }
    }
  };
  for (int b = b0, odd = 0;; b += S::GB, odd ^= 1) {
    S next;
    const int at = (b + S::GB - b0) & 63;
    if (at == 0) {  // (64 is a multiple of GB)
      numbers = table[min(b + S::GB + lane, b1)];
      asm volatile("" : "+v"(numbers));  // (waited for in here, not behind the branch)
    }
#pragma unroll
    for (int u = 0; u < S::GB; ++u)
      ask_block<HD, GB>(a, kvh, __builtin_amdgcn_readlane(numbers, at + u), b + S::GB + u <= b1, wave, c16, g, u, next);
    take(b, odd, cur);
    if (b + S::GB > b1) break;
    cur = next;
  }
  if (own) {  // the row's key and value go into the cache; nobody reads them there in this launch
    const long long blk = table[last];
    const int off = p & (BS - 1);
    if (wave == 0 && c16 == 0) {
      bf16_t* kd = const_cast<bf16_t*>(a.kcache) + ((blk * a.nkv + kvh) * BS + off) * (long long)HD + g * 8;
#pragma unroll
      for (int kk = 0; kk < S::KS; ++kk) *(u32x4*)(kd + kk * 32) = k_own[kk];
    }
    if (g == 0) {
      bf16_t* vd = const_cast<bf16_t*>(a.vcache) + ((blk * a.nkv + kvh) * (long long)HD + c16) * BS + off;
#pragma unroll
      for (int x = 0; x < S::VW; ++x)
        if (wave + NW * x < S::VT) vd[(wave + NW * x) * 16 * BS].bits = (uint16_t)(pack_bf16(v_own[x], 0.f) & 0xffffu);
    }
  }
  l = rows_sum(l);
  if (shares == 1) {
    const float inv = 1.0f / l;
    bf16_t* to = a.out + (long long)r * a.ldo + h * HD + g * 4;
    if (c16 < G)
#pragma unroll
      for (int x = 0; x < S::VW; ++x)
        if (wave + NW * x < S::VT) {
          u32x2 w;
          w[0] = pack_bf16(o[x][0] * inv, o[x][1] * inv);
          w[1] = pack_bf16(o[x][2] * inv, o[x][3] * inv);
          *(u32x2*)(to + (wave + NW * x) * 16) = w;
        }
    return;
  }
  // Share s of head c of the group lies at entry `place(s)` + c * apart: by (row, head, share), or by (kv head, unit, head of the
  // group), where a row's whole splits are units next to each other and its last, part-filled one is another.
  const int apart = a.units > 0 ? 1 : a.nsplit, step = a.units > 0 ? G : 1;
  const int place0 = a.units > 0 ? (kvh * a.units + first_unit) * G : (r * a.nh + kvh * G) * a.nsplit;
  const int place_last = a.units > 0 && n_full < shares ? (kvh * a.units + last_unit) * G : place0 + (shares - 1) * step;
  auto place = [&](int s) { return s == shares - 1 ? place_last : place0 + s * step; };
  if (c16 < G) {
    const int at = place(split) + c16 * apart;
    float* to = a.part_o + (long long)at * HD + wave * 16 + g * 4;
#pragma unroll
    for (int x = 0; x < S::VW; ++x)
      if (wave + NW * x < S::VT) {
        publish2(to + NW * x * 16, o[x][0], o[x][1]);
        publish2(to + NW * x * 16 + 2, o[x][2], o[x][3]);
      }
    if (wave == 0 && g == 0) publish2(a.part_ml + 2LL * at, m, l);
  }
  // Once every thread's stores have completed the workgroup takes a ticket; the one that takes the last one adds the
  // shares up.
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this thread's stores have been acknowledged
  __syncthreads();
  if (tid == 0) {
    const int done = __hip_atomic_fetch_add(&a.tickets[(long long)r * a.nkv + kvh], 1, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT);
    last_workgroup = done == shares - 1;
  }
  __syncthreads();
  if (!last_workgroup) return;
  for (int i = tid; i < G * HD / 2; i += NW * 64) {
    const int c = i / (HD / 2), d = 2 * (i % (HD / 2));
    constexpr int AT_ONCE = 8;
    const float* ml = a.part_ml + 2LL * c * apart;
    const float* po = a.part_o + (long long)c * apart * HD + d;
    float M = -INFINITY, L = 0.f;
    float2 acc = make_float2(0.f, 0.f);
    // eight shares, or twice eight, are asked for together, as far as there are so many (partial results come past the caches, at 13 GB/s
    // a compute unit: 12 rows of 250 keys in two shares each, with requests for eight, 8.9 us, with two 8.5)
    auto ask = [&](int s0, float2 (&stat)[AT_ONCE], float2 (&sum)[AT_ONCE]) {
#pragma unroll
      for (int j = 0; j < AT_ONCE; ++j) {
        stat[j] = make_float2(-INFINITY, 0.f), sum[j] = make_float2(0.f, 0.f);
        if (s0 + j < shares) {  // (the same for the whole workgroup)
          const long long at = place(s0 + j);
          stat[j] = published2(ml + 2 * at), sum[j] = published2(po + at * HD);
        }
      }
    };
    auto add = [&](int s0, const float2 (&stat)[AT_ONCE], const float2 (&sum)[AT_ONCE]) {
      float top = M;
#pragma unroll
      for (int j = 0; j < AT_ONCE; ++j) top = fmaxf(top, stat[j].x);
      const float safe = top == -INFINITY ? 0.f : top, keep = fast_exp2(M - safe);
      acc.x *= keep, acc.y *= keep, L *= keep, M = top;
#pragma unroll
      for (int j = 0; j < AT_ONCE; ++j) {
        const float f = s0 + j < shares ? fast_exp2(stat[j].x - safe) : 0.f;
        acc.x = fmaf(f, sum[j].x, acc.x), acc.y = fmaf(f, sum[j].y, acc.y), L = fmaf(f, stat[j].y, L);
      }
    };
    for (int s0 = 0; s0 < shares; s0 += 2 * AT_ONCE) {
      float2 stat[2][AT_ONCE], sum[2][AT_ONCE];
      ask(s0, stat[0], sum[0]);
      const bool more = s0 + AT_ONCE < shares;
      if (more) ask(s0 + AT_ONCE, stat[1], sum[1]);
      add(s0, stat[0], sum[0]);
      if (more) add(s0 + AT_ONCE, stat[1], sum[1]);
    }
    const float inv = 1.0f / L;
    *(unsigned*)(a.out + (long long)r * a.ldo + (kvh * G + c) * HD + d) = pack_bf16(acc.x * inv, acc.y * inv);
  }
  if (tid == 0)  // for the next launch
    __hip_atomic_store(&a.tickets[(long long)r * a.nkv + kvh], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int HD, int GB, int HELD>
int launch(const DecodeArgs& a, hipStream_t stream) {
  const dim3 grid = a.units > 0 ? dim3(a.nkv, a.units) : dim3(a.batch, a.nkv, a.nsplit);
  if (a.pieces > 1) attn_decode_kernel<HD, true, GB, HELD><<<grid, NW * 64, 0, stream>>>(a);
  else attn_decode_kernel<HD, false, GB, HELD><<<grid, NW * 64, 0, stream>>>(a);
  LQ_CHECK_LAUNCH("attention(single tokens)");
  return 0;
}

// Which kernel of a head size.  Of 64, one block at a time in a workgroup of which a unit holds four instead of two blocks in one of which it holds
// three: where rows are one to three a unit, or nearly fill four, but for few more than one that go in shares (16 heads over as many, us: 17 rows of 130 keys
// 7.7 -> 6.8, of 1 000 21.6 -> 19.6, of 7 000 in fives 94 either way; 20 of 7 000 in fours 105 and 109; 24 of 130 8.0 -> 7.0, of 4 000 77 -> 71; 32 of 130
// 8.3 -> 7.5, of 4 000 92 -> 90; 48 of 60 6.5 -> 5.8; 64 of 60 8.3 -> 6.3, of 130 13.8 -> 12.1, of 4 000 either; but 16 of 4 000 46 and 56, 56 of 1 000 45.2
// and 47.2, 80 of 1 000 59 and 65).  Of 128, in 168 registers instead of 170, so that a unit holds three, where there are three (32 over 8: 96 of
// 1 000 80.7 -> 73.7, in two shares 77.4, of 4 000 295 -> 266 and 272; but 104 of 2 000 160 and 165; pieces have the room anyway).
template <int HD>
int launch(const DecodeArgs& a, hipStream_t stream) {
  const long long pairs = (long long)a.batch * a.nkv, cus = lq_compute_units();
  if constexpr (HD == 64)
    if (a.units == 0 && ((pairs > cus && pairs <= 3 * cus && !(a.long_from > 0 && 4 * pairs <= 5 * cus)) || (4 * pairs >= 15 * cus && pairs <= 4 * cus)))
      return launch<HD, 1, 4>(a, stream);
  if constexpr (HD == 128)
    if (a.units == 0 && a.pieces <= 1 && 2 * pairs > 5 * cus && pairs <= 3 * cus) return launch<HD, 1, 3>(a, stream);
  return launch<HD, HD <= 64 ? 2 : 1, HD <= 192 ? 2 : 1>(a, stream);
}

}  // namespace

// How rows are shared out that take more than half of the compute units with one workgroup a kv head: in `shares` from `from` blocks on
// (0: never).  A unit draws at most 29 GB/s and holds two workgroups (three at head sizes up to 64, four of 96, one of 256);
// the memory gives all of them 20 each.  Up to a row a unit that is enough, but for the units that have none: few more rows than half
// of them go in thirds, which give every unit two, and the longest up to four fifths of them in fifths, four in turn (heads of 96, of
// which a unit has 24 KB on the way, from shorter ones on).  With more
// rows than units whole ones would leave some units two and most one, and with more than twice as many some three: shares even that out where
// they fill a whole number of rounds of two (three) nearly.  A share more costs its ticket and partial results, and a round its chain of round
// trips: short rows stay whole.
// 32 heads over 8, whole -> so, microseconds; a wavefront with a block of its own and up to 2 048 workgroups in brackets:
// head size 128: 17 sequences of 1 500 keys 31 -> 28 (38), of 6 000 106 -> 84 (91); 22 of 6 000 114 -> 107 (108); 33 of 1 000 41.5 -> 38 (46), of
// 3 000 106 -> 84 (101), of 6 000 203 -> 161 (176); 40 of 3 000 108 -> 94 (107); 48 of 6 000 223 -> 206 (214); 66 of 3 000 176 -> 153; 80 of 1 500
// 108 -> 100, of 6 000 418 -> 341; 88 of 3 000 in twos 216 -> 196 (and whole, where a unit holds three, 190).  Head size 64: 17 of 3 000 34 -> 27
// (30); 24 of 6 000 66 -> 60 (62); 33 of 6 000 105 -> 84 (90); 66 of 3 000 92 -> 81; 80 of 7 000 216 -> 203; 16 heads over
// as many, 33 of 8 000 235 -> 194 (197).  12 heads of 96: 16 of 3 000 48 -> 43; 43 of 750 36 -> 33, of 3 000 130 -> 112; 48 of 4 000 177 -> 154 (159); 96 of 2 000 166 -> 159 (155).
// Eight heads over 4 of 192: 75 of 750 45 -> 39; 144 of 3 000 257 -> 234.
// (Rows whole that would do in shares, or the reverse: 24 of 200 keys in two shares each 12.5, whole 9.5; 24 of 6 000 118 and 110; 52 of 3 000
// in sixes 127, whole 118; 104 of 1 500 in threes 125, whole 122; 128 of 3 000 in twos 279, whole 266.)
struct ManyRows {
  int shares, from;
};
static ManyRows many_rows(long long pairs, int hd) {
  const long long cus = lq_compute_units();
  const bool small = hd <= 64, narrow = hd == 96;  // (less than 32 KB a block)
  if (3 * pairs <= 2 * cus) return {3, small ? 16 : 12};
  if ((small || narrow) && 4 * pairs <= 3 * cus) return {4, small ? 32 : 20};
  if (!small && 5 * pairs <= 4 * cus) return {5, narrow ? 20 : 80};
  if (pairs <= cus) return {1, 0};
  if (5 * pairs <= 6 * cus) return {5, small ? 17 : hd > 128 ? 10 : 14};
  if (!small && 3 * pairs <= 4 * cus) return {3, hd > 128 ? 10 : 14};
  if (small ? 4 * pairs <= 5 * cus : 2 * pairs <= 3 * cus) return {4, 28};
  if (pairs <= 2 * cus) return {1, 0};
  if (hd > 192) return {1, 0};
  if (small && 5 * pairs > 12 * cus) return 2 * pairs <= 5 * cus ? ManyRows{4, 48} : ManyRows{1, 0};
  if (2 * pairs <= 5 * cus) return {4, narrow ? 10 : 18};
  if (narrow && pairs > 4 * cus && pairs <= 5 * cus) return {3, 14};
  return {1, 0};
}

// Workgroups a row and kv head for a launch whose longest sequence may hold `max_len` tokens: two for every compute unit in all, where rows
// leave half of the units free.  It depends on the bound rounded up to LQ_DECODE_LENGTH_BUCKET, so that launches whose bounds
// differ less than that add up their sums in the same order.
static int decode_splits(int rows, int nkv, int hd, int max_len) {
  const long long bound = (long long)lq_ceil_div(max_len, LQ_DECODE_LENGTH_BUCKET) * LQ_DECODE_LENGTH_BUCKET;
  const int blocks = (int)(bound / BS);
  const long long pairs = (long long)rows * nkv, cus = lq_compute_units();
  if (2 * pairs > cus) {
    const ManyRows many = many_rows(pairs, hd);
    return blocks >= many.from ? many.shares : 1;
  }
  const long long room = 2 * cus / pairs;
  return (int)(room < blocks ? room : blocks);
}

// Units a kv head for a decoding launch whose workgroups share the splits out themselves (0: the grid is
// (sequence, kv head, split)): as many as keep the launch within MAX_DECODE_BLOCKS workgroups, or, where that
// is less than two a sequence, LQ_UNITS_A_SEQUENCE a sequence (the workgroups beyond what a compute unit holds
// wait their turn); no more than the sequences have splits of 256 within their bound, and at least two a
// sequence, with which a split length that fits is sure to exist.  Taken for 2 to 64 sequences (a wave's
// lanes) without a window.
#ifndef LQ_UNITS_A_SEQUENCE
#define LQ_UNITS_A_SEQUENCE 4
#endif
static int decode_units(int rows, int nkv, int max_len, int window) {
  if (window > 0 || rows < 2 || rows > 64) return 0;
  const long long bound = (long long)lq_ceil_div(max_len, LQ_DECODE_LENGTH_BUCKET) * LQ_DECODE_LENGTH_BUCKET;
  long long by_cap = MAX_DECODE_BLOCKS / nkv;
  if (by_cap < 2 * rows) by_cap = (long long)LQ_UNITS_A_SEQUENCE * rows;
  const long long by_bound = (long long)rows * (bound / 256);
  const long long units = by_cap < by_bound ? by_cap : by_bound;
  if (units < 2 * rows || units > 65535) return 0;
  // The kernel looks for the split length upwards from (all keys) / (256 units) and finds it before twice
  // that; it gives the search 1 024 steps.
  if (rows * bound / (256 * units) > 512) return 0;
  return (int)units;
}

// The host's check of the search that the kernel's units make for their split length (balanced_item): the tries
// it takes for sequences whose newest positions are `pos[0..rows)`, or -1 if it does not end within
// UNIT_SEARCH_TRIES (which the choice of the units is meant to rule out), or 0 where the launch would not take
// the units' way at all.  The same arithmetic, one sequence after another instead of a lane each.
int lq_attention_unit_tries(const int* pos, int rows, int nkv, int max_len) {
  const int units = decode_units(rows, nkv, max_len, 0);
  if (units <= 0) return 0;
  long long total = 0;
  for (int i = 0; i < rows; ++i) total += pos[i] + 1;
  int k = (int)((total + 256LL * units - 1) / (256LL * units));
  if (k < 1) k = 1;
  for (int tries = 0; tries < UNIT_SEARCH_TRIES; ++tries, ++k) {
    long long cnt = 0;
    for (int i = 0; i < rows; ++i) cnt += splits_with_keys(pos[i], k);
    if (cnt <= units) return tries + 1;
  }
  return -1;
}

// Floats of workspace a launch needs (0 when no row has several shares): enough for either grid, the
// window being unknown here.
long long lq_attention_decode_workspace(int rows, int nh, int nkv, int hd, int max_len) {
  const int nsplit = decode_splits(rows, nkv, hd, max_len);
  const long long classic = nsplit <= 1 ? 0 : (long long)rows * nh * nsplit * (hd + 2);
  const long long shared = (long long)decode_units(rows, nkv, max_len, 0) * nh * (hd + 2);
  return classic > shared ? classic : shared;
}

int lq_attention_decode(const void* q, int ldq, void* out, int ldo, int rows, int nh, int nkv,
                      int hd, const int* row_pos, const int* seq_slot,
                      const int* block_table, int bt_stride, const void* kcache, const void* vcache,
                      float scale, int window, int max_len, float* workspace,
                      long long workspace_floats, int* tickets, long long tickets_n, const void* k_new,
                      const void* v_new, int ldk, int ldv, const float* cs, int uneven, int pieces,
                      long long piece_stride, hipStream_t stream) {
  DecodeArgs a;
  a.pieces = pieces;
  a.piece_stride = piece_stride;
  if (pieces > 1) {
    LQ_REQUIRE(cs != nullptr, "attention: pieces of q, k and v are taken by the launch that rotates them only");
    LQ_REQUIRE(pieces <= 64 && piece_stride > 0 && piece_stride % 4 == 0 && ldq % 4 == 0,
               "attention: %d pieces %lld floats apart with rows of %d floats are not taken", pieces, piece_stride, ldq);
  }
  a.q = (const bf16_t*)q;
  a.ldq = ldq;
  a.out = (bf16_t*)out;
  a.ldo = ldo;
  a.nh = nh;
  a.nkv = nkv;
  a.group = nh / nkv;
  a.row_pos = row_pos;
  a.seq_slot = seq_slot;
  a.block_table = block_table;
  a.bt_stride = bt_stride;
  a.kcache = (const bf16_t*)kcache;
  a.vcache = (const bf16_t*)vcache;
  a.scale_log2 = scale * 1.44269504088896340736f;
  a.window = window;
  a.batch = rows;
  a.part_o = nullptr;
  a.part_ml = nullptr;
  a.units = 0;
  a.tickets = tickets;
  a.k_new = (const bf16_t*)k_new;
  a.v_new = (const bf16_t*)v_new;
  a.ldk = ldk;
  a.ldv = ldv;
  a.cs = cs;
  if (cs != nullptr) {
    LQ_REQUIRE(hd % 64 == 0 && k_new && v_new && ldk >= nkv * hd && ldv >= nkv * hd,
               "attention: the folded rotation needs a decoding step, a head size that is a multiple of 64 and the step's keys and values");
    LQ_REQUIRE(((uintptr_t)cs % 16) == 0, "attention: the cos/sin table must be 16-byte aligned");
  }
  LQ_REQUIRE(max_len > 0, "attention: decoding needs the longest sequence length");
  a.nsplit = decode_splits(rows, nkv, hd, max_len);
  a.units = uneven ? decode_units(rows, nkv, max_len, window) : 0;  // (by the bound in 1 024s, as everything here)
  // Up to 256 keys a launch needs no workspace and no counters: where none are given, its rows stay whole.
  if (a.units == 0 && a.nsplit > 1 && max_len <= 4 * BS &&
      (workspace == nullptr || workspace_floats < lq_attention_decode_workspace(rows, nh, nkv, hd, max_len) || tickets == nullptr ||
       tickets_n < (long long)rows * nkv))
    a.nsplit = 1;
  if (a.units > 0 || a.nsplit > 1) {
    const long long need = a.units > 0 ? (long long)a.units * nh * (hd + 2) : lq_attention_decode_workspace(rows, nh, nkv, hd, max_len);
    LQ_REQUIRE(workspace != nullptr && workspace_floats >= need,
               "attention: workspace of %lld floats needed, %lld given", need, workspace_floats);
    LQ_REQUIRE(tickets != nullptr && tickets_n >= (long long)rows * nkv,
               "attention: %lld ticket counters needed for %d rows and %d kv heads, %lld given",
               (long long)rows * nkv, rows, nkv, tickets_n);
    a.part_o = workspace;
    a.part_ml = workspace + (a.units > 0 ? (long long)a.units : (long long)rows * a.nsplit) * nh * hd;
    if ((uintptr_t)workspace % 8 != 0) a.units = 0, a.nsplit = 1;  // (partial results go in pairs: rows stay whole)
  }
  const long long pairs = (long long)rows * nkv;
  a.narrow_splits = pairs < lq_compute_units() ? (int)(lq_compute_units() / pairs) : 1;
  if (a.narrow_splits > a.nsplit) a.narrow_splits = a.nsplit;  // (no row in more shares than the grid has for it)
  a.long_from = 2 * pairs > lq_compute_units() && a.nsplit > 1 ? many_rows(pairs, hd).from : 0;
  switch (hd) {
    case 32: return launch<32>(a, stream);
    case 64: return launch<64>(a, stream);
    case 96: return launch<96>(a, stream);
    case 128: return launch<128>(a, stream);
    case 192: return launch<192>(a, stream);
    case 256: return launch<256>(a, stream);
  }
  lq_set_error("attention: head size %d has no matrix-core kernel", hd);
  return -1;
}
