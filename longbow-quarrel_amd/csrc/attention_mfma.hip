// Causal grouped-query attention over the paged bfloat16 cache on the matrix cores.
//
// One wavefront owns 16 query columns and walks its keys in chunks of 32.  The score tile is
// computed transposed, S^T[key][q] = K . Q^T, so that after the softmax each lane already holds
// the probabilities of one query column in the layout the second product wants as its B operand
// (O^T[d][q] += V^T[d][key] . P^T[key][q]); nothing goes through LDS.  The cache stores V
// transposed per block for exactly this read: V[block][kv head][d][offset].
//
//   v_mfma_f32_16x16x32_bf16: lane l gives A[row l%16][k (l/16)*8 .. +8], B[col l%16][same k],
//   receives D[(l/16)*4 + e][l%16].
//   First product: A = 16 keys x 32 of head_dim, B = 16 queries x the same 32.
//   Second product: its 32 k are keys; MFMA k index (l/16)*8 + j stands for key
//   (l/16)*4 + j of the chunk's first 16 keys when j < 4, else 16 + (l/16)*4 + (j - 4):
//   the keys whose scores lane l already holds.
//
// Softmax statistics, scores and the output accumulator are 32-bit; probabilities are rounded to
// bfloat16 only as MFMA operands (their sum is taken before rounding).
//
// Prompts: a wave owns QT tiles of 16 consecutive rows of one sequence for one query head and reuses every key/value
// fragment it loads for all of them; the waves of a block are the query heads of one kv head over the same rows, so that they read the
// same keys at the same time.  Chunks are aligned to absolute positions.  Single tokens: attention_decode.hip.
#include "attention_mfma.h"

namespace {

// Which key of a 32-key chunk row r of score tile j stands for: the rows are dealt out so that the
// eight probabilities a lane ends up with (rows (lane/16)*4 + e of both tiles) belong to eight
// consecutive keys, (lane/16)*8 .. +7: the second product then takes its V^T operand as one
// 16-byte run of keys.
__device__ inline int chunk_key(int j, int r) { return (r >> 2) * 8 + j * 4 + (r & 3); }

// One chunk of 32 keys for one query tile: from the raw score tiles s[2] (S^T, lane holds rows
// (lane/16)*4 + e of each 16-row tile, i.e. keys (lane/16)*8 + 4 j + e, for column lane%16) to the packed probabilities, updating the
// running maximum m (log2 domain, scores scaled by c = scale * log2 e) and normaliser share l.
// Returns the factor the output accumulator has to be multiplied with (1 if the maximum stayed).
// `masked` is wave-uniform: false when every key of the chunk is visible to every column.
__device__ inline float softmax_chunk(const f32x4 (&s)[2], float c, bool masked, bool col_valid, int t0, int lo,
                                      int pos, float& m, float& l, u32x4& pw) {
  const int g = (threadIdx.x & 63) >> 4;
  float sv[8];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) sv[j * 4 + e] = s[j][e];
  if (masked) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int t = t0 + g * 8 + j * 4 + e;
        if (!(col_valid && t >= lo && t <= pos)) sv[j * 4 + e] = -INFINITY;
      }
  }
  float cmax = fmaxf(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3])), fmaxf(fmaxf(sv[4], sv[5]), fmaxf(sv[6], sv[7])));
  cmax = rows_max(cmax) * c;  // c > 0: scaling commutes with the maximum
  float alpha = 1.0f;
  if (__any(cmax > m + RESCALE_SLACK)) {  // (false for -inf against -inf, true for anything against -inf)
    const float m_new = fmaxf(m, cmax);
    alpha = fast_exp2(m - ((m_new == -INFINITY) ? 0.f : m_new));
    l *= alpha;
    m = m_new;
  }
  const float m_safe = (m == -INFINITY) ? 0.f : m;  // a column with no key yet
  float psum = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    sv[i] = fast_exp2(fmaf(sv[i], c, -m_safe));  // -inf stays -inf, 2^-inf = 0
    psum += sv[i];
  }
  l += psum;
  pw[0] = pack_bf16(sv[0], sv[1]);
  pw[1] = pack_bf16(sv[2], sv[3]);
  pw[2] = pack_bf16(sv[4], sv[5]);
  pw[3] = pack_bf16(sv[6], sv[7]);
  return alpha;
}

struct AttnArgs {
  const bf16_t* q;
  int ldq;
  bf16_t* out;
  int ldo;
  int nh, nkv;
  const int* row_pos;
  const int* seq_slot;
  const int* cu_rows;
  const int* block_table;
  int bt_stride;
  const bf16_t* kcache;
  const bf16_t* vcache;
  float scale_log2;  // scale * log2(e)
  int window;
  int batch;
};

// What a wave carries for each of its QT query tiles.  Column c = lane % 16 of tile qt is valid if
// valid[qt]; its position is pos[qt], its first key lo[qt].  o[qt][dt][e] is the unnormalised
// O^T[dt*16 + (lane/16)*4 + e][c], m the running maximum (log2 domain), l this lane's share of
// the normaliser (to be summed over lane/16).
template <int HD, int QT>
struct QTiles {
  bf16x8 q[QT][HD / 32];
  f32x4 o[QT][HD / 16];
  float m[QT], l[QT];
  bool valid[QT];
  int pos[QT], lo[QT];
  int last_key[QT];   // largest position any column of the tile may see (wave-uniform)
  int first_key[QT];  // smallest (wave-uniform)
  int free_to[QT];    // chunks that end at or before this key and start at or after free_from are
  int free_from[QT];  //   visible to every column: no masking needed (wave-uniform; free_to = -1: never)
};

template <int HD, int QT>
__device__ inline void init_tiles(QTiles<HD, QT>& w) {
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) w.o[qt][dt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    w.m[qt] = -INFINITY;
    w.l[qt] = 0.f;
  }
}

// ------------------------------------------------------------------ rows (prompts)
// Block = NW waves = NW query heads of one kv head over the same QT * 16 rows.  The block walks
// the keys one cache block (64 positions) at a time: all threads copy the block's K [64][HD] and
// V^T [HD][64] from memory into padded LDS (next block's copy in registers while the current one is
// multiplied), and every wave reads its MFMA operands from there, so a key is fetched once for
// all the heads that share it.  LDS rows are padded (K: +16 bytes, V^T: +16 bytes) so that the
// operand reads of a quarter wave fall into distinct banks.  Keys lie in LDS in the order the score
// tiles read them (chunk_key).
template <int HD>
struct RowsLds {
  static constexpr int K_STRIDE = HD * 2 + 16;   // bytes per key row
  static constexpr int V_STRIDE = BS * 2 + 16;   // bytes per d row
  static constexpr int K_BYTES = BS * K_STRIDE;
  static constexpr int V_BYTES = HD * V_STRIDE;
  static constexpr int STAGE = K_BYTES + V_BYTES;
  static constexpr int PIECES = HD * 8;          // 16-byte pieces of K (and of V^T) in one cache block
};

template <int HD, int QT, int HW, int RT>
__global__ __launch_bounds__(HW * RT * 64, (HD <= 128 && HW * RT > 1 ? 2 : 1)) void attn_rows_kernel(AttnArgs a, int heads_per_block_group, int tiles, int units) {
  using L = RowsLds<HD>;
  constexpr int NW = HW * RT;  // wave = row group * HW + head: HW query heads of one kv head, RT groups of QT row tiles
  constexpr int ROWS = QT * 16 * RT;
  constexpr int THREADS = NW * 64;
  constexpr int PER_THREAD = (L::PIECES + THREADS - 1) / THREADS;  // pieces of K, and of V, per thread
  constexpr bool EARLY = PER_THREAD <= 8;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  // Tasks (a tile of ROWS rows, counted sequence by sequence, for one group of heads) in descending
  // order of their keys: late tiles first.  Workgroups i, i + units, i + 2 units, ... land on the
  // same compute unit, so the tasks are dealt out in a snake (0 .. units-1, then back): a unit's
  // heavy task gets a light partner and the units finish together.
  const int per_tile = gridDim.x / tiles;  // groups of heads
  const int round = blockIdx.x / units, place = blockIdx.x % units;
  int task = round * units + ((round & 1) ? units - 1 - place : place);
  if ((round + 1) * units > (int)gridDim.x) task = blockIdx.x;  // the last, partial round stays in order
  const int head_group = task % per_tile;
  int t = tiles - 1 - task / per_tile, b = 0, r0 = -1, nrows = 0;
  for (; b < a.batch; ++b) {
    const int begin = a.cu_rows[b], n = a.cu_rows[b + 1] - begin;
    const int tiles = (n + ROWS - 1) / ROWS;
    if (t < tiles) {
      r0 = begin + t * ROWS;
      nrows = min(ROWS, n - t * ROWS);
      break;
    }
    t -= tiles;
  }
  if (r0 < 0) return;  // the whole block
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c16 = lane & 15, g = lane >> 4;
  const int G = a.nh / a.nkv;
  // blockIdx.y = kv head * groups + group, a group being HW consecutive query heads of the kv head
  const int kvh = head_group / heads_per_block_group;
  const int hq = (head_group % heads_per_block_group) * HW + wave % HW;
  const int tile0 = (wave / HW) * QT;  // this wave's first row tile within the block
  const bool wave_active = hq < G;  // an idle wave still copies and meets the barriers
  const int h = kvh * G + min(hq, G - 1);
  const int* table = a.block_table + (long long)a.seq_slot[b] * a.bt_stride;
  const int p0 = a.row_pos[r0];

  QTiles<HD, QT> w;
  init_tiles<HD, QT>(w);
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int rows_here = min(16, nrows - (tile0 + qt) * 16);  // may be <= 0: the tile is empty
    const int rc = (tile0 + qt) * 16 + min(c16, max(rows_here, 1) - 1);
    const int row = r0 + min(rc, nrows - 1);
    w.valid[qt] = wave_active && c16 < rows_here;
    w.pos[qt] = p0 + min(rc, nrows - 1);
    w.lo[qt] = (a.window > 0 && w.pos[qt] >= a.window) ? w.pos[qt] - a.window + 1 : 0;
    const int first_pos = p0 + min((tile0 + qt) * 16, nrows - 1);
    w.last_key[qt] = (wave_active && rows_here > 0) ? p0 + (tile0 + qt) * 16 + rows_here - 1 : -1;
    w.first_key[qt] = (a.window > 0 && first_pos >= a.window) ? first_pos - a.window + 1 : 0;
    // keys up to the tile's first row's position and from its last row's window start on are visible to
    // all of its columns (those past a partial tile's rows run as copies of its last row, never stored)
    const int last_pos = p0 + (tile0 + qt) * 16 + rows_here - 1;
    w.free_to[qt] = (wave_active && rows_here > 0) ? first_pos : -1;
    w.free_from[qt] = (a.window > 0 && last_pos >= a.window) ? last_pos - a.window + 1 : 0;
    const bf16_t* qr = a.q + (long long)row * a.ldq + h * HD + g * 8;
#pragma unroll
    for (int kk = 0; kk < HD / 32; ++kk) w.q[qt][kk] = as_bf16x8(*(const u32x4*)(qr + kk * 32));
  }
  const int t_end = p0 + nrows - 1;  // the last key anyone here sees, and the last one written
  const int lo_tile = (a.window > 0 && p0 >= a.window) ? p0 - a.window + 1 : 0;
  const int blk_first = lo_tile / BS, blk_last = t_end / BS;

  u32x4 rk[PER_THREAD], rv[PER_THREAD];
  auto fetch = [&](int lb) {
    const long long blk = table[lb];
    const bf16_t* kb = a.kcache + (blk * a.nkv + kvh) * (long long)(BS * HD);
    const bf16_t* vb = a.vcache + (blk * a.nkv + kvh) * (long long)(HD * BS);
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
      const int pc = tid + i * THREADS;
      if (pc < L::PIECES) {
        rk[i] = *(const u32x4*)(kb + pc * 8);
        rv[i] = *(const u32x4*)(vb + pc * 8);
      }
    }
  };
  auto stash = [&](int lb, unsigned char* stage) {
    // values of keys that were never written must not reach the product (0 * garbage may be NaN)
    const int base_key = lb * BS;
    const bool tail = base_key + BS - 1 > t_end;
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
      const int pc = tid + i * THREADS;
      if (pc < L::PIECES) {
        // keys go to the row their score tile reads them from: row 16 j + r holds key chunk_key(j, r)
        const int key = pc / (HD / 8), part = pc % (HD / 8);
        const int k32 = key & 31;
        const int krow = (key & 32) + ((k32 >> 2) & 1) * 16 + (k32 >> 3) * 4 + (k32 & 3);
        *(u32x4*)(stage + krow * L::K_STRIDE + part * 16) = rk[i];
        const int d = pc >> 3, vpart = pc & 7;
        u32x4 v = rv[i];
        if (tail) {
          const int k0 = base_key + vpart * 8;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (k0 + 2 * e > t_end) v[e] &= 0xffff0000u;
            if (k0 + 2 * e + 1 > t_end) v[e] &= 0x0000ffffu;
          }
        }
        *(u32x4*)(stage + L::K_BYTES + d * L::V_STRIDE + vpart * 16) = v;
      }
    }
  };

  fetch(blk_first);
  stash(blk_first, smem);
  __syncthreads();
  for (int lb = blk_first; lb <= blk_last; ++lb) {
    unsigned char* cur = smem + ((lb - blk_first) & 1) * L::STAGE;
    unsigned char* nxt = smem + ((lb - blk_first + 1) & 1) * L::STAGE;
    const bool more = lb < blk_last;
    // The next block's loads are on their way during this block's products where a thread's share
    // of them is small enough to stay in registers meanwhile; else they follow the products.
    if (EARLY && more) fetch(lb + 1);
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int t0 = lb * BS + half * 32;
      if (t0 > t_end) break;
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        if (t0 > w.last_key[qt] || t0 + 31 < w.first_key[qt]) continue;  // nothing of this chunk is visible
        f32x4 sc[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          sc[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
          const unsigned char* kr = cur + (half * 32 + 16 * j + c16) * L::K_STRIDE + g * 16;
#pragma unroll
          for (int kk = 0; kk < HD / 32; ++kk)
            sc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(*(const u32x4*)(kr + kk * 64)), w.q[qt][kk],
                                                            sc[j], 0, 0, 0);
        }
        const bool masked = !(t0 + 31 <= w.free_to[qt] && t0 >= w.free_from[qt]);
        u32x4 pw;
        const float alpha = softmax_chunk(sc, a.scale_log2, masked, w.valid[qt], t0, w.lo[qt], w.pos[qt], w.m[qt],
                                          w.l[qt], pw);
        const bf16x8 pb = as_bf16x8(pw);
        if (!__all(alpha == 1.0f)) {  // the maximum moved for some column: rescale what has been summed
#pragma unroll
          for (int dt = 0; dt < HD / 16; ++dt)
#pragma unroll
            for (int e = 0; e < 4; ++e) w.o[qt][dt][e] *= alpha;
        }
#pragma unroll
        for (int dt = 0; dt < HD / 16; ++dt) {
          const u32x4 vv = *(const u32x4*)(cur + L::K_BYTES + (dt * 16 + c16) * L::V_STRIDE + half * 64 + g * 16);
          w.o[qt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(vv), pb, w.o[qt][dt], 0, 0, 0);
        }
      }
    }
    // Nobody reads nxt: its last readers passed the barrier below one round ago.
    if (more) {
      if (!EARLY) fetch(lb + 1);
      stash(lb + 1, nxt);
    }
    __syncthreads();
  }
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    float l = w.l[qt];
    l = rows_sum(l);
    if (!w.valid[qt]) continue;
    const float inv = 1.0f / l;
    bf16_t* orow = a.out + (long long)(r0 + (tile0 + qt) * 16 + c16) * a.ldo + h * HD + g * 4;
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) {
      u32x2 ww;
      ww[0] = pack_bf16(w.o[qt][dt][0] * inv, w.o[qt][dt][1] * inv);
      ww[1] = pack_bf16(w.o[qt][dt][2] * inv, w.o[qt][dt][3] * inv);
      *(u32x2*)(orow + dt * 16) = ww;
    }
  }
}

template <int HD, int QT, int HW, int RT>
int launch_rows(const AttnArgs& a, int rows, int groups, hipStream_t stream) {
  using L = RowsLds<HD>;
  constexpr int ROWS = QT * 16 * RT, NW = HW * RT;
  const size_t smem = 2 * (size_t)L::STAGE;
  auto kernel = attn_rows_kernel<HD, QT, HW, RT>;
  static bool configured = false;
  if (!configured && smem > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) {
      lq_set_error("attention: cannot reserve %zu bytes of LDS: %s", smem, hipGetErrorString(e));
      return -2;
    }
    configured = true;
  }
  const int tiles = lq_ceil_div(rows, ROWS) + a.batch;  // an upper bound: a sequence's last tile may be partial
  kernel<<<dim3(tiles * a.nkv * groups), NW * 64, smem, stream>>>(a, groups, tiles, lq_compute_units());
  LQ_CHECK_LAUNCH("attention(mfma rows)");
  return 0;
}

// ------------------------------------------------------------------ rows, 32 x 32 score tiles
// The same launch shape with the wider product, v_mfma_f32_32x32x16_bf16: a wave owns 32 consecutive
// rows of one query head, a block is the HW query heads of one kv head over the same 32 rows.  A K or
// V^T fragment read from LDS (1 KB) now feeds a product of 32 x 32 x 16 instead of 16 x 16 x 32: half
// the LDS traffic a flop, which is what bounded the narrower tile.
//   lane l gives A[row l%32][k (l/32)*8 .. +8] and B[col l%32][the same k]; it receives
//   D[(e/4)*8 + (l/32)*4 + e%4][l%32], e < 16.
//   First product: A = 32 keys x 16 of head_dim (LDS), B = 32 rows x the same 16 (registers):
//   S^T[key][row]; lane (row r, half h) holds keys (e/4)*8 + 4 h + e%4 of the chunk.
//   Second product, two steps of 16 keys: step s takes the lane's probabilities e = 8 s .. 8 s + 7 as
//   they are, so its k index 8 h + j stands for key 16 s + (j/4)*8 + 4 h + j%4; V^T lies in LDS with
//   the keys of every 16 in the order [0-3][8-11][4-7][12-15], which makes those eight one 16-byte run.
typedef float f32x16 __attribute__((ext_vector_type(16)));

// With KS = 2 a head's 32 rows are shared by two waves that take the first and the second 32 keys of every
// cache block and add their results up through LDS at the end: a tile's time is set by its last row tile's
// walk through all the keys before it, and on a short prompt, where the chip holds every tile at once, that
// walk is the launch's time.
template <int HD, int HW, int KS>
__global__ __launch_bounds__(HW * KS * 64, KS == 2 ? 1 : 2) void attn_rows32_kernel(AttnArgs a, int heads_per_block_group,
                                                                                   int tiles, int units) {
  using L = RowsLds<HD>;
  constexpr int ROWS = 32, THREADS = HW * KS * 64;
  constexpr int MERGE_FLOATS = HD / 32 * 16 * 64 + 2 * 64;  // a wave's accumulators, maxima and normaliser shares
  static_assert(KS == 1 || (KS == 2 && HW * MERGE_FLOATS * 4 <= 2 * L::STAGE), "the second waves' results fit the stages");
  constexpr int PER_THREAD = (L::PIECES + THREADS - 1) / THREADS;  // pieces of K, and of V, per thread
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  // tasks as in attn_rows_kernel: late (heavy) tiles first, dealt out over the compute units in a snake
  const int per_tile = gridDim.x / tiles;
  const int round = blockIdx.x / units, place = blockIdx.x % units;
  int task = round * units + ((round & 1) ? units - 1 - place : place);
  if ((round + 1) * units > (int)gridDim.x) task = blockIdx.x;
  const int head_group = task % per_tile;
  int t = tiles - 1 - task / per_tile, b = 0, r0 = -1, nrows = 0;
  for (; b < a.batch; ++b) {
    const int begin = a.cu_rows[b], n = a.cu_rows[b + 1] - begin;
    const int tiles_b = (n + ROWS - 1) / ROWS;
    if (t < tiles_b) {
      r0 = begin + t * ROWS;
      nrows = min(ROWS, n - t * ROWS);
      break;
    }
    t -= tiles_b;
  }
  if (r0 < 0) return;  // the whole block
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c32 = lane & 31, hf = lane >> 5;
  const int head_slot = wave % HW, ks = wave / HW;  // (ks: which 32 keys of a cache block, with KS = 2)
  const int G = a.nh / a.nkv;
  const int kvh = head_group / heads_per_block_group;
  const int hq = (head_group % heads_per_block_group) * HW + head_slot;
  const bool wave_active = hq < G;  // an idle wave still copies and meets the barriers
  const int h = kvh * G + min(hq, G - 1);
  const int* table = a.block_table + (long long)a.seq_slot[b] * a.bt_stride;
  const int p0 = a.row_pos[r0];

  // this lane's row (column of the score tile)
  const int rc = min(c32, nrows - 1);
  const bool valid = wave_active && c32 < nrows;
  const int pos = p0 + rc;
  const int lo = (a.window > 0 && pos >= a.window) ? pos - a.window + 1 : 0;
  const int last_key = wave_active ? p0 + nrows - 1 : -1;                       // wave-uniform
  const int first_key = (a.window > 0 && p0 >= a.window) ? p0 - a.window + 1 : 0;
  // keys up to the first row's position and from the last row's window start on are visible to all 32 rows
  // (the columns past a partial tile run as copies of its last row and are never stored: they see these keys too)
  const int free_to = wave_active ? p0 : -1;
  const int free_from = (a.window > 0 && p0 + nrows - 1 >= a.window) ? p0 + nrows - 1 - a.window + 1 : 0;
  bf16x8 q[HD / 16];
  {
    const bf16_t* qr = a.q + (long long)(r0 + rc) * a.ldq + h * HD + hf * 8;
#pragma unroll
    for (int kk = 0; kk < HD / 16; ++kk) q[kk] = as_bf16x8(*(const u32x4*)(qr + kk * 16));
  }
  f32x16 o[HD / 32];
#pragma unroll
  for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[dt][e] = 0.f;
  float m = -INFINITY, l = 0.f;  // running maximum of the row (log2 domain); this lane's share of the normaliser

  const int t_end = p0 + nrows - 1;  // the last key anyone here sees, and the last one written
  const int blk_first = first_key / BS, blk_last = t_end / BS;

  u32x4 rk[PER_THREAD], rv[PER_THREAD];
  auto fetch = [&](int lb) {
    const long long blk = table[lb];
    const bf16_t* kb = a.kcache + (blk * a.nkv + kvh) * (long long)(BS * HD);
    const bf16_t* vb = a.vcache + (blk * a.nkv + kvh) * (long long)(HD * BS);
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
      const int pc = tid + i * THREADS;
      if (pc < L::PIECES) {
        rk[i] = *(const u32x4*)(kb + pc * 8);
        rv[i] = *(const u32x4*)(vb + pc * 8);
      }
    }
  };
  auto stash = [&](int lb, unsigned char* stage) {
    // values of keys that were never written must not reach the product (0 * garbage may be NaN)
    const int base_key = lb * BS;
    const bool tail = base_key + BS - 1 > t_end;
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
      const int pc = tid + i * THREADS;
      if (pc < L::PIECES) {
        const int key = pc / (HD / 8), part = pc % (HD / 8);  // keys in their own order: row = key
        *(u32x4*)(stage + key * L::K_STRIDE + part * 16) = rk[i];
        const int d = pc >> 3, vpart = pc & 7;  // eight keys of one d: 8 vpart .. + 7
        u32x4 v = rv[i];
        if (tail) {
          const int k0 = base_key + vpart * 8;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (k0 + 2 * e > t_end) v[e] &= 0xffff0000u;
            if (k0 + 2 * e + 1 > t_end) v[e] &= 0x0000ffffu;
          }
        }
        // within every 16 keys the order in LDS is [0-3][8-11][4-7][12-15]
        unsigned char* vrow = stage + L::K_BYTES + d * L::V_STRIDE + (vpart >> 1) * 32;
        const int odd = vpart & 1;
        *(u32x2*)(vrow + (odd ? 8 : 0)) = (u32x2){v[0], v[1]};
        *(u32x2*)(vrow + (odd ? 24 : 16)) = (u32x2){v[2], v[3]};
      }
    }
  };

  fetch(blk_first);
  stash(blk_first, smem);
  __syncthreads();
  for (int lb = blk_first; lb <= blk_last; ++lb) {
    unsigned char* cur = smem + ((lb - blk_first) & 1) * L::STAGE;
    unsigned char* nxt = smem + ((lb - blk_first + 1) & 1) * L::STAGE;
    const bool more = lb < blk_last;
    if (more) fetch(lb + 1);  // on their way during this block's products
#pragma unroll
    for (int hh = 0; hh < 2 / KS; ++hh) {
      const int half = KS == 2 ? ks : hh;
      const int t0 = lb * BS + half * 32;
      if (t0 > t_end) break;
      if (t0 > last_key || t0 + 31 < first_key) continue;  // nothing of this chunk is visible to this wave
      f32x16 sc;
#pragma unroll
      for (int e = 0; e < 16; ++e) sc[e] = 0.f;
      const unsigned char* kr = cur + (half * 32 + c32) * L::K_STRIDE + hf * 16;
      const unsigned char* vr = cur + L::K_BYTES + c32 * L::V_STRIDE + half * 64 + hf * 16;
      // All of the half's K fragments are asked for before the first product, and its V^T fragments as soon
      // as the products have been issued, so that they arrive during the products and the softmax: a wave
      // that asks for each fragment just before its product waits out the LDS latency sixteen times a half.
      u32x4 kf[HD / 16], vf[2][HD / 32];
#pragma unroll
      for (int kk = 0; kk < HD / 16; ++kk) kf[kk] = *(const u32x4*)(kr + kk * 32);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < HD / 16; ++kk)
        sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(kf[kk]), q[kk], sc, 0, 0, 0);
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
        for (int dt = 0; dt < HD / 32; ++dt) vf[s2][dt] = *(const u32x4*)(vr + dt * 32 * L::V_STRIDE + s2 * 32);
      __builtin_amdgcn_sched_barrier(0);
      const bool masked = !(t0 + 31 <= free_to && t0 >= free_from);
      if (masked) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int tk = t0 + (e >> 2) * 8 + hf * 4 + (e & 3);
          if (!(valid && tk >= lo && tk <= pos)) sc[e] = -INFINITY;
        }
      }
      float cmax = sc[0];
#pragma unroll
      for (int e = 1; e < 16; ++e) cmax = fmaxf(cmax, sc[e]);
      {  // the row's other sixteen keys are in the lane 32 places away
        auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(cmax), __float_as_uint(cmax), false, false);
        cmax = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
      }
      cmax *= a.scale_log2;  // the scale is positive: it commutes with the maximum
      if (__any(cmax > m + RESCALE_SLACK)) {  // some row's maximum moved far: rescale what has been summed
        const float m_new = fmaxf(m, cmax);
        const float alpha = fast_exp2(m - ((m_new == -INFINITY) ? 0.f : m_new));
        l *= alpha;
        m = m_new;
#pragma unroll
        for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
          for (int e = 0; e < 16; ++e) o[dt][e] *= alpha;
      }
      const float m_safe = (m == -INFINITY) ? 0.f : m;  // a row with no key yet
      float psum = 0.f;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        sc[e] = fast_exp2(fmaf(sc[e], a.scale_log2, -m_safe));  // -inf stays -inf, 2^-inf = 0
        psum += sc[e];
      }
      l += psum;
      u32x4 pw[2];
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
        for (int j = 0; j < 4; ++j) pw[s2][j] = pack_bf16(sc[8 * s2 + 2 * j], sc[8 * s2 + 2 * j + 1]);
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
        for (int dt = 0; dt < HD / 32; ++dt)
          o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(vf[s2][dt]), as_bf16x8(pw[s2]), o[dt], 0, 0, 0);
    }
    // Nobody reads nxt: its last readers passed the barrier below one round ago.
    if (more) stash(lb + 1, nxt);
    __syncthreads();
  }
  if constexpr (KS == 2) {
    // the second waves' sums go to the first through LDS (everyone is past the last stage's reads)
    float* mine = (float*)smem + head_slot * MERGE_FLOATS;
    if (ks == 1) {
#pragma unroll
      for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) mine[(dt * 16 + e) * 64 + lane] = o[dt][e];
      mine[HD / 32 * 16 * 64 + lane] = m;
      mine[HD / 32 * 16 * 64 + 64 + lane] = l;
    }
    __syncthreads();
    if (ks == 1) return;
    const float m1 = mine[HD / 32 * 16 * 64 + lane], l1 = mine[HD / 32 * 16 * 64 + 64 + lane];
    const float m_all = fmaxf(m, m1);
    const float m_safe = (m_all == -INFINITY) ? 0.f : m_all;
    const float f0 = fast_exp2(m - m_safe), f1 = fast_exp2(m1 - m_safe);  // 2^-inf = 0: a wave that saw no key
    l = l * f0 + l1 * f1;
#pragma unroll
    for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[dt][e] = o[dt][e] * f0 + mine[(dt * 16 + e) * 64 + lane] * f1;
  }
  {
    auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    l = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
  }
  if (!valid) return;
  const float inv = 1.0f / l;
  bf16_t* orow = a.out + (long long)(r0 + c32) * a.ldo + h * HD + hf * 4;
#pragma unroll
  for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {  // d = dt*32 + g4*8 + hf*4 + (0..3)
      u32x2 ww;
      ww[0] = pack_bf16(o[dt][g4 * 4 + 0] * inv, o[dt][g4 * 4 + 1] * inv);
      ww[1] = pack_bf16(o[dt][g4 * 4 + 2] * inv, o[dt][g4 * 4 + 3] * inv);
      *(u32x2*)(orow + dt * 32 + g4 * 8) = ww;
    }
}

template <int HD, int HW, int KS>
int launch_rows32(const AttnArgs& a, int rows, int groups, hipStream_t stream) {
  using L = RowsLds<HD>;
  const size_t smem = 2 * (size_t)L::STAGE;
  auto kernel = attn_rows32_kernel<HD, HW, KS>;
  static bool configured = false;
  if (!configured && smem > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) {
      lq_set_error("attention: cannot reserve %zu bytes of LDS: %s", smem, hipGetErrorString(e));
      return -2;
    }
    configured = true;
  }
  const int tiles = lq_ceil_div(rows, 32) + a.batch;  // an upper bound: a sequence's last tile may be partial
  kernel<<<dim3(tiles * a.nkv * groups), HW * KS * 64, smem, stream>>>(a, groups, tiles, lq_compute_units());
  LQ_CHECK_LAUNCH("attention(mfma rows, 32 x 32)");
  return 0;
}

template <int HD>
int launch(const AttnArgs& a, int rows, hipStream_t stream) {
  const int G = a.nh / a.nkv;
  constexpr int QT = HD <= 64 ? 4 : (HD <= 128 ? 2 : 1);
  constexpr int QT2 = QT > 1 ? QT / 2 : 1;  // with two row groups of waves: the same rows a block, half a wave
  if constexpr (HD % 32 == 0 && HD <= 128) {
    // The 32 x 32 score tile (its accumulators fit up to this head size) reads half as much from LDS for a
    // product, with half as many waves on a compute unit to hide one wave's softmax behind another's
    // products.  As measured (32 heads over 8): at head size 64 it wins at every length (46 against 68 us at
    // 2 048 tokens, 353 against 429 at 8 192); at head size 128 it wins or ties at every length too (one
    // sequence of 256 tokens 16.7 against 16.6 us, of 1 000 tokens 33.8 against 34.2, of 2 048 tokens 65.9
    // against 67.7, of 8 192 tokens 612 against 682; sixteen sequences of 512 tokens 79 against 84, eight of 300
    // tokens 29.0 against 28.5) since its fragments are asked for early and partial tiles take the unmasked
    // path below the diagonal.  With one head a kv head a workgroup would be one wave that stages a whole
    // cache block through its own registers: then the narrow tiles stay for head sizes above 64.
    // Two waves a head (each half of every cache block's keys) where the workgroups would not even be one a
    // compute unit: the chip then holds twice the waves and a tile's walk through its keys takes half as
    // long (one sequence of 1 000 tokens 32.6 -> 28.5 us, of 700 tokens 24.8 -> 22.2).  With more workgroups
    // than that they would run one after the other, eight waves each, where two of four waves run side by
    // side (2 048 tokens 64.8 -> 72.8 us, 8 192 tokens 597 -> 648).
    const int hw = G >= 4 ? 4 : (G >= 2 ? 2 : 1);
    const bool two = (long long)lq_ceil_div(rows, 32) * a.nkv * lq_ceil_div(G, hw) <= lq_compute_units();
    if (G >= 4)
      return two ? launch_rows32<HD, 4, 2>(a, rows, lq_ceil_div(G, 4), stream)
                 : launch_rows32<HD, 4, 1>(a, rows, lq_ceil_div(G, 4), stream);
    if (G >= 2)
      return two ? launch_rows32<HD, 2, 2>(a, rows, lq_ceil_div(G, 2), stream)
                 : launch_rows32<HD, 2, 1>(a, rows, lq_ceil_div(G, 2), stream);
    if constexpr (HD <= 64)
      return two ? launch_rows32<HD, 1, 2>(a, rows, 1, stream) : launch_rows32<HD, 1, 1>(a, rows, 1, stream);
    else
      return launch_rows<HD, QT, 1, 1>(a, rows, 1, stream);
  } else {
    if (G >= 4) return launch_rows<HD, QT2, 4, 2>(a, rows, lq_ceil_div(G, 4), stream);
    if (G >= 2) return launch_rows<HD, QT, 2, 1>(a, rows, lq_ceil_div(G, 2), stream);
    return launch_rows<HD, QT, 1, 1>(a, rows, 1, stream);
  }
}

}  // namespace

bool lq_attention_mfma_accepts(int dtype, int nh, int nkv, int hd, int block_size, int ldq, int ldo,
                               const void* q, const void* out, int decode) {
  if (dtype != LQ_BF16 || block_size != BS) return false;
  if (!(hd == 32 || hd == 64 || hd == 96 || hd == 128 || hd == 192 || hd == 256)) return false;
  if (ldq % 8 != 0 || ldo % 4 != 0 || ((uintptr_t)q % 16) != 0 || ((uintptr_t)out % 8) != 0) return false;
  if (decode && nh / nkv > 16) return false;
  if (nh > 65535 || nkv > 65535) return false;
  return true;
}

int lq_attention_mfma(const void* q, int ldq, void* out, int ldo, int rows, int batch, int nh, int nkv,
                      int hd, const int* row_pos, const int* seq_slot, const int* cu_rows,
                      const int* block_table, int bt_stride, const void* kcache, const void* vcache,
                      float scale, int window, hipStream_t stream) {
  AttnArgs a;
  a.q = (const bf16_t*)q;
  a.ldq = ldq;
  a.out = (bf16_t*)out;
  a.ldo = ldo;
  a.nh = nh;
  a.nkv = nkv;
  a.row_pos = row_pos;
  a.seq_slot = seq_slot;
  a.cu_rows = cu_rows;
  a.block_table = block_table;
  a.bt_stride = bt_stride;
  a.kcache = (const bf16_t*)kcache;
  a.vcache = (const bf16_t*)vcache;
  a.scale_log2 = scale * 1.44269504088896340736f;
  a.window = window;
  a.batch = batch;
  switch (hd) {
    case 32: return launch<32>(a, rows, stream);
    case 64: return launch<64>(a, rows, stream);
    case 96: return launch<96>(a, rows, stream);
    case 128: return launch<128>(a, rows, stream);
    case 192: return launch<192>(a, rows, stream);
    case 256: return launch<256>(a, rows, stream);
  }
  lq_set_error("attention: head size %d has no matrix-core kernel", hd);
  return -1;
}
