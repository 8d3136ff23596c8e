// Steps of single tokens of a bfloat16 run through the windowed attention of attention_sink.hip (the same masks, sinks,
// shaped scores, maps and gates).
//
// A workgroup of four wavefronts takes one row of the step, up to 16 query heads of one key head and one of `splits`
// shares of the keys: the blocks of 64 positions that the row sees, numbered from the kept first ones on, go to the
// wavefronts of all shares in turn, so that at a few thousand keys every wavefront has one.  It asks for all of a block's
// keys and values before it waits for any: what bounds such a step is the chain of round trips to memory, not the bytes
// (tiles that asked for a few bytes of a key row at a time, a product between, and a second launch that merged the
// shares: microseconds before and now, 8 rows, 16 heads: 4 key heads of 128 at 512 keys 20 -> 12, at 1 500 keys under a
// window of 1 024 31 -> 13, with values of 256 and two maps 28 -> 16; one key head of 256 with values of 192 28 -> 21;
// 64 rows at 500 keys 34 -> 19; 2 rows with capped scores and a table of biases 30 -> 15).  The shares of a row meet in its
// last workgroup to finish (a ticket a row and key head; partial results pass the dies' caches as device-scope atomics),
// which adds them up in their order; a caller who gives no tickets gets a second launch that does the same.
//
//   S^T[key][head] = K . Q^T by v_mfma_f32_16x16x32_bf16: lane (c = l % 16, g = l / 16) gives A[c][8 g .. + 8] and B[c][the
//   same] and receives D[4 g + e][c].  Row i of tile j (of a run of 32 keys) is key 8 (i / 4) + 4 j + i % 4: a lane's scores
//   of both tiles are then keys 8 g .. + 7 of its head, which O^T[d][head] += V^T . P^T takes as they are.
// The probabilities stay 32-bit, multiplied in three bfloat16 parts that add up to them exactly (attention_sink_rows.hip).
// Values of positions that were never written count as zero.
#include "attention_sink.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int BLOCK = 64, NW = 4, MAX_SPLITS = 64;

// over the four lanes that share l % 16
__device__ inline float across_max(float x) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ inline float across_sum(float x) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

__device__ inline void publish(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline float published(const float* p) {
  return __hip_atomic_load(const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline float2 published2(const float* p) {  // two neighbours on 8 bytes
  const unsigned long long v = __hip_atomic_load((unsigned long long*)const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return make_float2(__uint_as_float((unsigned)v), __uint_as_float((unsigned)(v >> 32)));
}

struct Shares {
  int splits;
  float* part;   // [row][key head's tile][split]: cols x VD results, then cols maxima and cols sums
  int* tickets;  // [row][key head's tile], zero between launches; or null: a second launch adds the shares up
};

// Which keys a row sees, in blocks of 64 positions, the kept first ones below the window's.
struct Blocks {
  int lo, wstart, kept, n;
};
__device__ inline Blocks blocks_of(const SinkArgs& a, int pos) {
  Blocks b;
  b.lo = first_key(a, pos);
  b.wstart = b.lo / BLOCK * BLOCK;                                // first block of the window
  b.kept = (min(a.keep_first, b.wstart) + BLOCK - 1) / BLOCK;     // blocks of kept keys below it
  b.n = b.kept + pos / BLOCK - b.wstart / BLOCK + 1;
  return b;
}
__device__ inline int live_shares(const Shares& sh, const Blocks& b) {  // shares with a block for some wavefront
  return min(sh.splits, (b.n + NW - 1) / NW);
}

// A workgroup's row and key head's tile: its query heads hbase .. hbase + cols - 1.
struct Heads {
  int kvh, hbase, cols, share_floats;
};
__device__ inline Heads heads_of(const SinkArgs& a) {
  const int group = a.nh / a.nkv, tiles = (group + 15) / 16, kvh = blockIdx.y / tiles;
  const int hbase = kvh * group + blockIdx.y % tiles * 16;
  return {kvh, hbase, min(16, (kvh + 1) * group - hbase), min(16, group) * (a.VD + 2)};
}

// A head's entry (idx: of the tile's cols x VD) from its sum over the keys and that of the probabilities.
__device__ inline void finish(void* out, const bf16_t* gate, const SinkArgs& a, int r, int hbase, int idx, float sum, float L) {
  float f = 1.0f / L;
  const int hh = hbase + idx / a.VD, first = hbase * a.VD;
  if (gate != nullptr) f /= 1.f + expf(-to_f32(gate[(long long)r * a.ldg + hh]));
  float v = sum * f;
  if (a.wide_gate != nullptr) v /= 1.f + expf(-a.wide_gate[(long long)r * a.ldwg + first + idx]);
  put_out((bf16_t*)out, (long long)r * a.ldo + first + idx, v, a.out_f32);
}

// The shares of a row and tile added up in their order, by a whole workgroup.
__device__ inline void add_shares(void* out, const bf16_t* gate, const SinkArgs& a, const Shares& sh, const Heads& hd, int live) {
  __shared__ float factor[MAX_SPLITS][16], sums[MAX_SPLITS][16], whole[16];
  const int tid = threadIdx.x, r = blockIdx.x, cols = hd.cols, VD = a.VD;
  const float* shares = sh.part + ((long long)r * gridDim.y + blockIdx.y) * sh.splits * hd.share_floats;
  // The results of the first eight shares (three pairs of entries a thread) are asked for together with every share's factor
  // for every head and the heads' sums: all that a row of up to eight shares waits for is one round trip for every 1 536 entries.
  // (Entries one by one, four of four shares together, behind the factors, 16 heads of 192 of five shares waited for seven: 8 rows
  // of 700 keys 20.8 -> 19.2 us, 4 rows of 2 900 and 32 heads 26.4 -> 22.7; 8 rows of 32 heads of 128 over 8 14.7 -> 13.6.)
  constexpr int PAIRS = 3, SHARES = 8;
  const int entries = cols * VD;
  float2 v[SHARES][PAIRS];
  auto ask = [&](int s0, int i0) {
#pragma unroll
    for (int j = 0; j < SHARES; ++j)
      if (s0 + j < live)  // (the same for the whole workgroup)
#pragma unroll
        for (int x = 0; x < PAIRS; ++x)
          v[j][x] = published2(shares + (s0 + j) * hd.share_floats + min(i0 + 2 * x * NW * 64, entries - 2));
  };
  ask(0, 2 * tid);
  for (int x = tid; x < live * cols; x += NW * 64) {
    const int s = x / cols, cc = x - s * cols;
    const float* p = shares + s * hd.share_floats + entries + cc;
    factor[s][cc] = published(p), sums[s][cc] = published(p + cols);
  }
  __syncthreads();
  if (tid < cols) {
    float M = NONE, L = 0.f;
    for (int s = 0; s < live; ++s) M = fmaxf(M, factor[s][tid]);
    for (int s = 0; s < live; ++s) {
      const float f = __builtin_amdgcn_exp2f(factor[s][tid] - M);
      factor[s][tid] = f, L = fmaf(f, sums[s][tid], L);
    }
    whole[tid] = L;
  }
  __syncthreads();
  for (int i0 = 2 * tid; i0 < entries; i0 += 2 * PAIRS * NW * 64) {
    float2 sum[PAIRS];
#pragma unroll
    for (int x = 0; x < PAIRS; ++x) sum[x] = make_float2(0.f, 0.f);
    for (int s0 = 0; s0 < live; s0 += SHARES) {
      if (s0 > 0 || i0 > 2 * tid) ask(s0, i0);
#pragma unroll
      for (int j = 0; j < SHARES; ++j)
        if (s0 + j < live)
#pragma unroll
          for (int x = 0; x < PAIRS; ++x) {
            const float f = factor[s0 + j][min(i0 + 2 * x * NW * 64, entries - 2) / VD];  // (VD is even: a pair is one head's)
            sum[x].x = fmaf(f, v[j][x].x, sum[x].x), sum[x].y = fmaf(f, v[j][x].y, sum[x].y);
          }
    }
#pragma unroll
    for (int x = 0; x < PAIRS; ++x) {
      const int idx = i0 + 2 * x * NW * 64;
      if (idx >= entries) continue;
      finish(out, gate, a, r, hd.hbase, idx, sum[x].x, whole[idx / VD]);
      finish(out, gate, a, r, hd.hbase, idx + 1, sum[x].y, whole[idx / VD]);
    }
  }
}

__global__ __launch_bounds__(NW * 64) void sink_add_shares_kernel(void* __restrict__ out, const bf16_t* __restrict__ gate,
                                                                  SinkArgs a, Shares sh) {
  const int live = live_shares(sh, blocks_of(a, a.row_pos[blockIdx.x]));
  if (live > 1) add_shares(out, gate, a, sh, heads_of(a), live);  // (else the row is finished)
}

// KD and VD up to 32 KS and 16 VT: sizes in between run with zeros behind their keys and values.
template <int KS, int VT, bool SHAPED>
__global__ __launch_bounds__(NW * 64, 16 * KS + 8 * VT <= 128 ? 2 : 1) void sink_decode_kernel(
    const bf16_t* __restrict__ q, void* __restrict__ out, const bf16_t* __restrict__ gate,
    const bf16_t* __restrict__ kcache, const bf16_t* __restrict__ vcache, SinkArgs a, Shares sh) {
  extern __shared__ __attribute__((aligned(16))) float lds[];  // [NW][16][VD + 4]
  __shared__ float lds_m[NW][16], lds_l[NW][16];
  __shared__ int last;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c = lane & 15, g = lane >> 4;
  const int r = blockIdx.x, split = blockIdx.z;
  const Heads hd = heads_of(a);
  const int kvh = hd.kvh, hbase = hd.hbase, cols = hd.cols, h = hbase + min(c, cols - 1);
  const int nvh = a.nkv / a.maps, vh = kvh / a.maps, KD = a.KD, VD = a.VD, row_floats = VD + 4;
  const long long krow = (long long)a.maps * KD;

  const int pos = a.row_pos[r];
  const int* table = a.block_table + (long long)a.seq_slot[a.row_seq[r]] * a.bt_stride;
  const Blocks seen = blocks_of(a, pos);
  const int lo = seen.lo, wstart = seen.wstart, kept = seen.kept, blocks = seen.n, live = live_shares(sh, seen);
  if (split >= live) return;  // the whole workgroup

  u32x4 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int d = 32 * ks + 8 * g;
    qf[ks] = d < KD ? __builtin_bit_cast(u32x4, load_q8(q + (long long)r * a.ldq + h * KD + d)) : (u32x4){0u, 0u, 0u, 0u};
  }
  HeadShape hs;
  if constexpr (SHAPED) hs = head_shape(a, h);
  const float c2 = a.scale * LOG2E;
  float m = NONE, l = 0.f;  // the head's running maximum (in powers of two); this lane's share of its sum
  if (a.sink && split == 0 && w == 0) {
    const SinkStart start = sink_start(a, h);
    m = start.m, l = g == 0 ? start.l : 0.f;
  }
  f32x4 o[VT];  // o[dt][e]: value entry 16 dt + 4 g + e of head c
#pragma unroll
  for (int dt = 0; dt < VT; ++dt) o[dt] = (f32x4){0.f, 0.f, 0.f, 0.f};

  for (int i = split * NW + w; i < blocks; i += live * NW) {
    const int t0 = i < kept ? i * BLOCK : wstart + (i - kept) * BLOCK;
    const long long blk = table[t0 / BLOCK];
    const bf16_t* kb = kcache + (blk * nvh + vh) * BLOCK * krow + (kvh % a.maps) * KD + 8 * g;
    const bf16_t* vb = vcache + (blk * nvh + vh) * (long long)VD * BLOCK + 8 * g;
    u32x4 kf[4][KS], vf[VT][2];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int key = 32 * (j >> 1) + (c >> 2) * 8 + (j & 1) * 4 + (c & 3);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        kf[j][ks] = 32 * ks + 8 * g < KD ? *(const u32x4*)(kb + key * krow + 32 * ks) : (u32x4){0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int dt = 0; dt < VT; ++dt)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        vf[dt][j] = 16 * dt + c < VD ? *(const u32x4*)(vb + (16 * dt + c) * BLOCK + 32 * j) : (u32x4){0u, 0u, 0u, 0u};
    __builtin_amdgcn_sched_barrier(0);  // (all of them before the first product)
    f32x4 st[4];  // st[j][e]: key t0 + 32 (j / 2) + 8 g + 4 (j % 2) + e
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      st[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        st[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(kf[j][ks]), as_bf16x8(qf[ks]), st[j], 0, 0, 0);
    }
    float top = NONE;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int t = t0 + 32 * (j >> 1) + 8 * g + 4 * (j & 1) + e;
        float s;
        if constexpr (SHAPED) s = shaped<false>(st[j][e], max(pos - t, 0), hs) * LOG2E;
        else s = st[j][e] * c2;
        st[j][e] = t <= pos && (t >= lo || t < a.keep_first) ? s : -INFINITY;
        top = fmaxf(top, st[j][e]);
      }
    const float m_new = fmaxf(m, across_max(top)), alpha = __builtin_amdgcn_exp2f(m - m_new);
    m = m_new;
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        st[j][e] = __builtin_amdgcn_exp2f(st[j][e] - m);
        sum += st[j][e];
      }
    l = l * alpha + sum;
#pragma unroll
    for (int dt = 0; dt < VT; ++dt) o[dt] *= alpha;
    if (t0 + BLOCK - 1 > pos) {  // (0 times what lies in unwritten memory may be NaN)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const int t = t0 + 32 * j + 8 * g + 2 * x;
          const unsigned keep = t + 1 <= pos ? 0xffffffffu : t <= pos ? 0x0000ffffu : 0u;
#pragma unroll
          for (int dt = 0; dt < VT; ++dt) vf[dt][j][x] &= keep;
        }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      u32x4 part[3];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float p0 = st[2 * j + (x >> 1)][2 * (x & 1)], p1 = st[2 * j + (x >> 1)][2 * (x & 1) + 1];
        const float q0 = below_upper(p0), q1 = below_upper(p1);
        part[0][x] = upper2(p0, p1), part[1][x] = upper2(q0, q1), part[2][x] = upper2(below_upper(q0), below_upper(q1));
      }
#pragma unroll
      for (int i3 = 2; i3 >= 0; --i3)
#pragma unroll
        for (int dt = 0; dt < VT; ++dt)
          o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(vf[dt][j]), as_bf16x8(part[i3]), o[dt], 0, 0, 0);
    }
  }
  // the wavefronts' results meet
  l = across_sum(l);
#pragma unroll
  for (int dt = 0; dt < VT; ++dt)
    if (16 * dt + 4 * g < VD && c < cols) *(f32x4*)(lds + (w * 16 + c) * row_floats + 16 * dt + 4 * g) = o[dt];
  if (g == 0) lds_m[w][c] = m, lds_l[w][c] = l;
  __syncthreads();
  const long long at = (long long)r * gridDim.y + blockIdx.y;
  float* mine = sh.part + (at * sh.splits + split) * hd.share_floats;
  for (int idx = tid; idx < cols * VD; idx += NW * 64) {
    const int cc = idx / VD, d = idx - cc * VD;
    float M = lds_m[0][cc];
#pragma unroll
    for (int j = 1; j < NW; ++j) M = fmaxf(M, lds_m[j][cc]);
    float sum = 0.f, L = 0.f;
#pragma unroll
    for (int j = 0; j < NW; ++j) {
      const float f = __builtin_amdgcn_exp2f(lds_m[j][cc] - M);
      sum = fmaf(f, lds[(j * 16 + cc) * row_floats + d], sum), L = fmaf(f, lds_l[j][cc], L);
    }
    if (live == 1) {
      finish(out, gate, a, r, hbase, idx, sum, L);
    } else {
      publish(mine + idx, sum);
      if (d == 0) publish(mine + cols * VD + cc, M), publish(mine + cols * VD + cols + cc, L);
    }
  }
  if (live == 1 || sh.tickets == nullptr) return;
  // Once every thread's stores have completed the workgroup takes a ticket; the last one adds the shares up.
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  __syncthreads();
  if (tid == 0)
    last = __hip_atomic_fetch_add(sh.tickets + at, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == live - 1;
  __syncthreads();
  if (!last) return;
  add_shares(out, gate, a, sh, hd, live);
  if (tid == 0) __hip_atomic_store(sh.tickets + at, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
}

template <int KS, int VT>
int launch(const bf16_t* q, void* out, const bf16_t* gate, const bf16_t* kcache, const bf16_t* vcache, const SinkArgs& a,
           const Shares& sh, dim3 grid, hipStream_t stream) {
  const int bytes = NW * 16 * (a.VD + 4) * (int)sizeof(float);
  const bool with_shape = scores_shaped(a.shape);
  const auto kernel = with_shape ? sink_decode_kernel<KS, VT, true> : sink_decode_kernel<KS, VT, false>;
  static bool configured[2] = {false, false};
  if (!configured[with_shape]) {
    const int most = NW * 16 * (16 * VT + 4) * (int)sizeof(float);
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, most);
    if (e != hipSuccess) {
      lq_set_error("sink_attention: cannot reserve %d bytes of LDS: %s", most, hipGetErrorString(e));
      return -2;
    }
    configured[with_shape] = true;
  }
  kernel<<<grid, NW * 64, bytes, stream>>>(q, out, gate, kcache, vcache, a, sh);
  LQ_CHECK_LAUNCH("sink_attention(single tokens)");
  if (sh.splits > 1 && sh.tickets == nullptr) {
    sink_add_shares_kernel<<<dim3(grid.x, grid.y), NW * 64, 0, stream>>>(out, gate, a, sh);
    LQ_CHECK_LAUNCH("sink_attention(shares of single tokens)");
  }
  return 1;
}

// Shares of a row's keys: as many as give every wavefront one block of the `max_len` bound, within two rounds of
// workgroups.
int splits_for(int rows, int nh, int nkv, int window, int keep_first, int chunk, int max_len) {
  if (max_len <= 0) return 1;
  const long long seen = window > 0 ? (long long)window + keep_first + 2 * BLOCK : max_len;
  int keys = seen < max_len ? (int)seen : max_len;
  if (chunk > 0 && chunk + BLOCK < keys) keys = chunk + BLOCK;
  const long long tiles = (long long)rows * nkv * lq_ceil_div(nh / nkv, 16);
  const int wanted = lq_ceil_div(lq_ceil_div(keys, BLOCK) + 1, NW), room = (int)(2 * lq_compute_units() / tiles);
  const int most = room > MAX_SPLITS ? MAX_SPLITS : room;
  return wanted < most ? wanted : most > 1 ? most : 1;
}

bool takes(int KD, int VD, int block_size, int nh, int nkv, int rows) {
  return block_size == BLOCK && KD % 8 == 0 && VD % 4 == 0 && KD <= 256 && VD <= 256 &&
         (long long)nkv * lq_ceil_div(nh / nkv, 16) <= 65535 && rows < (1 << 22);
}

}  // namespace

long long lq_sink_decode_workspace(int rows, int nh, int nkv, int KD, int VD, int block_size, int window, int keep_first,
                                   int chunk, int max_len) {
  if (!takes(KD, VD, block_size, nh, nkv, rows)) return 0;
  const int splits = splits_for(rows, nh, nkv, window, keep_first, chunk, max_len), group = nh / nkv;
  if (splits == 1) return 0;
  return (long long)rows * nkv * lq_ceil_div(group, 16) * splits * (group < 16 ? group : 16) * (VD + 2);
}

int lq_sink_decode(const bf16_t* q, void* out, const bf16_t* gate, const bf16_t* kcache, const bf16_t* vcache,
                   const SinkArgs& a, int max_len, float* part, long long part_floats, int* tickets, long long tickets_n,
                   hipStream_t stream) {
  if (a.ldq % 4 != 0 || (uintptr_t)q % 8 != 0 || ((uintptr_t)kcache | (uintptr_t)vcache) % 16 != 0 ||
      !takes(a.KD, a.VD, a.BS, a.nh, a.nkv, a.rows))
    return 0;
  const int tiles = a.nkv * lq_ceil_div(a.nh / a.nkv, 16);
  Shares sh = {1, part, (long long)a.rows * tiles <= tickets_n ? tickets : nullptr};
  if (part != nullptr && (uintptr_t)part % 8 == 0) {  // (shares are read in pairs)
    const long long need = lq_sink_decode_workspace(a.rows, a.nh, a.nkv, a.KD, a.VD, a.BS, a.window, a.keep_first, a.chunk, max_len);
    if (need > 0 && need <= part_floats) sh.splits = splits_for(a.rows, a.nh, a.nkv, a.window, a.keep_first, a.chunk, max_len);
  }
  const dim3 grid(a.rows, tiles, sh.splits);
#define LQ_DECODE(KS, VT) launch<KS, VT>(q, out, gate, kcache, vcache, a, sh, grid, stream)
  if (a.KD <= 64 && a.VD <= 64) return LQ_DECODE(2, 4);
  if (a.KD <= 128 && a.VD <= 128) return LQ_DECODE(4, 8);
  if (a.KD <= 128) return LQ_DECODE(4, 16);
  if (a.VD <= 192) return LQ_DECODE(8, 12);
  return LQ_DECODE(8, 16);
#undef LQ_DECODE
}
