// Steps of single tokens of a bfloat16 run through the windowed attention of attention_sink.hip (the same masks, sinks,
// shaped scores, maps and gates).
//
// A workgroup of four wavefronts takes one row of the step, up to 16 query heads of one key head and one of up to `splits`
// shares of the blocks of 64 positions that the row sees, numbered from the kept first ones on.  All four work on the same block (two of
// key and value sizes up to 64): 16 keys' scores a wavefront, whose probabilities meet in LDS, and a quarter of the value
// entries each, so that nothing is merged at a share's end.  The next block is asked for ahead of this one's products.  What bounds
// such a step is the rate at which one compute unit draws its blocks (1.1 us for 32 KB), the chain of round trips around it and the
// code's own way from memory (attention_decode.hip, which has the same structure for plain causal attention): so blocks are
// dealt out evenly over as many workgroups as pay for it, and a key head's query heads over several workgroups where rows are few
// (`shares_for`).  The shares of a row meet in its last workgroup to finish (a ticket a row and tile of heads; partial
// results pass the dies' caches as device-scope atomics), which adds them up in their order; a caller who gives no tickets gets
// a second launch that does the same.
//
// Microseconds a launch, a wavefront with a block of its own, shares of at least four blocks and 16 heads a workgroup -> this:
// one key head of 256 with values of 192 under 16 heads, 8 rows of 216 to 716 keys 18.2 -> 11.0, one of 700 18.0 -> 9.2, one of 3 000 21.4 -> 12.9,
// 24 of 100 11.5 -> 8.7; 16 heads of 128 over 4: 8 rows of 520 keys 11.8 -> 8.9, with two maps over values of 256 15.1 -> 11.1, 2 rows of
// 1 000 with capped scores 13.2 -> 10.2, with a table of biases 14.6 -> 10.6; 24 rows of 120 keys, 32 heads over 8, 8.2 -> 8.0.
//
//   S^T[key][head] = K . Q^T by v_mfma_f32_16x16x32_bf16: lane (c = l % 16, g = l / 16) gives A[c][8 g .. + 8] and B[c][the
//   same] and receives D[4 g + e][c]; O^T[d][head] += V^T . P^T with eight consecutive keys a lane, read back from LDS.
// The probabilities stay 32-bit, multiplied in three bfloat16 parts that add up to them exactly (attention_sink_rows.hip).
// Values of positions that were never written count as zero.
#include "attention_sink.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int BLOCK = 64, NW = 4, MAX_SPLITS = 64;
constexpr int NARROW = 3;  // blocks a share up to which one workgroup a compute unit is better than two

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

__device__ inline void publish2(float* p, float x, float y) {  // two neighbours on 8 bytes
  const unsigned long long v = (unsigned long long)__float_as_uint(y) << 32 | __float_as_uint(x);
  __hip_atomic_store((unsigned long long*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline float2 published2(const float* p) {  // two neighbours on 8 bytes
  const unsigned long long v = __hip_atomic_load((unsigned long long*)const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return make_float2(__uint_as_float((unsigned)v), __uint_as_float((unsigned)(v >> 32)));
}

struct Shares {
  int splits, narrow;    // workgroups a row and tile at most; the same without a second one on any compute unit
  int heads, tiles;      // query heads a workgroup; how many such tiles a key head has
  int whole;             // blocks up to which a row stays whole
  int long_from;         // > 0: a row goes in `splits` shares from this many blocks on, else whole (many_rows)
  float apart;           // what a share more costs, in blocks' time
  float* part;   // [row][key head's tile][split]: heads x VD results, then maximum and sum of each head
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

// n / d and its ceiling for whole numbers below 2^20: half a unit of the numerator is more than the reciprocal's error.
__device__ inline int quotient(int n, int d) {
  return __builtin_amdgcn_readfirstlane((int)(((float)n + 0.5f) * __builtin_amdgcn_rcpf((float)d)));
}

// Blocks a share of a row that has n: the rule of attention_decode.hip, with the costs of these sizes (`shares_for`).
__device__ inline int blocks_a_share(const Shares& sh, int n) {
  if (n <= sh.whole || sh.splits == 1 || n < sh.long_from) return n;
  if (sh.long_from > 0) return quotient(n - 1, sh.splits) + 1;
  const int narrow = quotient(n - 1, sh.narrow) + 1;
  const bool alone = narrow <= NARROW || 0.1f * narrow < sh.apart * (sh.splits - sh.narrow);
  const int even = alone ? narrow : quotient(n - 1, sh.splits) + 1;
  return max(even, __builtin_amdgcn_readfirstlane((int)(__builtin_amdgcn_sqrtf((float)n * sh.apart) + 0.5f)));
}

// A workgroup's row and key head's tile: its query heads hbase .. hbase + cols - 1.
struct Heads {
  int kvh, hbase, cols, share_floats;
};
__device__ inline Heads heads_of(const SinkArgs& a, const Shares& sh) {
  const int group = a.heads_per_tile, kvh = sh.tiles == 1 ? blockIdx.y : quotient(blockIdx.y, sh.tiles);
  const int hbase = kvh * group + (blockIdx.y - kvh * sh.tiles) * sh.heads;
  return {kvh, hbase, min(sh.heads, (kvh + 1) * group - hbase), sh.heads * (a.VD + 2)};
}

__device__ inline float gate_of(const bf16_t* gate, const SinkArgs& a, int r, int h) {
  return gate != nullptr ? to_f32(gate[(long long)r * a.ldg + h]) : 0.f;
}
// What a head's entries are multiplied with, from the sum of its probabilities and the logit of its gate.
__device__ inline float head_factor(const bf16_t* gate, float logit, float L) {
  float f = 1.0f / L;
  if (gate != nullptr) f /= 1.f + expf(-logit);
  return f;
}

// Two neighbouring entries (d, even, of head h) from their sums over the keys.
__device__ inline void finish2(void* out, const SinkArgs& a, int r, int h, int d, float2 sum, float factor) {
  float2 v = make_float2(sum.x * factor, sum.y * factor);
  if (a.wide_gate != nullptr) {
    const float* p = a.wide_gate + (long long)r * a.ldwg + h * a.VD + d;
    v.x /= 1.f + expf(-p[0]), v.y /= 1.f + expf(-p[1]);
  }
  const long long at = (long long)r * a.ldo + h * a.VD + d;
  put_out((bf16_t*)out, at, v.x, a.out_f32);
  put_out((bf16_t*)out, at + 1, v.y, a.out_f32);
}

// The shares of a row and tile added up in their order, by a whole workgroup: PAIRS times two neighbouring entries a thread, and eight
// shares of each, are asked for at once, as far as there are so many.  What bounds it is these round trips: partial results come past the
// caches, and requests for shares that a row does not have would be as slow as any others (16 heads of 192, 24 rows of 160 keys, a pair at a time
// and always eight shares 12.9 -> 12.0 us; of 1 000 17.4 -> 16.1; 4 heads of 128 with two maps, 33 rows of 500 keys 19.9 -> 18.3).
template <int PAIRS>
__device__ inline void add_shares(void* out, const bf16_t* gate, const SinkArgs& a, const Shares& sh, const Heads& hd, int live) {
  constexpr int AT_ONCE = 8;
  const int r = blockIdx.x, VD = a.VD, entries = hd.cols * VD;
  const float* shares = sh.part + ((long long)r * gridDim.y + blockIdx.y) * sh.splits * hd.share_floats;
  for (int i0 = 2 * threadIdx.x; i0 < entries; i0 += 2 * PAIRS * NW * 64) {  // (VD is even: a pair is one head's)
    int c[PAIRS];
    float logit[PAIRS], M[PAIRS], L[PAIRS];
    float2 acc[PAIRS];
#pragma unroll
    for (int x = 0; x < PAIRS; ++x) {
      c[x] = (int)(((float)min(i0 + 2 * x * NW * 64, entries - 2) + 0.5f) * __builtin_amdgcn_rcpf((float)VD));
      logit[x] = gate_of(gate, a, r, hd.hbase + c[x]);
      M[x] = NONE, L[x] = 0.f, acc[x] = make_float2(0.f, 0.f);
    }
    for (int s0 = 0; s0 < live; s0 += AT_ONCE) {
      float2 stat[PAIRS][AT_ONCE], sum[PAIRS][AT_ONCE];
#pragma unroll
      for (int j = 0; j < AT_ONCE; ++j)
#pragma unroll
        for (int x = 0; x < PAIRS; ++x) {
          stat[x][j] = make_float2(NONE, 0.f), sum[x][j] = make_float2(0.f, 0.f);
          if (s0 + j < live && (x == 0 || 2 * x * NW * 64 < entries)) {  // (the same for the whole workgroup)
            const float* p = shares + (s0 + j) * hd.share_floats;
            stat[x][j] = published2(p + sh.heads * VD + 2 * c[x]), sum[x][j] = published2(p + min(i0 + 2 * x * NW * 64, entries - 2));
          }
        }
#pragma unroll
      for (int x = 0; x < PAIRS; ++x) {
        float top = M[x];
#pragma unroll
        for (int j = 0; j < AT_ONCE; ++j) top = fmaxf(top, stat[x][j].x);
        const float keep = __builtin_amdgcn_exp2f(M[x] - top);
        acc[x].x *= keep, acc[x].y *= keep, L[x] *= keep, M[x] = top;
#pragma unroll
        for (int j = 0; j < AT_ONCE; ++j) {
          const float f = s0 + j < live ? __builtin_amdgcn_exp2f(stat[x][j].x - M[x]) : 0.f;
          acc[x].x = fmaf(f, sum[x][j].x, acc[x].x), acc[x].y = fmaf(f, sum[x][j].y, acc[x].y), L[x] = fmaf(f, stat[x][j].y, L[x]);
        }
      }
    }
#pragma unroll
    for (int x = 0; x < PAIRS; ++x) {
      const int i = i0 + 2 * x * NW * 64;
      if (i < entries) finish2(out, a, r, hd.hbase + c[x], i - c[x] * VD, acc[x], head_factor(gate, logit[x], L[x]));
    }
  }
}

__global__ __launch_bounds__(NW * 64) void sink_add_shares_kernel(void* __restrict__ out, const bf16_t* __restrict__ gate,
                                                                  SinkArgs a, Shares sh) {
  const int n = blocks_of(a, a.row_pos[blockIdx.x]).n, live = quotient(n - 1, blocks_a_share(sh, n)) + 1;
  if (live > 1) add_shares<2>(out, gate, a, sh, heads_of(a, sh), live);  // (else the row is finished)
}

// KD and VD up to 32 KS and 16 VT: sizes in between run with zeros behind their keys and values.  GB blocks are taken together.
template <int KS, int VT>
struct Share {
  static constexpr int VW = VT / NW, GB = KS + VT / 2 <= 4 ? 2 : 1;
  u32x4 k[GB][KS];     // of the wavefront's 16 keys row lane % 16, entries 32 ks + 8 (lane / 16) ..
  u32x4 v[GB][VW][2];  // of its tiles of value entries row lane % 16, positions 32 j + 8 (lane / 16) ..
  float bias[GB][4];   // by distance, for scores 4 (lane / 16) + e
};

template <int KS, int VT, bool SHAPED>
__global__ __launch_bounds__(NW * 64, KS <= 4 ? 2 : 1) void sink_decode_kernel(
    const bf16_t* __restrict__ q, void* __restrict__ out, const bf16_t* __restrict__ gate,
    const bf16_t* __restrict__ kcache, const bf16_t* __restrict__ vcache, SinkArgs a, Shares sh) {
  using S = Share<KS, VT>;
  __shared__ __attribute__((aligned(16))) float scores[2][16][S::GB * BLOCK + 4];  // (apart so that neighbouring heads' lie in other banks)
  __shared__ __attribute__((aligned(16))) float tops[2][16][NW];  // (what wavefronts' probabilities were taken against)
  __shared__ int last;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
  const int r = blockIdx.x, split = blockIdx.z;
  // (rows of single tokens mostly are their sequences' in order: that one's slot is asked for beside the row's sequence, not behind it)
  const int pos = a.row_pos[r], seq = a.row_seq[r], likely = a.seq_slot[r];
  const Heads hd = heads_of(a, sh);
  const int kvh = hd.kvh, cols = hd.cols, h = hd.hbase + min(c, cols - 1);  // (columns beyond the tile's heads repeat the last one's)
  const int KD = a.KD, VD = a.VD, maps = a.maps, vh = maps == 1 ? kvh : quotient(kvh, maps), nvh = maps == 1 ? a.nkv : quotient(a.nkv, maps);
  // the query and what is asked of its head, before the position is known
  u32x4 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int d = 32 * ks + 8 * g;
    qf[ks] = d < KD ? __builtin_bit_cast(u32x4, load_q8(q + (long long)r * a.ldq + h * KD + d)) : (u32x4){0u, 0u, 0u, 0u};
  }
  HeadShape hs;
  const float* dist = nullptr;
  if constexpr (SHAPED) {
    hs = head_shape(a, h);
    dist = hs.dist, hs.dist = nullptr;
  }
  // (Asked for here and used behind the keys on their way: behind the keys' requests they waited for all of these, one row under a window of 128
  // with sinks 7.5 -> 6.6 us.  Without a sink's value or a gate something else is read, and not used.)
  const float sink = *(a.sinks != nullptr ? a.sinks + h : (const float*)a.row_pos + r);
  const bf16_t logit = *(gate != nullptr ? gate + (long long)r * a.ldg + h : q + (long long)r * a.ldq);
  __builtin_amdgcn_sched_barrier(0);
  const int* table = a.block_table + (long long)(seq == r ? likely : a.seq_slot[seq]) * a.bt_stride;
  const Blocks seen = blocks_of(a, pos);
  const int lo = seen.lo, wstart = seen.wstart, kept = seen.kept;
  const int per = blocks_a_share(sh, seen.n), live = quotient(seen.n - 1, per) + 1;
  if (split >= live) return;  // the whole workgroup
  const int i0 = split * per, i1 = min(i0 + per, seen.n) - 1;
  auto start_of = [&](int i) { return i < kept ? i * BLOCK : wstart + (i - kept) * BLOCK; };

  const int krow = maps * KD * 2;  // bytes
  const int k_at = (16 * w + c) * krow + ((kvh - vh * maps) * KD + 8 * g) * 2, v_at = ((16 * w + c) * BLOCK + 8 * g) * 2;
  // Asks for a block, or, with the same instructions, for nothing at all (a descriptor of no bytes, every access of which is
  // out of bounds and yields zero), as entries beyond KD and VD are.
  auto ask = [&](int i, int blk, int u, S& s) {
    const bool there = i <= i1;
    const long long at = (long long)blk * nvh + vh;
    const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc((void*)(kcache + at * BLOCK * (maps * KD)), 0, there ? BLOCK * krow : 0, 0x00020000);
    const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc((void*)(vcache + at * BLOCK * VD), 0, there ? BLOCK * VD * 2 : 0, 0x00020000);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      s.k[u][ks] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(kr, 32 * ks + 8 * g < KD ? k_at + 64 * ks : 0x40000000, 0, 0));
#pragma unroll
    for (int x = 0; x < S::VW; ++x)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        s.v[u][x][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(vr, v_at + x * (NW * 16 * BLOCK * 2) + 64 * j, 0, 0));
    if constexpr (SHAPED)
      if (dist != nullptr)
#pragma unroll
        for (int e = 0; e < 4; ++e) s.bias[u][e] = dist[min(max(pos - (start_of(i) + 16 * w + 4 * g + e), 0), hs.last)];
  };
  // (the first blocks' numbers by scalar loads, those of the blocks behind them 64 at a time, lane l that of the share's l-th: attention_decode.hip;
  // one row of 160 keys, 16 heads of 64 over 8, 7.6 -> 6.7 us)
  S cur;
  int numbers = table[start_of(min(i0 + lane, i1)) / BLOCK];
#pragma unroll
  for (int u = 0; u < S::GB; ++u) ask(i0 + u, table[start_of(min(i0 + u, i1)) / BLOCK], u, cur);
  __builtin_amdgcn_sched_barrier(0);

  const float c2 = a.scale * LOG2E;
  float m = NONE, l = 0.f;  // the head's running maximum (in powers of two); this lane's share of its sum
  if (a.sink && split == 0) {
    const SinkStart start = a.sinks != nullptr ? start_at(sink) : SinkStart{0.f, 1.f};
    m = start.m, l = g == 0 ? start.l : 0.f;
  }
  f32x4 o[S::VW];  // o[x][e]: value entry 16 (w + NW x) + 4 g + e of head c
#pragma unroll
  for (int x = 0; x < S::VW; ++x) o[x] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // Blocks i .. i + GB - 1 of the share, as far as it reaches; `turn`: whose turn it is of the two buffers.  A wavefront takes its
  // keys' probabilities against their own maximum; whoever reads them multiplies them up to the row's.
  auto take = [&](int i, int turn, S& s) {
    f32x4 st[S::GB];  // keys 16 w + 4 g + e of each block
    float own_top = NONE;
#pragma unroll
    for (int u = 0; u < S::GB; ++u) {
      if (u > 0 && i + u > i1) break;  // (a share's odd last block goes alone: 160 keys as above 6.5 -> 6.1 us)
      const int t0 = start_of(i + u);
      st[u] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        st[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(s.k[u][ks]), as_bf16x8(qf[ks]), st[u], 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int t = t0 + 16 * w + 4 * g + e;
        float x;
        if constexpr (SHAPED) {
          x = shaped<false>(st[u][e], max(pos - t, 0), hs);
          if (dist != nullptr) x += s.bias[u][e];
          x *= LOG2E;
        } else {
          x = st[u][e] * c2;
        }
        st[u][e] = x;
      }
      if (t0 + BLOCK - 1 > pos || (t0 < lo && t0 + BLOCK > a.keep_first))  // (not all of its positions are seen)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int t = t0 + 16 * w + 4 * g + e;
          if ((t > pos) | ((t < lo) & (t >= a.keep_first))) st[u][e] = -INFINITY;
        }
      own_top = fmaxf(own_top, fmaxf(fmaxf(st[u][0], st[u][1]), fmaxf(st[u][2], st[u][3])));
      if (t0 + BLOCK - 1 > pos) {  // (0 times what lies in unwritten memory may be NaN)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            const int t = t0 + 32 * j + 8 * g + 2 * x;
            const unsigned keep = t + 1 <= pos ? 0xffffffffu : t <= pos ? 0x0000ffffu : 0u;
#pragma unroll
            for (int y = 0; y < S::VW; ++y) s.v[u][y][j][x] &= keep;
          }
      }
    }
    own_top = across_max(own_top);
#pragma unroll
    for (int u = 0; u < S::GB; ++u) {
      if (u > 0 && i + u > i1) break;
#pragma unroll
      for (int e = 0; e < 4; ++e) st[u][e] = __builtin_amdgcn_exp2f(st[u][e] - own_top);
      *(f32x4*)&scores[turn][c][u * BLOCK + 16 * w + 4 * g] = st[u];
    }
    if (g == 0) tops[turn][c][w] = own_top;
    // (loads fly on; the other buffer's readers have passed this barrier once more than its writers)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const f32x4 tw = *(const f32x4*)&tops[turn][c][0];
    const float m_new = fmaxf(m, fmaxf(fmaxf(tw[0], tw[1]), fmaxf(tw[2], tw[3]))), alpha = __builtin_amdgcn_exp2f(m - m_new);
    m = m_new;
    l *= alpha;
#pragma unroll
    for (int x = 0; x < S::VW; ++x) o[x] *= alpha;
    const float up[2] = {__builtin_amdgcn_exp2f((g < 2 ? tw[0] : tw[1]) - m), __builtin_amdgcn_exp2f((g < 2 ? tw[2] : tw[3]) - m)};
#pragma unroll
    for (int u = 0; u < S::GB; ++u) {
      if (u > 0 && i + u > i1) break;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        f32x4 pr[2];  // keys 32 j + 8 g .. + 7
        u32x4 part[3];
#pragma unroll
        for (int x = 0; x < 2; ++x) pr[x] = *(const f32x4*)&scores[turn][c][u * BLOCK + 32 * j + 8 * g + 4 * x] * up[j];
        const f32x4 both = pr[0] + pr[1];
        l += (both[0] + both[1]) + (both[2] + both[3]);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const float p0 = pr[x >> 1][2 * (x & 1)], p1 = pr[x >> 1][2 * (x & 1) + 1];
          const float q0 = below_upper(p0), q1 = below_upper(p1);
          part[0][x] = upper2(p0, p1), part[1][x] = upper2(q0, q1), part[2][x] = upper2(below_upper(q0), below_upper(q1));
        }
#pragma unroll
        for (int i3 = 2; i3 >= 0; --i3)
#pragma unroll
          for (int x = 0; x < S::VW; ++x)
            o[x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(s.v[u][x][j]), as_bf16x8(part[i3]), o[x], 0, 0, 0);
      }
    }
  };
  for (int i = i0, odd = 0;; i += S::GB, odd ^= 1) {
    S next;
    const int at = (i + S::GB - i0) & 63;
    if (at == 0) {  // (64 is a multiple of GB)
      numbers = table[start_of(min(i + S::GB + lane, i1)) / BLOCK];
      asm volatile("" : "+v"(numbers));  // (waited for in here, not behind the branch)
    }
#pragma unroll
    for (int u = 0; u < S::GB; ++u) ask(min(i + S::GB + u, i1 + 1), __builtin_amdgcn_readlane(numbers, at + u), u, next);
    take(i, odd, cur);
    if (i + S::GB > i1) break;
    cur = next;
  }
  l = across_sum(l);
  const long long at = (long long)r * gridDim.y + blockIdx.y;
  if (c < cols) {
    const float factor = live == 1 ? head_factor(gate, to_f32(logit), l) : 0.f;
    float* mine = sh.part + (at * sh.splits + split) * hd.share_floats;
#pragma unroll
    for (int x = 0; x < S::VW; ++x) {
      const int d = 16 * (w + NW * x) + 4 * g;
      if (d < VD)  // (VD is a multiple of 4)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
          if (live == 1) finish2(out, a, r, h, d + 2 * y, make_float2(o[x][2 * y], o[x][2 * y + 1]), factor);
          else publish2(mine + c * VD + d + 2 * y, o[x][2 * y], o[x][2 * y + 1]);
        }
    }
    if (live > 1 && w == 0 && g == 0) publish2(mine + sh.heads * VD + 2 * c, m, l);
  }
  if (live == 1 || sh.tickets == nullptr) return;
  // Once every thread's stores have completed the workgroup takes a ticket; the last one adds the shares up.
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  __syncthreads();
  if (tid == 0)
    last = __hip_atomic_fetch_add(sh.tickets + at, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == live - 1;
  __syncthreads();
  if (!last) return;
  // (few entries by the short code: a launch finds none of it in the instruction cache, and the longer one costs it 0.9 us)
  if (hd.cols * VD <= 4 * NW * 64) add_shares<1>(out, gate, a, sh, hd, live);
  else add_shares<VT <= 4 ? 2 : 3>(out, gate, a, sh, hd, live);
  if (tid == 0) __hip_atomic_store(sh.tickets + at, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
}

template <int KS, int VT>
int launch(const bf16_t* q, void* out, const bf16_t* gate, const bf16_t* kcache, const bf16_t* vcache, const SinkArgs& a,
           const Shares& sh, dim3 grid, hipStream_t stream) {
  if (scores_shaped(a.shape)) sink_decode_kernel<KS, VT, true><<<grid, NW * 64, 0, stream>>>(q, out, gate, kcache, vcache, a, sh);
  else sink_decode_kernel<KS, VT, false><<<grid, NW * 64, 0, stream>>>(q, out, gate, kcache, vcache, a, sh);
  LQ_CHECK_LAUNCH("sink_attention(single tokens)");
  if (sh.splits > 1 && sh.tickets == nullptr) {
    sink_add_shares_kernel<<<dim3(grid.x, grid.y), NW * 64, 0, stream>>>(out, gate, a, sh);
    LQ_CHECK_LAUNCH("sink_attention(shares of single tokens)");
  }
  return 1;
}

// How rows are shared out that take more than half of the compute units with one workgroup a tile of heads: in `shares` from `from` units of
// 32 KB on (0: never); the reasons are attention_decode.hip's, the lines where this kernel has them, whose workgroups have more to
// work out for what they draw, so that two a unit hide more of one another.  Whole -> so, microseconds, 32 heads of 128 over 8: 17 rows of 1 500 keys
// 35 -> 27, 24 of 3 000 68 -> 60, 26 of 3 000 with capped scores 75 -> 67, 33 of 750 30.7 -> 28, of 3 000 102 -> 85, 40 of 3 000 109 -> 97, 48 of 1 500
// 64 -> 61; 16 heads of 64 over 8: 17 of 1 500 22.6 -> 17.3, 28 of 3 000 45 -> 40, 33 of 3 000 55 -> 47.  (Shares that cost: 17 of 250 9.5 and, in
// three, 11.2; 32 of 3 000 in two 75 for 72; 56 of 1 000 in any number.)  A row a unit is not enough where tiles of one
// key head draw the same keys (40 heads of 64 with values of 40 over 2, 64 rows of 3 000 40 -> 33) and for sizes up to 64 (16 heads over 4, 64 of 3 000
// 42.1 -> 40.5; 64 of 1 000 18.4, in two 18.7): `light`.
struct ManyRows {
  int shares, from;
};
ManyRows many_rows(long long tiles, bool light) {
  const long long cus = lq_compute_units();
  if (3 * tiles <= 2 * cus) return {3, 8};
  if (4 * tiles <= 3 * cus) return {4, 12};
  if (8 * tiles <= 7 * cus || (light && tiles <= cus)) return {2, 28};
  if (tiles <= cus) return {1, 0};
  if (5 * tiles <= 6 * cus) return {5, 9};
  if (3 * tiles <= 4 * cus) return {4, 10};
  if (2 * tiles <= 3 * cus) return {2, 8};
  return {1, 0};
}

// How a launch is shared out: `splits` is 1 where no row goes in shares.
//
// In units of the time for 32 KB (1.1 us): a block of KD + VD entries takes (KD + VD) / 256, a share more its ticket and its results'
// way into the last workgroup, 0.06 + 0.07 for every 512 entries.  A row of up to 3.4 units and four shares' cost stays whole, else a
// share has the blocks that an even deal gives it and no fewer than the root of n times the quotient of the two.
//
// Query heads a workgroup: 16 where rows are many; half as many, and half again, while that makes no more than 128 workgroups a
// share, down to 4 (the last workgroup of a row then adds up a quarter: 8 rows of 216 to 716 keys 17.6 us with 16 heads, 13.7 with 8, 11.2 with 4), and
// down to 2 while it makes no more than 32 (4 rows of 700 keys 12.1 -> 10.3, one 10.7 -> 9.2; with 64 of them 11.0 -> 12.0); and while rows of the
// bound's length give a compute unit no more than 7.5 units to draw: every workgroup draws all of its row's keys (24 rows of 2 500, one key
// head of 256 with values of 192 under 16 heads, four heads a workgroup 34.6 us, 16 24.0).
//
// Sizes of up to 64 take two blocks together, in 0.75 us each: a row of two such takes stays whole, or of three where there are many tiles (one to eight
// rows, 16 heads over 8 or 4, 260 keys whole 7.6 us, in shares 6.7, 380 8.1 and 6.8, 440 9.3 and 7.1; 16 rows over 8, 320 keys 8.1 and 8.4, 440 9.8 and 8.9).
// Their heads are split no further than to a pair of entries a thread of the last workgroup, from where on it has nothing to save (64 heads over 8 under
// a window of 128, one to four rows, two heads a workgroup 6.5 us, eight 6.2; 32 over 4, one row of 500 7.3 and 6.2, of 3 000 11.5 and 9.1).
Shares shares_for(int rows, int nh, int nkv, int KD, int VD, int window, int keep_first, int chunk, int max_len) {
  Shares sh = {};
  const int group = nh / nkv, cus = lq_compute_units();
  const float block = (KD + VD) / 256.f;
  const bool small = KD <= 64 && VD <= 64;
  auto tiles = [&](int heads) { return (long long)rows * nkv * lq_ceil_div(group, heads); };
  // blocks that a row may see, within a bound of the lengths
  auto most_blocks = [&](long long bound) {
    const long long seen = window > 0 ? (long long)window + keep_first + 2 * BLOCK : bound;
    long long keys = seen < bound ? seen : bound;
    if (chunk > 0 && chunk + BLOCK < keys) keys = chunk + BLOCK;
    return (int)((keys + BLOCK - 1) / BLOCK) + 1;
  };
  int heads = 16;
  if (max_len > 0) {
    // (by the bound in 1 024s: launches whose bounds differ less than that add up their sums in the same order)
    const long long bound = ((long long)max_len + LQ_DECODE_LENGTH_BUCKET - 1) / LQ_DECODE_LENGTH_BUCKET * LQ_DECODE_LENGTH_BUCKET;
    const float units = most_blocks(bound) * block / cus;
    while (((heads > 4 && tiles(heads / 2) <= 128) || (heads > 2 && tiles(heads / 2) <= 32)) && tiles(heads / 2) * units <= 7.5f &&
           !(small && (group < heads ? group : heads) * VD <= 2 * NW * 64))
      heads /= 2;
  }
  const float share = 0.06f + 0.07f * (group < heads ? group : heads) * VD / 512.f;
  sh.heads = group < heads ? group : heads;
  sh.tiles = lq_ceil_div(group, sh.heads);
  sh.whole = (int)((3.4f + 4 * share) / block) > 1 ? (int)((3.4f + 4 * share) / block) : 1;
  if (small) sh.whole = tiles(heads) > 64 ? 6 : 4;
  sh.apart = share / block;
  sh.splits = sh.narrow = 1;
  if (max_len <= 0) return sh;
  const long long all = tiles(heads), room = 2 * cus / all, alone = cus / all;
  if (2 * all > cus) {
    const ManyRows many = many_rows(all, sh.tiles > 1 || small);
    const int from = (int)(many.from / (block > 1.f ? block : 1.f));
    if (many.shares > 1 && most_blocks(max_len) > from) sh.splits = sh.narrow = many.shares, sh.long_from = from;
    return sh;
  }
  const int wanted = most_blocks(max_len), most = room > MAX_SPLITS ? MAX_SPLITS : (int)room;
  sh.splits = wanted < most ? wanted : most;
  sh.narrow = alone > sh.splits ? sh.splits : (int)alone;
  return sh;
}

bool takes(int KD, int VD, int block_size, int nh, int nkv, int rows) {
  return block_size == BLOCK && KD % 8 == 0 && VD % 4 == 0 && KD <= 256 && VD <= 256 &&
         (long long)nkv * lq_ceil_div(nh / nkv, 16) <= 65535 && rows < (1 << 22);
}

}  // namespace

long long lq_sink_decode_workspace(int rows, int nh, int nkv, int KD, int VD, int block_size, int window, int keep_first,
                                   int chunk, int max_len) {
  if (!takes(KD, VD, block_size, nh, nkv, rows)) return 0;
  const Shares sh = shares_for(rows, nh, nkv, KD, VD, window, keep_first, chunk, max_len);
  if (sh.splits == 1) return 0;
  return (long long)rows * nkv * sh.tiles * sh.splits * sh.heads * (VD + 2);
}

int lq_sink_decode(const bf16_t* q, void* out, const bf16_t* gate, const bf16_t* kcache, const bf16_t* vcache,
                   const SinkArgs& a, int max_len, float* part, long long part_floats, int* tickets, long long tickets_n,
                   hipStream_t stream) {
  if (a.ldq % 4 != 0 || (uintptr_t)q % 8 != 0 || ((uintptr_t)kcache | (uintptr_t)vcache) % 16 != 0 ||
      !takes(a.KD, a.VD, a.BS, a.nh, a.nkv, a.rows))
    return 0;
  Shares sh = shares_for(a.rows, a.nh, a.nkv, a.KD, a.VD, a.window, a.keep_first, a.chunk, max_len);
  const long long need = lq_sink_decode_workspace(a.rows, a.nh, a.nkv, a.KD, a.VD, a.BS, a.window, a.keep_first, a.chunk, max_len);
  if (part == nullptr || need <= 0 || need > part_floats || (uintptr_t)part % 8 != 0)  // (shares are read in pairs)
    sh = shares_for(a.rows, a.nh, a.nkv, a.KD, a.VD, a.window, a.keep_first, a.chunk, 0);
  sh.part = part;
  sh.tickets = (long long)a.rows * a.nkv * sh.tiles <= tickets_n ? tickets : nullptr;
  SinkArgs b = a;
  b.heads_per_tile = a.nh / a.nkv;  // (here: query heads a key head)
  const dim3 grid(a.rows, a.nkv * sh.tiles, sh.splits);
#define LQ_DECODE(KS, VT) launch<KS, VT>(q, out, gate, kcache, vcache, b, sh, grid, stream)
  if (a.KD <= 64 && a.VD <= 64) return LQ_DECODE(2, 4);
  if (a.KD <= 128 && a.VD <= 128) return LQ_DECODE(4, 8);
  if (a.KD <= 128) return LQ_DECODE(4, 16);
  if (a.VD <= 192) return LQ_DECODE(8, 12);
  return LQ_DECODE(8, 16);
#undef LQ_DECODE
}
