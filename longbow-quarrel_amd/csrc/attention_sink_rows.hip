// Prompts of a bfloat16 run through the windowed attention of attention_sink.hip (the same masks, sinks, shaped
// scores, maps and gates), on 32 x 32 score tiles.
//
// A workgroup takes 128 tile rows of one sequence: 32 (4 / heads) rows of the step times 4, 2 or 1 query heads of one
// key head (as many as divide the key head's).  It walks the keys that any of its rows sees by cache blocks
// of 64 positions, which all its threads bring into LDS together (the next block's loads are in flight while this
// one is multiplied; one barrier a block).  A tile of 32 rows belongs to two wavefronts, which take the first and the
// second 32 keys of every block and add their results up through LDS at the end (KS = 2; with KS = 1 one wavefront
// takes both).  What bounded the tiles of 16 rows
// that prompts ran on before (attention_sink.hip, which keeps single tokens and 32-bit runs): every wavefront read
// all its keys and values from the caches itself, and the second product ran in the matrix cores' 32-bit mode at a
// sixteenth of their bfloat16 rate.
//
// v_mfma_f32_32x32x16_bf16: lane l gives A[row l % 32][k (l / 32) * 8 .. + 8] and B[column l % 32][the same k], and
// receives D[(e / 4) * 8 + (l / 32) * 4 + e % 4][l % 32], e < 16.
//   S^T[key][row] = K . Q^T.  Row i of the A tile is the key with bits 2 and 3 of i exchanged: a lane's sixteen
//   scores are then those of keys 16 s + 8 (l / 32) + 0 .. 7 for s = 0, 1, and
//   O^T[d][row] += V^T[d][key] . P^T[key][row] takes eight of its probabilities as they are, with V^T operands of
//   eight neighbouring keys.
// The probabilities stay 32-bit: each is the sum of three bfloat16 numbers (its upper, middle and lower eight bits of
// mantissa, cut off one after the other, exactly), and each part is multiplied with the values, which are bfloat16
// anyway: every product is exact and the sums are 32-bit, as in the 32-bit mode, at three products of sixteen times
// its rate.
//
// LDS rows are whole runs of 16-byte units, unit u of row r stored at u ^ (r or r / 2, modulo 16 or 8) so that the
// rows that sixteen lanes read at once lie in different banks.  Values of positions that were never written count as
// zero, and a tile's rows are of one sequence, so that nothing of another one (a NaN in its cache, for one) reaches it.
//
// A block of 64 keys takes 2.7 microseconds at 128 entries a head, of which the matrix instructions of a SIMD's two
// wavefronts are 0.85: the softmax, the cutting of the probabilities and the round trips through LDS between the
// products bound it.
#include "attention_sink.h"
#include "sequence_parts.h"

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

namespace {

constexpr int BLOCK = 64;                    // positions a cache block
constexpr int SLOTS = 4;                     // tiles of 32 rows a workgroup
constexpr float SLACK = 8.0f;                // the maximum moves when a score lies this far (in powers of two) above it

__device__ inline unsigned pack2(float lo, float hi) {  // round to nearest even
  return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){lo, hi}, bf16x2));
}

__device__ inline float halves_max(float x) {
  auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}
__device__ inline float halves_sum(float x) {
  auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

__device__ inline int wave_least(int v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = min(v, __shfl_xor(v, off, 64));
  return __builtin_amdgcn_readfirstlane(v);
}
__device__ inline int wave_most(int v) { return -wave_least(-v); }

// KD and VD up to 16 KS16 and 32 VT: sizes in between run with zeros behind their keys and values.
template <int KS16, int VT>
struct RowsLds {
  static constexpr int K_UNITS = KS16 * 2, K_BYTES = BLOCK * K_UNITS * 16, V_BYTES = VT * 32 * BLOCK * 2;
  static constexpr int STAGE = K_BYTES + V_BYTES;
  static constexpr int MERGE = SLOTS * (2 * 16 + 2) * 64 * 4;  // two output tiles, maximum and sum of every second wavefront
  static constexpr int BYTES = 2 * STAGE > MERGE ? 2 * STAGE : MERGE;
  __device__ static int k_at(int key, int unit) {
    return key * (K_UNITS * 16) + (K_UNITS >= 16 ? unit ^ (key & 15) : unit ^ ((key >> 1) & 7)) * 16;
  }
  __device__ static int v_at(int d, int unit) { return K_BYTES + d * 128 + (unit ^ ((d >> 1) & 7)) * 16; }
};

template <int KS16, int VT, int KS, bool SHAPED>
__global__ __launch_bounds__(SLOTS * KS * 64, KS) void sink_rows32_kernel(const bf16_t* __restrict__ q, void* __restrict__ out,
                                                                         const bf16_t* __restrict__ gate,
                                                                         const bf16_t* __restrict__ kcache,
                                                                         const bf16_t* __restrict__ vcache,
                                                                         const int* __restrict__ cu_rows, SinkArgs a,
                                                                         int batch, int heads, int tiles) {
  using L = RowsLds<KS16, VT>;
  constexpr int THREADS = SLOTS * KS * 64;
  constexpr int K_PER = (BLOCK * L::K_UNITS + THREADS - 1) / THREADS, V_PER = (VT * 32 * 8 + THREADS - 1) / THREADS;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 31, hf = lane >> 5;
  const int slot = wave & (SLOTS - 1), ks = wave / SLOTS;
  // late tiles, which see the most keys, come first; neighbouring workgroups are different heads, so that a die's L2
  // holds few heads' keys
  const int per_tile = gridDim.x / tiles;
  const Part tile = find_part(cu_rows, batch, 32 * (SLOTS / heads), 1, tiles - 1 - (int)blockIdx.x / per_tile);
  if (tile.rows <= 0) return;  // the whole workgroup
  const int hbase = (int)(blockIdx.x % per_tile) * heads, kvh = hbase / (a.nh / a.nkv);
  const int h = hbase + slot % heads;
  const int nvh = a.nkv / a.maps, vh = kvh / a.maps;
  const int KD = a.KD, VD = a.VD, k_units = KD / 8;
  const long long krow = (long long)a.maps * KD;
  const int my_at = slot / heads * 32 + c;  // this lane's row within the workgroup's: maybe past its last
  const bool mine = my_at < tile.rows;
  const int my_row = tile.first + min(my_at, tile.rows - 1);
  const int my_pos = a.row_pos[my_row], my_lo = first_key(a, my_pos);
  HeadShape hs;
  if constexpr (SHAPED) hs = head_shape(a, h);
  const float c2 = a.scale * LOG2E;

  u32x4 qf[KS16];
#pragma unroll
  for (int kk = 0; kk < KS16; ++kk) {
    const int unit = 2 * kk + hf;
    qf[kk] = unit < k_units ? __builtin_bit_cast(u32x4, load_q8(q + (long long)my_row * a.ldq + h * KD + unit * 8))
                            : (u32x4){0u, 0u, 0u, 0u};
  }
  // (lane i reads the operand row of key i with bits 2 and 3 exchanged)
  const int key_of_lane = (c & ~12) | ((c & 4) << 1) | ((c & 8) >> 1);

  // what the workgroup's rows see together, and what this tile's do
  int lo_min = 0x7fffffff, pos_max = -1;
  for (int i = lane; i < tile.rows; i += 64) {
    const int p = a.row_pos[tile.first + i];
    lo_min = min(lo_min, first_key(a, p)), pos_max = max(pos_max, p);
  }
  lo_min = wave_least(lo_min), pos_max = wave_most(pos_max);
  const int t_lo_min = wave_least(mine ? my_lo : 0x7fffffff), t_lo_max = wave_most(mine ? my_lo : -1);
  const int t_pos_min = wave_least(mine ? my_pos : 0x7fffffff), t_pos_max = wave_most(mine ? my_pos : -1);
  const int* table = a.block_table + (long long)a.seq_slot[tile.seq] * a.bt_stride;
  const int wstart = lo_min / BLOCK * BLOCK;       // first block of the window of any of these rows
  const int kept_end = min(a.keep_first, wstart);  // kept keys that lie below that block

  float m = NONE, l = 0.f;  // the row's running maximum (in powers of two); this lane's share of its sum
  if (a.sink && ks == 0) {
    const SinkStart start = sink_start(a, h);
    m = start.m, l = hf == 0 ? start.l : 0.f;
  }
  f32x16 o[VT];
#pragma unroll
  for (int dt = 0; dt < VT; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[dt][e] = 0.f;

  u32x4 rk[K_PER], rv[V_PER];
  auto fetch = [&](int t0) {
    const long long blk = table[t0 / BLOCK];
    const bf16_t* kb = kcache + (blk * nvh + vh) * BLOCK * krow + (kvh % a.maps) * KD;
    const bf16_t* vb = vcache + (blk * nvh + vh) * (long long)VD * BLOCK;
#pragma unroll
    for (int i = 0; i < K_PER; ++i) {
      const int pc = tid + i * THREADS, key = pc / L::K_UNITS, unit = pc % L::K_UNITS;
      rk[i] = key < BLOCK && unit < k_units ? *(const u32x4*)(kb + key * krow + unit * 8) : (u32x4){0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int i = 0; i < V_PER; ++i) {
      const int pc = tid + i * THREADS;
      rv[i] = pc / 8 < VD ? *(const u32x4*)(vb + pc * 8) : (u32x4){0u, 0u, 0u, 0u};
    }
  };
  auto stash = [&](int t0, unsigned char* stage) {
#pragma unroll
    for (int i = 0; i < K_PER; ++i) {
      const int pc = tid + i * THREADS, key = pc / L::K_UNITS, unit = pc % L::K_UNITS;
      if (key < BLOCK) *(u32x4*)(stage + L::k_at(key, unit)) = rk[i];
    }
    const bool tail = t0 + BLOCK - 1 > pos_max;
#pragma unroll
    for (int i = 0; i < V_PER; ++i) {
      const int pc = tid + i * THREADS, d = pc / 8, unit = pc % 8;
      if (d >= VT * 32) continue;
      u32x4 v = rv[i];
      if (tail) {  // (0 times what lies in unwritten memory may be NaN)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (t0 + unit * 8 + 2 * e > pos_max) v[e] &= 0xffff0000u;
          if (t0 + unit * 8 + 2 * e + 1 > pos_max) v[e] &= 0x0000ffffu;
        }
      }
      *(u32x4*)(stage + L::v_at(d, unit)) = v;
    }
  };

  int t0 = kept_end > 0 ? 0 : wstart, turn = 0;
  fetch(t0);
  stash(t0, smem);
  __syncthreads();
  while (true) {
    int next = t0 + BLOCK;
    if (next >= kept_end && next < wstart) next = wstart;  // from the kept first tokens on to the window
    const bool more = next <= pos_max;
    if (more) fetch(next);
    const unsigned char* cur = smem + turn * L::STAGE;
#pragma unroll
    for (int half = KS == 2 ? ks : 0; half < (KS == 2 ? ks + 1 : 2); ++half) {
      const int tw = t0 + 32 * half;  // this wavefront's 32 keys
      if (tw <= t_pos_max && (tw + 31 >= t_lo_min || tw < a.keep_first)) {
        f32x16 sc;
#pragma unroll
        for (int e = 0; e < 16; ++e) sc[e] = 0.f;
        u32x4 kf[KS16];
#pragma unroll
        for (int kk = 0; kk < KS16; ++kk) kf[kk] = *(const u32x4*)(cur + L::k_at(32 * half + key_of_lane, 2 * kk + hf));
#pragma unroll
        for (int kk = 0; kk < KS16; ++kk)
          sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(kf[kk]), as_bf16x8(qf[kk]), sc, 0, 0, 0);
        // sc[e] is the score of key tw + 16 (e / 8) + 8 hf + e % 8
        const bool masked = !(tw + 31 <= t_pos_min && (tw >= t_lo_max || tw + 31 < a.keep_first));
        if constexpr (SHAPED) {
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const int t = tw + 16 * (e / 8) + 8 * hf + e % 8;
            sc[e] = shaped<false>(sc[e], max(my_pos - t, 0), hs) * LOG2E;
          }
        } else {
#pragma unroll
          for (int e = 0; e < 16; ++e) sc[e] *= c2;
        }
        if (masked) {
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const int t = tw + 16 * (e / 8) + 8 * hf + e % 8;
            if (!(mine && t <= my_pos && (t >= my_lo || t < a.keep_first))) sc[e] = -INFINITY;
          }
        }
        float top = sc[0];
#pragma unroll
        for (int e = 1; e < 16; ++e) top = fmaxf(top, sc[e]);
        top = halves_max(top);
        if (__any(top > m + SLACK)) {
          // (each row by its own scores: its roundings do not depend on which rows share the tile)
          const float m_new = top > m + SLACK ? top : m, alpha = __builtin_amdgcn_exp2f(m - m_new);
          l *= alpha;
          m = m_new;
#pragma unroll
          for (int dt = 0; dt < VT; ++dt)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[dt][e] *= alpha;
        }
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          sc[e] = __builtin_amdgcn_exp2f(sc[e] - m);
          sum += sc[e];
        }
        l += sum;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          u32x4 vf[VT];
#pragma unroll
          for (int dt = 0; dt < VT; ++dt) vf[dt] = *(const u32x4*)(cur + L::v_at(32 * dt + c, 4 * half + 2 * s + hf));
          u32x4 part[3];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float p0 = sc[8 * s + 2 * j], p1 = sc[8 * s + 2 * j + 1];
            const float q0 = below_upper(p0), q1 = below_upper(p1);
            part[0][j] = upper2(p0, p1);
            part[1][j] = upper2(q0, q1);
            part[2][j] = upper2(below_upper(q0), below_upper(q1));
          }
#pragma unroll
          for (int i = 2; i >= 0; --i)
#pragma unroll
            for (int dt = 0; dt < VT; ++dt)
              o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(vf[dt]), as_bf16x8(part[i]), o[dt], 0, 0, 0);
        }
      }
    }
    // Nobody reads the other stage: its last readers passed the barrier below a block ago.
    if (more) stash(next, smem + (turn ^ 1) * L::STAGE);
    __syncthreads();
    if (!more) break;
    t0 = next, turn ^= 1;
  }

  if constexpr (KS == 2) {
    // the second wavefront's sums go to the first, two output tiles at a time (the stages are no longer read)
    float* theirs = (float*)smem + slot * (2 * 16 + 2) * 64 + lane;
    float f0 = 1.f, f1 = 0.f;
#pragma unroll
    for (int d0 = 0; d0 < VT; d0 += 2) {
      if (d0 > 0) __syncthreads();
      if (ks == 1) {
#pragma unroll
        for (int dt = d0; dt < d0 + 2 && dt < VT; ++dt)
#pragma unroll
          for (int e = 0; e < 16; ++e) theirs[((dt - d0) * 16 + e) * 64] = o[dt][e];
        if (d0 == 0) theirs[32 * 64] = m, theirs[33 * 64] = l;
      }
      __syncthreads();
      if (ks == 0) {
        if (d0 == 0) {
          const float m1 = theirs[32 * 64], m_all = fmaxf(m, m1);
          f0 = __builtin_amdgcn_exp2f(m - m_all), f1 = __builtin_amdgcn_exp2f(m1 - m_all);
          l = l * f0 + theirs[33 * 64] * f1;
        }
#pragma unroll
        for (int dt = d0; dt < d0 + 2 && dt < VT; ++dt)
#pragma unroll
          for (int e = 0; e < 16; ++e) o[dt][e] = o[dt][e] * f0 + theirs[((dt - d0) * 16 + e) * 64] * f1;
      }
    }
  }
  l = halves_sum(l);
  if (ks == 0 && mine) {
    float f = 1.0f / l;
    if (gate != nullptr) f /= 1.f + expf(-to_f32(gate[(long long)my_row * a.ldg + h]));
    const float* wg = a.wide_gate != nullptr ? a.wide_gate + (long long)my_row * a.ldwg + h * VD : nullptr;
    const long long orow = (long long)my_row * a.ldo + h * VD;
#pragma unroll
    for (int dt = 0; dt < VT; ++dt)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int d = dt * 32 + g4 * 8 + hf * 4;
        if (d < VD) {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = o[dt][g4 * 4 + e] * f;
          if (wg != nullptr) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] /= 1.f + expf(-wg[d + e]);
          }
          if (a.out_f32) *(f32x4*)((float*)out + orow + d) = (f32x4){v[0], v[1], v[2], v[3]};
          else *(u32x2*)((bf16_t*)out + orow + d) = (u32x2){pack2(v[0], v[1]), pack2(v[2], v[3])};
        }
      }
  }
}

template <int KS16, int VT, int KS>
int launch(const bf16_t* q, void* out, const bf16_t* gate, const bf16_t* kcache, const bf16_t* vcache, const int* cu_rows,
           const SinkArgs& a, int batch, int heads, hipStream_t stream) {
  using L = RowsLds<KS16, VT>;
  const int tiles = a.rows / (32 * (SLOTS / heads)) + batch;  // no fewer: a sequence's last tile may be part-filled
  const long long blocks = (long long)tiles * (a.nh / heads);
  LQ_REQUIRE(blocks <= 0x7fffffff, "sink_attention: too many rows");
  const bool with_shape = scores_shaped(a.shape);
  const auto kernel = with_shape ? sink_rows32_kernel<KS16, VT, KS, true> : sink_rows32_kernel<KS16, VT, KS, false>;
  static bool configured[2] = {false, false};
  if (!configured[with_shape]) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, L::BYTES);
    if (e != hipSuccess) {
      lq_set_error("sink_attention: cannot reserve %d bytes of LDS: %s", L::BYTES, hipGetErrorString(e));
      return -2;
    }
    configured[with_shape] = true;
  }
  kernel<<<(int)blocks, SLOTS * KS * 64, L::BYTES, stream>>>(q, out, gate, kcache, vcache, cu_rows, a, batch, heads, tiles);
  LQ_CHECK_LAUNCH("sink_attention(32 x 32)");
  return 1;
}

}  // namespace

int lq_sink_rows32(const bf16_t* q, void* out, const bf16_t* gate, const bf16_t* kcache, const bf16_t* vcache,
                   const int* cu_rows, const SinkArgs& a, int batch, hipStream_t stream) {
  // Which launches: every prompt step of these alignments whose tile has the registers (keys and values both beyond
  // 128 and 192 entries stay with the tiles of 16 rows).  Each size runs at the smallest of four shapes that holds it.
  // Microseconds a launch before (tiles of 16 rows) and now, 16 heads over 4, bfloat16:
  //   128 entries a head, window 1 024: 17 rows 15.2 -> 9.8, 200 rows 16.8 -> 15.1, 512 rows 38.9 -> 23.0, 2 048 rows
  //   255 -> 47, 4 096 rows 503 -> 89; 8 prompts of 2 rows behind 1 000 keys each 85 -> 35; causal, three prompts of
  //   257, 878 and 1 500 rows 256 -> 54; two maps over values of 256, 8 prompts of 512 rows 329 -> 84; a latent of 192
  //   with keys of 256, one key head, 3 597 rows 300 -> 79; capped scores and a table of biases, 2 000 rows 226 -> 90.
  // Values of more than 128 or keys of more than 128 entries have no registers for two wavefronts a SIMD: a wavefront
  // there takes both halves of a block (two wavefronts, spilling: 126 and 146 microseconds for the two cases above).
  // 32-bit results against 64 bits: relative error 1.9e-7 (2.2e-7 before) at 2 048 rows.
  // Rows of q lie any multiple of 4 entries apart: they may be part of a product's wider rows (a gate a head behind 12
  // heads: 2 316 entries).
  const bool aligned = a.ldq % 4 == 0 && (uintptr_t)q % 8 == 0 && ((uintptr_t)kcache | (uintptr_t)vcache) % 16 == 0 &&
                       a.ldo % 4 == 0 && (uintptr_t)out % (a.out_f32 ? 16 : 8) == 0;
  if (!aligned || a.BS != BLOCK || a.KD % 8 != 0 || a.VD % 8 != 0 || a.KD > 256 || a.VD > 256 ||
      (a.KD > 128 && a.VD > 192))
    return 0;
  const int group = a.nh / a.nkv, heads = group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
#define LQ_ROWS32(KS16, VT, KS) launch<KS16, VT, KS>(q, out, gate, kcache, vcache, cu_rows, a, batch, heads, stream)
  if (a.KD <= 64 && a.VD <= 64) return LQ_ROWS32(4, 2, 2);
  if (a.KD <= 128 && a.VD <= 128) return LQ_ROWS32(8, 4, 2);
  if (a.KD <= 128) return LQ_ROWS32(8, 8, 1);
  return LQ_ROWS32(16, 6, 1);
#undef LQ_ROWS32
}
