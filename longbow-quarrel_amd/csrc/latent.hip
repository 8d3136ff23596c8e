// Kernels around attention through a cached latent: an RMS norm over a run of columns of a wider row, and a
// rotation by position of a part of every head's vector with a choice of pairing.  Both read 32-bit results of a
// product and write in the dtype of whatever reads them next, into a place of the caller's (a run of columns of a
// wider row), so that a norm, a rotation and the assembly of a cached row or of a query need no copies.
#include "common.h"

namespace {

// out[r, :] = src[r, :] / sqrt(mean(src[r, :]^2) + eps) * w; one workgroup a row
template <typename T>
__global__ __launch_bounds__(256) void rmsnorm_cols_kernel(const float* __restrict__ src, int lds_, const float* __restrict__ w,
                                                           float eps, T* __restrict__ out, int ldo, int n) {
  __shared__ float red[16];
  const float* s = src + (long long)blockIdx.x * lds_;
  T* o = out + (long long)blockIdx.x * ldo;
  float acc = 0.f;
  for (int i = threadIdx.x; i < n; i += 256) acc = fmaf(s[i], s[i], acc);
  const float inv = 1.f / sqrtf(block_sum(acc, red) / (float)n + eps);
  for (int i = threadIdx.x; i < n; i += 256) o[i] = from_f32<T>(s[i] * inv * w[i]);
}

// Row r, head h: the vector src[r, h * size .. + size) goes to out[r, h * ohs .. + size); its first `dims` entries
// are rotated by the angles row_pos[r] * freqs[j], in pairs (j, j + dims / 2) or (2 j, 2 j + 1): (u, v) ->
// (u c - v s, v c + u s) with c and s times `mag`; the rest pass.  Angles in double, reduced to [-pi, pi] before
// the 32-bit sine and cosine.
template <typename T>
__global__ __launch_bounds__(128) void rotary_kernel(const float* __restrict__ src, int lds_, T* __restrict__ out, int ldo,
                                                     int heads, int size, int ohs, int dims, int interleaved,
                                                     const double* __restrict__ freqs, float mag,
                                                     const int* __restrict__ row_pos) {
  extern __shared__ float cs[];  // cos[dims / 2], sin[dims / 2]
  const int r = blockIdx.x, half = dims / 2;
  const int p = row_pos[r];
  for (int j = threadIdx.x; j < half; j += blockDim.x) {
    const double a = (double)p * freqs[j];
    const double n = rint(a * 0.15915494309189533577);
    double rem = fma(-n, 6.283185307179586232, a);
    rem = fma(-n, 2.4492935982947064e-16, rem);
    float sn, c;
    sincosf((float)rem, &sn, &c);
    cs[j] = c * mag;
    cs[half + j] = sn * mag;
  }
  __syncthreads();
  const float* s = src + (long long)r * lds_;
  T* o = out + (long long)r * ldo;
  for (int e = threadIdx.x; e < heads * size; e += blockDim.x) {
    const int h = e / size, i = e - h * size;
    const float* v = s + h * size;
    float res;
    if (i >= dims) {
      res = v[i];
    } else {
      int j, mate;
      bool first;
      if (interleaved) j = i >> 1, first = !(i & 1), mate = i ^ 1;
      else first = i < half, j = first ? i : i - half, mate = first ? i + half : i - half;
      const float c = cs[j], sn = cs[half + j];
      res = first ? v[i] * c - v[mate] * sn : v[i] * c + v[mate] * sn;
    }
    o[h * ohs + i] = from_f32<T>(res);
  }
}

// Queries, keys and values of a step's rows, from the 32-bit result of their one product to what the attention
// kernel and the cache read.  src [rows, (H + G) D + G V]: H query heads, G key heads, G value heads.  Of every query
// and key head the first `dims` entries are rotated as in `rotary_kernel`; then, with norm_eps >= 0, the whole head
// is divided by its root mean square over D (eps inside the root); values pass.  gridDim.y workgroups a row share
// its heads and values out (one where the rows alone fill the chip); a wavefront takes a head at a time (its sum of
// squares is the wavefront's fixed tree, so it depends on the row alone, not on how the heads were shared out).
template <typename T>
__global__ __launch_bounds__(256) void rotary_qkv_kernel(const float* __restrict__ src, int lds_, T* __restrict__ q_out,
                                                         int ldq, T* __restrict__ k_out, int ldk, T* __restrict__ v_out,
                                                         int ldv, int H, int G, int D, int VW, int dims, int interleaved,
                                                         const double* __restrict__ freqs, float mag, float norm_eps,
                                                         const int* __restrict__ row_pos) {
  extern __shared__ float cs[];  // cos[dims / 2], sin[dims / 2]
  const int r = blockIdx.x, half = dims / 2;
  const int p = row_pos[r];
  for (int j = threadIdx.x; j < half; j += blockDim.x) {
    const double a = (double)p * freqs[j];
    const double n = rint(a * 0.15915494309189533577);
    double rem = fma(-n, 6.283185307179586232, a);
    rem = fma(-n, 2.4492935982947064e-16, rem);
    float sn, c;
    sincosf((float)rem, &sn, &c);
    cs[j] = c * mag;
    cs[half + j] = sn * mag;
  }
  __syncthreads();
  const float* s = src + (long long)r * lds_;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  for (int h = blockIdx.y * waves + wave; h < H + G; h += waves * gridDim.y) {
    const float* v = s + h * D;
    T* o = h < H ? q_out + (long long)r * ldq + h * D : k_out + (long long)r * ldk + (h - H) * D;
    auto turned = [&](int i) -> float {
      if (i >= dims) return v[i];
      int j, mate;
      bool first;
      if (interleaved) j = i >> 1, first = !(i & 1), mate = i ^ 1;
      else first = i < half, j = first ? i : i - half, mate = first ? i + half : i - half;
      const float c = cs[j], sn = cs[half + j];
      return first ? v[i] * c - v[mate] * sn : v[i] * c + v[mate] * sn;
    };
    float inv = 1.f;
    if (norm_eps >= 0.f) {
      float ss = 0.f;
      for (int i = lane; i < D; i += 64) {
        const float t = turned(i);
        ss = fmaf(t, t, ss);
      }
      inv = 1.f / sqrtf(wave_sum(ss) / (float)D + norm_eps);
    }
    for (int i = lane; i < D; i += 64) o[i] = from_f32<T>(turned(i) * inv);
  }
  const float* vs = s + (H + G) * D;
  T* vo = v_out + (long long)r * ldv;
  for (int e = blockIdx.y * blockDim.x + threadIdx.x; e < VW; e += blockDim.x * gridDim.y) vo[e] = from_f32<T>(vs[e]);
}

// Queries, keys and values of a step's rows, from the 32-bit result of their one product to what the attention kernel
// reads and straight into the paged cache.  src [rows, H D + G D (+ G V)]; `bias` (a number a column, or null) is added
// first.  With `cs` (cos and sin of the row's angles, [rows][dims / 2][2]) the first `dims` entries of every query and key
// unit are then rotated, pairs and magnitude as in `rotary_kernel` (units of a head, or of an equal part of one: the maps of
// differential attention, whose keys lie side by side in a head's cache row).  q and k are normed in units of `unit_q` and `unit_k` entries (a head each, or the whole row of
// all heads; units divided by their root mean square, eps inside the root, times a weight of the unit's size), values in
// units of a head without a weight (`norm_v`) or not at all; `v_from_k`: there are no value columns, the values are the
// keys as they are before rotation and norm.  k and v go to the row's position in the cache (K [block][G][BS][D],
// V [block][G][V][BS]); kcache null: q alone is wanted.  A wavefront takes a unit (WIDE: a workgroup), so a unit's sum of
// squares is one fixed tree whatever else is in the launch.
struct QkvUnits {
  int lds, ldq, H, G, D, V, unit_q, unit_k, norm_qk, norm_v, v_from_k;
  float eps;
  const float *bias, *wq, *wk;
  const int *row_pos, *row_seq, *seq_slot, *block_table;
  int bt_stride, BS;
  int unit_v;  // value entries a unit
  const float* cs;
  int dims, interleaved;
  float mag;
};

// Entry i of a head (v its value, `mate` what the entry of its pair holds) after the rotation.
__device__ inline float turned_entry(const QkvUnits& a, const float* cs, int i, float v, float mate) {
  const int half = a.dims >> 1, j = a.interleaved ? i >> 1 : i < half ? i : i - half;
  const bool first = a.interleaved ? !(i & 1) : i < half;
  const float c = cs[2 * j] * a.mag, s = cs[2 * j + 1] * a.mag;
  return first ? v * c - mate * s : v * c + mate * s;
}

__device__ inline int pair_mate(const QkvUnits& a, int i) {
  return a.interleaved ? i ^ 1 : i < (a.dims >> 1) ? i + (a.dims >> 1) : i - (a.dims >> 1);
}

template <typename T, bool WIDE>
__global__ __launch_bounds__(256) void qkv_norm_store_kernel(const float* __restrict__ src, T* __restrict__ q_out,
                                                             T* __restrict__ kcache, T* __restrict__ vcache, QkvUnits a) {
  __shared__ float red[16];
  const int r = blockIdx.x;
  const int i0 = WIDE ? threadIdx.x : threadIdx.x & 63;
  constexpr int STEP = WIDE ? 256 : 64;
  int u = WIDE ? (int)blockIdx.y : (int)blockIdx.y * 4 + (int)(threadIdx.x >> 6);
  const int QW = a.H * a.D, KW = a.G * a.D, VW = a.G * a.V, unit_v = a.unit_v;
  const int nq = QW / a.unit_q, nk = kcache != nullptr ? KW / a.unit_k : 0, nv = kcache != nullptr ? VW / unit_v : 0;
  if (u >= nq + nk + nv) return;  // (WIDE: the whole workgroup)
  const int which = u < nq ? 0 : u < nq + nk ? 1 : 2;
  int n, at, col;  // the unit's entries, its first entry among its kind, its first column in src
  const float* w = nullptr;
  bool norm = a.norm_qk != 0;
  if (which == 0) n = a.unit_q, at = u * n, col = at, w = a.wq;
  else if (which == 1) n = a.unit_k, at = (u - nq) * n, col = QW + at, w = a.wk;
  else n = unit_v, at = (u - nq - nk) * n, col = (a.v_from_k ? QW : QW + KW) + at, norm = a.norm_v != 0;
  const float* s = src + (long long)r * a.lds + col;
  const float* b = a.bias != nullptr ? a.bias + col : nullptr;
  const float* cs = a.cs != nullptr && which != 2 ? a.cs + (long long)r * a.dims : nullptr;
  auto entry = [&](int i) -> float {
    const float v = b != nullptr ? s[i] + b[i] : s[i];
    if (cs == nullptr || i >= a.dims) return v;
    const int m = pair_mate(a, i);
    return turned_entry(a, cs, i, v, b != nullptr ? s[m] + b[m] : s[m]);
  };
  float inv = 1.f;
  if (norm) {
    float ss = 0.f;
    for (int i = i0; i < n; i += STEP) {
      const float v = entry(i);
      ss = fmaf(v, v, ss);
    }
    inv = 1.f / sqrtf((WIDE ? block_sum(ss, red) : wave_sum(ss)) / (float)n + a.eps);
  }
  long long blk = 0;
  int off = 0;
  if (which != 0) {
    const int p = a.row_pos[r];
    blk = a.block_table[(long long)a.seq_slot[a.row_seq[r]] * a.bt_stride + p / a.BS];
    off = p % a.BS;
  }
  for (int i = i0; i < n; i += STEP) {
    float v = entry(i);
    if (norm) v *= inv;
    if (w != nullptr) v *= w[i];
    const int e = at + i;
    if (which == 0) {
      q_out[(long long)r * a.ldq + e] = from_f32<T>(v);
    } else if (which == 1) {
      const int g = e / a.D;
      kcache[((blk * a.G + g) * a.BS + off) * (long long)a.D + e - g * a.D] = from_f32<T>(v);
    } else {
      const int g = e / a.V;
      vcache[((blk * a.G + g) * (long long)a.V + e - g * a.V) * a.BS + off] = from_f32<T>(v);
    }
  }
}

// The same with a unit's entries in registers (a unit is read once), for units, head sizes and rows in fours: PER runs of
// four entries a thread.
template <typename T, bool WIDE, int PER>
__global__ __launch_bounds__(256) void qkv_norm_store4_kernel(const float* __restrict__ src, T* __restrict__ q_out,
                                                              T* __restrict__ kcache, T* __restrict__ vcache, QkvUnits a) {
  __shared__ float red[16];
  const int r = blockIdx.x;
  const int i0 = WIDE ? threadIdx.x : threadIdx.x & 63;
  constexpr int STEP = WIDE ? 256 : 64;
  const int u = WIDE ? (int)blockIdx.y : (int)blockIdx.y * 4 + (int)(threadIdx.x >> 6);
  const int QW = a.H * a.D, KW = a.G * a.D, VW = a.G * a.V, unit_v = a.unit_v;
  const int nq = QW / a.unit_q, nk = kcache != nullptr ? KW / a.unit_k : 0, nv = kcache != nullptr ? VW / unit_v : 0;
  if (u >= nq + nk + nv) return;  // (WIDE: the whole workgroup)
  const int which = u < nq ? 0 : u < nq + nk ? 1 : 2;
  int n, at, col;
  const float* w = nullptr;
  bool norm = a.norm_qk != 0;
  if (which == 0) n = a.unit_q, at = u * n, col = at, w = a.wq;
  else if (which == 1) n = a.unit_k, at = (u - nq) * n, col = QW + at, w = a.wk;
  else n = unit_v, at = (u - nq - nk) * n, col = (a.v_from_k ? QW : QW + KW) + at, norm = a.norm_v != 0;
  const float4* s = (const float4*)(src + (long long)r * a.lds + col);
  const float4* b = a.bias != nullptr ? (const float4*)(a.bias + col) : nullptr;
  const int quads = n / 4;
  float4 v[PER];
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = i0 + j * STEP;
    v[j] = i < quads ? s[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    if (b != nullptr && i < quads) {
      const float4 add = b[i];
      v[j].x += add.x, v[j].y += add.y, v[j].z += add.z, v[j].w += add.w;
    }
  }
  if (a.cs != nullptr && which != 2) {
    const float* cs = a.cs + (long long)r * a.dims;
    const float* sf = (const float*)s;
    const float* bf = (const float*)b;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int e = 4 * (i0 + j * STEP);
      if (e >= n || e >= a.dims) continue;
      float* x = &v[j].x;
      float mate[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (a.interleaved) mate[k] = x[k ^ 1];
        else {
          const int m = e + k < a.dims ? pair_mate(a, e + k) : e;
          mate[k] = bf != nullptr ? sf[m] + bf[m] : sf[m];
        }
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (e + k < a.dims) x[k] = turned_entry(a, cs, e + k, x[k], mate[k]);
    }
  }
  long long blk = 0;
  int off = 0;
  if (which != 0) {
    const int p = a.row_pos[r];
    blk = a.block_table[(long long)a.seq_slot[a.row_seq[r]] * a.bt_stride + p / a.BS];
    off = p % a.BS;
  }
  float inv = 1.f;
  if (norm) {
#pragma unroll
    for (int j = 0; j < PER; ++j)
      ss = fmaf(v[j].x, v[j].x, fmaf(v[j].y, v[j].y, fmaf(v[j].z, v[j].z, fmaf(v[j].w, v[j].w, ss))));
    inv = 1.f / sqrtf((WIDE ? block_sum(ss, red) : wave_sum(ss)) / (float)n + a.eps);
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = i0 + j * STEP;
    if (i >= quads) continue;
    float x0 = v[j].x * inv, x1 = v[j].y * inv, x2 = v[j].z * inv, x3 = v[j].w * inv;
    if (w != nullptr) {
      const float4 wv = ((const float4*)w)[i];
      x0 *= wv.x, x1 *= wv.y, x2 *= wv.z, x3 *= wv.w;
    }
    const int e = at + 4 * i;
    if (which == 2) {
      const int g = e / a.V;
      T* o = vcache + ((blk * a.G + g) * (long long)a.V + e - g * a.V) * a.BS + off;
      o[0] = from_f32<T>(x0), o[a.BS] = from_f32<T>(x1), o[2 * a.BS] = from_f32<T>(x2), o[3 * a.BS] = from_f32<T>(x3);
      continue;
    }
    const int g = e / a.D;
    T* o = which == 0 ? q_out + (long long)r * a.ldq + e : kcache + ((blk * a.G + g) * a.BS + off) * (long long)a.D + e - g * a.D;
    if constexpr (sizeof(T) == 4) {
      *(float4*)o = make_float4(x0, x1, x2, x3);
    } else {
      uint2 packed;
      packed.x = (uint32_t)f32_to_bf16(x0).bits | ((uint32_t)f32_to_bf16(x1).bits << 16);
      packed.y = (uint32_t)f32_to_bf16(x2).bits | ((uint32_t)f32_to_bf16(x3).bits << 16);
      *(uint2*)o = packed;
    }
  }
}

// The same for many rows, units of 4 LANES entries (a query or key head, or an equal part of one) and value heads of 4 VLANES: LANES
// lanes a unit.  Queries and keys: a thread takes four rows of its
// unit, all asked for together.  Values lie in the cache with the positions of an entry side by side: the first row of every
// aligned run of eight positions (or of a sequence) takes the run, eight rows at once, and writes 16 bytes an entry where the run is
// whole, in the place of a 2-byte store an entry and row.  A unit's sum of squares is the kernel's above, bit for bit.
constexpr int QKV_ROWS = 4, RUN = 8;

__device__ inline void store_run8(bf16_t* o, const float (&v)[RUN]) {
  uint4 packed;
  uint32_t* u = &packed.x;
#pragma unroll
  for (int i = 0; i < 4; ++i) u[i] = (uint32_t)f32_to_bf16(v[2 * i]).bits | ((uint32_t)f32_to_bf16(v[2 * i + 1]).bits << 16);
  *(uint4*)o = packed;
}
__device__ inline void store_run8(float* o, const float (&v)[RUN]) {
  ((float4*)o)[0] = make_float4(v[0], v[1], v[2], v[3]), ((float4*)o)[1] = make_float4(v[4], v[5], v[6], v[7]);
}

template <int LANES>
__device__ inline float unit_sum(float v) {
#pragma unroll
  for (int off = LANES / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

template <typename T, int LANES, int VLANES>
__global__ __launch_bounds__(256) void qkv_norm_store_rows_kernel(const float* __restrict__ src, T* __restrict__ q_out,
                                                                  T* __restrict__ kcache, T* __restrict__ vcache, QkvUnits a, int rows,
                                                                  int qk_blocks) {
  constexpr int UNITS = 256 / LANES, N = 4 * LANES, VUNITS = 256 / VLANES, VN = 4 * VLANES;
  const int QW = a.H * a.D, KW = a.G * a.D;
  const bool stored = kcache != nullptr;
  auto fetch = [&](int r, int col) {
    float4 v = *(const float4*)(src + (long long)r * a.lds + col);
    if (a.bias != nullptr) {
      const float4 add = *(const float4*)(a.bias + col);
      v.x += add.x, v.y += add.y, v.z += add.z, v.w += add.w;
    }
    return v;
  };
  auto squares = [](const float4& v) { return fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, fmaf(v.w, v.w, 0.f)))); };
  if ((int)blockIdx.x < qk_blocks) {
    const int lane = threadIdx.x % LANES, mine = threadIdx.x / LANES, e0 = 4 * lane, parts = a.D / N, queries = a.H * parts;
    const int units = queries + (stored ? a.G * parts : 0), per_rows = (units + UNITS - 1) / UNITS;
    const int u = (int)blockIdx.x % per_rows * UNITS + mine, r0 = (int)blockIdx.x / per_rows * QKV_ROWS;
    if (u >= units) return;
    const bool is_q = u < queries;
    const int col = u * N;  // (keys lie behind the queries)
    float4 v[QKV_ROWS];
#pragma unroll
    for (int j = 0; j < QKV_ROWS; ++j) v[j] = fetch(min(r0 + j, rows - 1), col + e0);
    const float* w = is_q ? a.wq : a.wk;
    const float4 gain = w != nullptr ? *(const float4*)(w + e0) : make_float4(1.f, 1.f, 1.f, 1.f);
#pragma unroll
    for (int j = 0; j < QKV_ROWS; ++j) {
      const int r = min(r0 + j, rows - 1);
      float x[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
      if (a.cs != nullptr && e0 < a.dims) {
        const float* cs = a.cs + (long long)r * a.dims;
        const float *sf = src + (long long)r * a.lds + col, *bf = a.bias != nullptr ? a.bias + col : nullptr;
        float mate[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (a.interleaved) {
            mate[k] = x[k ^ 1];
          } else {
            const int m = e0 + k < a.dims ? pair_mate(a, e0 + k) : e0;
            mate[k] = bf != nullptr ? sf[m] + bf[m] : sf[m];
          }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (e0 + k < a.dims) x[k] = turned_entry(a, cs, e0 + k, x[k], mate[k]);
      }
      if (a.norm_qk) {
        const float inv = 1.f / sqrtf(unit_sum<LANES>(squares(make_float4(x[0], x[1], x[2], x[3]))) / (float)N + a.eps);
        x[0] *= inv, x[1] *= inv, x[2] *= inv, x[3] *= inv;
      }
      if (w != nullptr) x[0] *= gain.x, x[1] *= gain.y, x[2] *= gain.z, x[3] *= gain.w;
      if (r0 + j >= rows) continue;
      T* o;
      if (is_q) {
        o = q_out + (long long)r * a.ldq + col + e0;
      } else {
        const int p = a.row_pos[r];
        const long long blk = a.block_table[(long long)a.seq_slot[a.row_seq[r]] * a.bt_stride + p / a.BS];
        const int ku = u - queries, head = ku / parts;
        o = kcache + ((blk * a.G + head) * a.BS + p % a.BS) * (long long)a.D + (ku - head * parts) * N + e0;
      }
      if constexpr (sizeof(T) == 4) {
        *(float4*)o = make_float4(x[0], x[1], x[2], x[3]);
      } else {
        uint2 packed;
        packed.x = (uint32_t)f32_to_bf16(x[0]).bits | ((uint32_t)f32_to_bf16(x[1]).bits << 16);
        packed.y = (uint32_t)f32_to_bf16(x[2]).bits | ((uint32_t)f32_to_bf16(x[3]).bits << 16);
        *(uint2*)o = packed;
      }
    }
    return;
  }
  // values (V = VN entries a head)
  const int e0 = 4 * (threadIdx.x % VLANES), per_row = (a.G + VUNITS - 1) / VUNITS, at = (int)blockIdx.x - qk_blocks;
  const int r = at / per_row, u = at % per_row * VUNITS + (int)threadIdx.x / VLANES;
  const int p = a.row_pos[r], seq = a.row_seq[r];
  if (p % RUN != 0 && r > 0 && a.row_seq[r - 1] == seq && a.row_pos[r - 1] == p - 1) return;  // (the whole workgroup: another row takes it)
  const int i0 = threadIdx.x & 63, ri = min(r + i0, rows - 1);  // (a lane looks at a row of the run: one trip to memory)
  const bool follows = i0 < RUN - p % RUN && r + i0 < rows && a.row_seq[ri] == seq && a.row_pos[ri] == p + i0;
  const int n = __ffsll(~(unsigned long long)__ballot(follows)) - 1;  // rows of the run, one at least
  if (u >= a.G) return;
  const int col = (a.v_from_k ? QW : QW + KW) + u * VN + e0;
  float4 v[RUN];
#pragma unroll
  for (int i = 0; i < RUN; ++i) v[i] = fetch(r + min(i, n - 1), col);
  if (a.norm_v)
#pragma unroll
    for (int i = 0; i < RUN; ++i) {
      const float inv = 1.f / sqrtf(unit_sum<VLANES>(squares(v[i])) / (float)VN + a.eps);
      v[i].x *= inv, v[i].y *= inv, v[i].z *= inv, v[i].w *= inv;
    }
  const long long blk = a.block_table[(long long)a.seq_slot[seq] * a.bt_stride + p / a.BS];
  T* o = vcache + ((blk * a.G + u) * (long long)VN + e0) * a.BS + p % a.BS;
#pragma unroll
  for (int k = 0; k < 4; ++k, o += a.BS) {
    float x[RUN];
#pragma unroll
    for (int i = 0; i < RUN; ++i) x[i] = k == 0 ? v[i].x : k == 1 ? v[i].y : k == 2 ? v[i].z : v[i].w;
    if (n == RUN) {
      store_run8(o, x);
    } else {
#pragma unroll
      for (int i = 0; i < RUN; ++i)
        if (i < n) o[i] = from_f32<T>(x[i]);
    }
  }
}

// A product a head: out[r, h ohs + n] = sum_k x[r, h K + k] w[h, n, k], bfloat16 operands on
// v_mfma_f32_16x16x16_bf16 or 16x16x32 (exact products, 32-bit sums).  A workgroup of four wavefronts takes 64 rows by 64
// columns of one head; a wavefront 16 rows by the 64 columns, its operands straight from memory (a head's weight
// is small and stays in the caches; the four wavefronts read the same columns).  K in ascending steps: a
// row's sums do not depend on what else is in the launch.
typedef short bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

// A run of STEP / 4 neighbouring k of one row, the operand of a matrix instruction; 32-bit numbers rounded to nearest even.
template <int STEP>
__device__ inline auto run_of_k(const bf16_t* p) {
  if constexpr (STEP == 32) return __builtin_bit_cast(bf16x8_t, *(const uint4*)p);
  else return __builtin_bit_cast(bf16x4_t, *(const uint2*)p);
}
__device__ inline uint32_t rounded2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){a, b}, bf16x2_t));
}
template <int STEP>
__device__ inline auto run_of_k(const float* p) {
  const float4 a = *(const float4*)p;
  if constexpr (STEP == 32) {
    const float4 b = *(const float4*)(p + 4);
    return __builtin_bit_cast(bf16x8_t, make_uint4(rounded2(a.x, a.y), rounded2(a.z, a.w), rounded2(b.x, b.y), rounded2(b.z, b.w)));
  } else {
    return __builtin_bit_cast(bf16x4_t, make_uint2(rounded2(a.x, a.y), rounded2(a.z, a.w)));
  }
}

// FEW: at most 16 rows, and the four wavefronts take 16 of the 64 columns each (else 16 of 64 rows): single tokens are bound by
// one wavefront's chain of loads and products.  STEP: k an instruction, 32 where K is a multiple of it and operands lie on 16
// bytes.  16 heads of 128 x 192, from 16 k and 64 columns a wavefront: 8 rows 5.05 -> 2.85 us,
// 2 000 rows 29.9 -> 17.6.
template <bool FEW, int STEP, typename TI, typename TO>
__device__ inline void linear_heads_tile(const TI* __restrict__ x, int ldx, const bf16_t* __restrict__ w, TO* __restrict__ out,
                                         int ldo, int rows, int N, int K, int ohs) {
  constexpr int COLS = FEW ? 1 : 4, RUN = STEP / 4;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int h = blockIdx.z, r0 = blockIdx.x * 64 + (FEW ? 0 : 16 * wave), n0 = blockIdx.y * 64 + (FEW ? 16 * wave : 0);
  if (r0 >= rows || n0 >= N) return;
  const TI* xa = x + (long long)min(r0 + c, rows - 1) * ldx + (long long)h * K + RUN * g;
  const bf16_t* wb[COLS];
#pragma unroll
  for (int j = 0; j < COLS; ++j) wb[j] = w + ((long long)h * N + min(n0 + 16 * j + c, N - 1)) * K + RUN * g;
  f32x4_t acc[COLS];
#pragma unroll
  for (int j = 0; j < COLS; ++j) acc[j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int ks = 0; ks < K; ks += STEP) {
    const auto a = run_of_k<STEP>(xa + ks);
#pragma unroll
    for (int j = 0; j < COLS; ++j) {
      const auto b = run_of_k<STEP>(wb[j] + ks);
      if constexpr (STEP == 32) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[j], 0, 0, 0);
      else acc[j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int j = 0; j < COLS; ++j) {
    const int n = n0 + 16 * j + c;
    if (n >= N) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = r0 + 4 * g + e;
      if (r < rows) out[(long long)r * ldo + (long long)h * ohs + n] = from_f32<TO>(acc[j][e]);
    }
  }
}

template <bool FEW, int STEP, typename TO>
__global__ __launch_bounds__(256) void linear_heads_kernel(const bf16_t* __restrict__ x, int ldx,
                                                           const bf16_t* __restrict__ w, TO* __restrict__ out, int ldo,
                                                           int rows, int N, int K, int ohs) {
  linear_heads_tile<FEW, STEP, bf16_t, TO>(x, ldx, w, out, ldo, rows, N, K, ohs);
}

// ---- a latent layer's rows in two launches: what its first product leaves, and what its second does ----------------------
// Single tokens pay a launch's three to four microseconds for every step between two products: the two norms, the two
// rotations, the store into the cache and the fold of the key's lift into the query were six launches and two products (31 us of
// a layer at 8 rows of width 2 048, of which the arithmetic is a few), and are two around one product (12).
struct Turn {  // cos and sin of a row's angles [rows][dims / 2][2], before `mag`
  const float* cs;
  int dims, interleaved;
  float mag;
};

// Entry i of a rotated vector v (dims of its entries turn, the rest pass).
__device__ inline float turned_at(const float* v, int i, const Turn& t, const float* cs) {
  if (i >= t.dims) return v[i];
  const int half = t.dims >> 1;
  int j, mate;
  bool first;
  if (t.interleaved) j = i >> 1, first = !(i & 1), mate = i ^ 1;
  else first = i < half, j = first ? i : i - half, mate = first ? i + half : i - half;
  const float c = cs[2 * j] * t.mag, s = cs[2 * j + 1] * t.mag;
  return first ? v[i] * c - v[mate] * s : v[i] * c + v[mate] * s;
}

struct LatentRows {
  int lds, q_rank, kv_rank, rot_dim, ldcq;
  float eps;
  const float *wq, *wkv;
  Turn turn;
  const int *row_pos, *row_seq, *seq_slot, *block_table;
  int bt_stride, BS;
};
constexpr int LATENT_PER = 8;  // entries of a normed run that a thread holds

// src [rows, q_rank (+ kv_rank + rot_dim)].  Workgroup (r, 0): cq = the RMS norm of the row's first q_rank entries.  (r, 1): the
// norm of the next kv_rank, and the rest rotated, as the row's key in the cache (K [block][BS][kv_rank + rot_dim]); the
// former also as its value (V [block][kv_rank][BS]).
template <typename T>
__global__ __launch_bounds__(256) void latent_rows_kernel(const float* __restrict__ src, T* __restrict__ cq, T* __restrict__ kcache,
                                                          T* __restrict__ vcache, LatentRows a) {
  __shared__ float red[16];
  const int r = blockIdx.x;
  const bool own = blockIdx.y == 1;
  const int n = own ? a.kv_rank : a.q_rank;
  const float* s = src + (long long)r * a.lds + (own ? a.q_rank : 0);
  const float* w = own ? a.wkv : a.wq;
  float v[LATENT_PER], gain[LATENT_PER], acc = 0.f;
#pragma unroll
  for (int i = 0; i < LATENT_PER; ++i) {
    const int e = threadIdx.x + 256 * i;
    v[i] = e < n ? s[e] : 0.f, gain[i] = e < n ? w[e] : 0.f;
    acc = fmaf(v[i], v[i], acc);
  }
  T *k = nullptr, *val = nullptr;
  if (own) {
    const int p = a.row_pos[r], kd = a.kv_rank + a.rot_dim, off = p % a.BS;
    const long long blk = a.block_table[(long long)a.seq_slot[a.row_seq[r]] * a.bt_stride + p / a.BS];
    k = kcache + (blk * a.BS + off) * kd, val = vcache + blk * a.kv_rank * a.BS + off;
    const float* cs = a.turn.cs + (long long)r * a.turn.dims;
    for (int i = threadIdx.x; i < a.rot_dim; i += 256) k[a.kv_rank + i] = from_f32<T>(turned_at(s + n, i, a.turn, cs));
  }
  const float inv = 1.f / sqrtf(block_sum(acc, red) / (float)n + a.eps);
#pragma unroll
  for (int i = 0; i < LATENT_PER; ++i) {
    const int e = threadIdx.x + 256 * i;
    if (e >= n) continue;
    const T o = from_f32<T>(v[i] * inv * gain[i]);
    if (own) k[e] = o, val[(long long)e * a.BS] = o;
    else cq[(long long)r * a.ldcq + e] = o;
  }
}

// x [rows, heads K + heads rot_dim] (32-bit: every head's unrotated entries, then every head's rotated ones): out's head h gets
// w[h] (N x K) times its unrotated entries, rounded to bfloat16, and behind them its rotated ones.  The last of gridDim.y
// workgroups rotates.
template <bool FEW, int STEP>
__global__ __launch_bounds__(256) void latent_query_kernel(const float* __restrict__ x, int ldx, const bf16_t* __restrict__ w,
                                                           bf16_t* __restrict__ out, int ldo, int rows, int N, int K, int rot_dim,
                                                           Turn turn) {
  if (blockIdx.y + 1 < gridDim.y) {
    linear_heads_tile<FEW, STEP, float, bf16_t>(x, ldx, w, out, ldo, rows, N, K, N + rot_dim);
    return;
  }
  const int h = blockIdx.z, heads = gridDim.z, lane = threadIdx.x & 63;
  for (int r = blockIdx.x * 64 + (threadIdx.x >> 6); r < min(rows, (int)blockIdx.x * 64 + 64); r += 4) {  // a wavefront a row
    const float *v = x + (long long)r * ldx + heads * K + h * rot_dim, *cs = turn.cs + (long long)r * turn.dims;
    bf16_t* o = out + (long long)r * ldo + h * (N + rot_dim) + N;
    for (int i = lane; i < rot_dim; i += 64) o[i] = f32_to_bf16(turned_at(v, i, turn, cs));
  }
}

}  // namespace

extern "C" int lq_rmsnorm_cols(const float* src, int lds_, const float* w, float eps, void* out, int out_dtype, int ldo,
                               int rows, int n, hipStream_t stream) {
  LQ_REQUIRE(rows > 0 && n > 0 && lds_ >= n && ldo >= n, "rmsnorm_cols: rows %d, columns %d, strides %d and %d", rows, n, lds_, ldo);
  LQ_REQUIRE(src && w && out, "rmsnorm_cols: null pointer");
  if (out_dtype == LQ_F32) rmsnorm_cols_kernel<float><<<rows, 256, 0, stream>>>(src, lds_, w, eps, (float*)out, ldo, n);
  else if (out_dtype == LQ_BF16) rmsnorm_cols_kernel<bf16_t><<<rows, 256, 0, stream>>>(src, lds_, w, eps, (bf16_t*)out, ldo, n);
  else LQ_REQUIRE(false, "rmsnorm_cols: unknown dtype %d", out_dtype);
  LQ_CHECK_LAUNCH("rmsnorm_cols");
  return 0;
}

extern "C" int lq_rotary(const float* src, int lds_, void* out, int out_dtype, int ldo, int rows, int heads, int size,
                         int out_head_stride, int dims, int interleaved, const double* freqs, float magnitude,
                         const int* row_pos, hipStream_t stream) {
  LQ_REQUIRE(rows > 0 && heads > 0 && size > 0, "rotary: rows %d, heads %d, size %d", rows, heads, size);
  LQ_REQUIRE(dims >= 2 && dims % 2 == 0 && dims <= size && dims <= 8192, "rotary: %d rotated entries of %d", dims, size);
  LQ_REQUIRE(out_head_stride >= size && lds_ >= heads * size && ldo >= (heads - 1) * out_head_stride + size,
             "rotary: a stride is smaller than what it steps over");
  LQ_REQUIRE(src && out && freqs && row_pos, "rotary: null pointer");
  const size_t lds_bytes = (size_t)dims * sizeof(float);
  if (out_dtype == LQ_F32)
    rotary_kernel<float><<<rows, 128, lds_bytes, stream>>>(src, lds_, (float*)out, ldo, heads, size, out_head_stride, dims,
                                                           interleaved, freqs, magnitude, row_pos);
  else if (out_dtype == LQ_BF16)
    rotary_kernel<bf16_t><<<rows, 128, lds_bytes, stream>>>(src, lds_, (bf16_t*)out, ldo, heads, size, out_head_stride, dims,
                                                            interleaved, freqs, magnitude, row_pos);
  else LQ_REQUIRE(false, "rotary: unknown dtype %d", out_dtype);
  LQ_CHECK_LAUNCH("rotary");
  return 0;
}

// src [rows, (heads + kv_heads) * key_dim + kv_heads * value_dim] float32 (stride lds_): queries, keys, values.
// dims = 0: no rotation (freqs may be null); norm_eps < 0: no norm.
extern "C" int lq_rotary_qkv(const float* src, int lds_, void* q_out, int ldq, void* k_out, int ldk, void* v_out, int ldv,
                             int out_dtype, int rows, int heads, int kv_heads, int key_dim, int value_dim, int dims,
                             int interleaved, const double* freqs, float magnitude, float norm_eps, const int* row_pos,
                             int value_width, hipStream_t stream) {
  // `value_width` > 0: so many value entries a row pass, in the place of kv_heads * value_dim (key heads that share
  // a value head)
  const int VW = value_width > 0 ? value_width : kv_heads * value_dim;
  LQ_REQUIRE(rows > 0 && heads > 0 && kv_heads > 0 && key_dim > 0 && value_dim > 0, "rotary_qkv: rows %d, heads %d and %d, sizes %d and %d",
             rows, heads, kv_heads, key_dim, value_dim);
  LQ_REQUIRE(dims >= 0 && dims % 2 == 0 && dims <= key_dim && dims <= 8192, "rotary_qkv: %d rotated entries of %d", dims, key_dim);
  LQ_REQUIRE(lds_ >= (heads + kv_heads) * key_dim + VW && ldq >= heads * key_dim && ldk >= kv_heads * key_dim &&
                 ldv >= VW, "rotary_qkv: a row stride is smaller than its row");
  LQ_REQUIRE(src && q_out && k_out && v_out && row_pos && (dims == 0 || freqs), "rotary_qkv: null pointer");
  const size_t lds_bytes = (size_t)dims * sizeof(float);
  // few rows (single tokens): a wavefront a head, so that no wavefront walks through its heads one after the other
  const int share = rows >= 512 ? 1 : (lq_ceil_div(heads + kv_heads, 4) < 64 ? lq_ceil_div(heads + kv_heads, 4) : 64);
  const dim3 grid(rows, share);
  if (out_dtype == LQ_F32)
    rotary_qkv_kernel<float><<<grid, 256, lds_bytes, stream>>>(src, lds_, (float*)q_out, ldq, (float*)k_out, ldk, (float*)v_out,
                                                               ldv, heads, kv_heads, key_dim, VW, dims, interleaved,
                                                               freqs, magnitude, norm_eps, row_pos);
  else if (out_dtype == LQ_BF16)
    rotary_qkv_kernel<bf16_t><<<grid, 256, lds_bytes, stream>>>(src, lds_, (bf16_t*)q_out, ldq, (bf16_t*)k_out, ldk,
                                                                (bf16_t*)v_out, ldv, heads, kv_heads, key_dim, VW, dims,
                                                                interleaved, freqs, magnitude, norm_eps, row_pos);
  else LQ_REQUIRE(false, "rotary_qkv: unknown dtype %d", out_dtype);
  LQ_CHECK_LAUNCH("rotary_qkv");
  return 0;
}

// bias: null or a number for every column of src; wq, wk: weights of unit_q and unit_k entries, or null (a rotation is one of
// every unit: of a head, or of an equal part of one) (with
// `norm_qk` off: no norm of q and k); kcache and vcache null: q alone.
extern "C" int lq_qkv_norm_store(const float* src, int lds_, const float* bias, const float* wq, const float* wk, int unit_q,
                                 int unit_k, int norm_qk, int norm_v, int v_from_k, float eps, void* q_out, int ldq, int dtype,
                                 int rows, int heads, int kv_heads, int key_dim, int value_dim, const int* row_pos,
                                 const int* row_seq, const int* seq_slot, const int* block_table, int bt_stride, void* kcache,
                                 void* vcache, int block_size, const float* cos_sin, int dims, int interleaved,
                                 float magnitude, hipStream_t stream) {
  LQ_REQUIRE(cos_sin == nullptr || (dims >= 2 && dims % 2 == 0 && dims <= unit_q && unit_q == unit_k && unit_q > 0 && key_dim % unit_q == 0),
             "qkv_norm_store: %d rotated entries in units of %d and %d for heads of %d", dims, unit_q, unit_k, key_dim);
  LQ_REQUIRE(rows > 0 && rows <= 0x7fffffff && heads > 0 && kv_heads > 0 && key_dim > 0 && value_dim > 0,
             "qkv_norm_store: rows %d, heads %d and %d, sizes %d and %d", rows, heads, kv_heads, key_dim, value_dim);
  LQ_REQUIRE(!v_from_k || key_dim == value_dim, "qkv_norm_store: values that are the keys have their size (%d, %d)", key_dim, value_dim);
  const int QW = heads * key_dim, KW = kv_heads * key_dim, VW = kv_heads * value_dim;
  LQ_REQUIRE(unit_q > 0 && unit_k > 0 && QW % unit_q == 0 && KW % unit_k == 0, "qkv_norm_store: units of %d and %d entries", unit_q, unit_k);
  LQ_REQUIRE(lds_ >= QW + KW + (v_from_k ? 0 : VW) && ldq >= QW, "qkv_norm_store: a row stride is smaller than its row");
  LQ_REQUIRE(src && q_out && (kcache == nullptr) == (vcache == nullptr), "qkv_norm_store: null pointer");
  LQ_REQUIRE(kcache == nullptr || (row_pos && row_seq && seq_slot && block_table && block_size > 0 && bt_stride > 0),
             "qkv_norm_store: the cache needs the rows' places");
  LQ_REQUIRE(norm_qk || (wq == nullptr && wk == nullptr), "qkv_norm_store: weights without a norm");
  // (values go head by head where queries and keys do; they are only copied there)
  const int unit_v = norm_v || (key_dim % unit_q == 0 && key_dim % unit_k == 0) ? value_dim : VW;
  QkvUnits a = {lds_, ldq, heads, kv_heads, key_dim, value_dim, unit_q, unit_k, norm_qk, norm_v, v_from_k,
                eps, bias, wq, wk, row_pos, row_seq, seq_slot, block_table, bt_stride, block_size,
                unit_v, cos_sin, cos_sin != nullptr ? dims : 0, interleaved, magnitude};
  const int units = QW / unit_q + (kcache ? KW / unit_k + VW / unit_v : 0);
  const bool wide = unit_q > 512 || unit_k > 512 || (kcache && unit_v > 512);
  const int gy = wide ? units : lq_ceil_div(units, 4);
  LQ_REQUIRE(gy <= 65535, "qkv_norm_store: too many heads");
  const dim3 grid(rows, gy);
  // what fits the kernel that keeps a unit in registers: everything in fours on whole vectors (the choice follows from
  // the model's sizes and the buffers' alignment, which are the same in every step)
  const int el = dtype == LQ_F32 ? 4 : 2;
  int most = unit_q > unit_k ? unit_q : unit_k;
  if (kcache != nullptr && unit_v > most) most = unit_v;
  const bool fours = key_dim % 4 == 0 && unit_q % 4 == 0 && unit_k % 4 == 0 && value_dim % 4 == 0 && lds_ % 4 == 0 && ldq % 4 == 0 && (uintptr_t)src % 16 == 0 &&
                     (uintptr_t)bias % 16 == 0 && (uintptr_t)wq % 16 == 0 && (uintptr_t)wk % 16 == 0 &&
                     (uintptr_t)q_out % (4 * el) == 0 && (uintptr_t)kcache % (4 * el) == 0 && most <= 16384;
  // many rows of units of 64, 128 or 256, values of a unit's size or twice it: the kernel that takes runs of rows.  It gains where rows
  // are wide: a workgroup has lanes for 1 024 entries of the values, which few heads leave idle.  Microseconds by units and by runs, one
  // sequence (and a row a sequence): 32 query heads of 64 over 8, 640 rows 17.4 / 10.9 (21.9 / 14.2); 64 of 128 over 8, 640 rows 29.3 / 19.7 (32.2 / 22.9);
  // 16 of 128 over 4, 640 rows 11.1 / 11.0 (13.0 / 14.3), 900 14.5 / 13.4 (17.5 / 16.9), 2 000 26.2 / 16.0, 4 096 48.8 / 31.1; 16 of 256 over 4, 640 rows 15.5 /
  // 16.3 (18.9 / 20.2), 900 20.5 / 19.9 (25.0 / 24.5); 8 of 256 over 2, 640 rows 9.3 / 11.0 (10.8 / 14.5), 1 300 15.8 / 17.0; 4 of 256 over 1, 640 rows 6.7 / 9.3,
  // 4 096 21.5 / 23.7
  const int least = unit_q == 64 || (unit_q == 128 && kv_heads >= 8) ? 640 : unit_q == 128 || kv_heads >= 4 ? 1024 : 2048;
  const bool runs = fours && rows >= least && (unit_q != 256 || kv_heads >= 2) && unit_q == unit_k && key_dim % unit_q == 0 &&
                    (kcache == nullptr || (unit_v == value_dim && (value_dim == unit_q || value_dim == 2 * unit_q))) &&
                    (unit_q == 64 || unit_q == 128 || (unit_q == 256 && (kcache == nullptr || value_dim == 256))) && block_size % RUN == 0 &&
                    (uintptr_t)vcache % 16 == 0 && (long long)rows * (heads + kv_heads) * (key_dim / unit_q) < (1ll << 30);
  if (runs) {
    const int in_block = 1024 / unit_q, qk = (heads + (kcache != nullptr ? kv_heads : 0)) * (key_dim / unit_q);
    const int qk_blocks = lq_ceil_div(rows, QKV_ROWS) * lq_ceil_div(qk, in_block);
    const bool twice = kcache != nullptr && value_dim != unit_q;
    const int blocks = qk_blocks + (kcache != nullptr ? rows * lq_ceil_div(kv_heads, 1024 / value_dim) : 0);
#define LQ_QKV_ROWS(T)                                                                                                     \
  (twice ? unit_q == 64 ? qkv_norm_store_rows_kernel<T, 16, 32> : qkv_norm_store_rows_kernel<T, 32, 64>                   \
   : unit_q == 64 ? qkv_norm_store_rows_kernel<T, 16, 16>                                                                 \
   : unit_q == 128 ? qkv_norm_store_rows_kernel<T, 32, 32> : qkv_norm_store_rows_kernel<T, 64, 64>)                       \
      <<<blocks, 256, 0, stream>>>(src, (T*)q_out, (T*)kcache, (T*)vcache, a, rows, qk_blocks)
    if (dtype == LQ_F32) LQ_QKV_ROWS(float);
    else if (dtype == LQ_BF16) LQ_QKV_ROWS(bf16_t);
    else LQ_REQUIRE(false, "qkv_norm_store: unknown dtype %d", dtype);
#undef LQ_QKV_ROWS
    LQ_CHECK_LAUNCH("qkv_norm_store(rows)");
    return 0;
  }
#define LQ_QKV4(T, WIDE, PER)                                                                                        \
  qkv_norm_store4_kernel<T, WIDE, PER><<<grid, 256, 0, stream>>>(src, (T*)q_out, (T*)kcache, (T*)vcache, a)
#define LQ_QKV(T)                                                                                                    \
  do {                                                                                                               \
    if (fours && !wide && most <= 256) LQ_QKV4(T, false, 1);                                                         \
    else if (fours && !wide) LQ_QKV4(T, false, 2);                                                                   \
    else if (fours && most <= 4096) LQ_QKV4(T, true, 4);                                                             \
    else if (fours) LQ_QKV4(T, true, 16);                                                                            \
    else                                                                                                             \
    if (wide) qkv_norm_store_kernel<T, true><<<grid, 256, 0, stream>>>(src, (T*)q_out, (T*)kcache, (T*)vcache, a);   \
    else qkv_norm_store_kernel<T, false><<<grid, 256, 0, stream>>>(src, (T*)q_out, (T*)kcache, (T*)vcache, a);       \
  } while (0)
  if (dtype == LQ_F32) LQ_QKV(float);
  else if (dtype == LQ_BF16) LQ_QKV(bf16_t);
  else LQ_REQUIRE(false, "qkv_norm_store: unknown dtype %d", dtype);
#undef LQ_QKV
#undef LQ_QKV4
  LQ_CHECK_LAUNCH("qkv_norm_store");
  return 0;
}

// Whether lq_linear_heads takes these operands (else the caller runs a product a head).
extern "C" int lq_linear_heads_accepts(const void* x, const void* w, int in_dtype, int K, int ldx) {
  return in_dtype == LQ_BF16 && K % 16 == 0 && ldx % 4 == 0 && ((uintptr_t)x % 8) == 0 && ((uintptr_t)w % 8) == 0;
}

// x [rows, heads * K] (stride ldx), w [heads, N, K] dense, out: head h's N columns from column h * out_head_stride
extern "C" int lq_linear_heads(const void* x, int ldx, const void* w, void* out, int in_dtype, int out_dtype, int ldo,
                               int rows, int heads, int N, int K, int out_head_stride, hipStream_t stream) {
  LQ_REQUIRE(rows > 0 && heads > 0 && heads <= 65535 && N > 0 && K > 0, "linear_heads: rows %d, heads %d, N %d, K %d", rows,
             heads, N, K);
  LQ_REQUIRE(ldx >= heads * K && out_head_stride >= N && ldo >= (heads - 1) * out_head_stride + N,
             "linear_heads: a stride is smaller than what it steps over");
  LQ_REQUIRE(x && w && out, "linear_heads: null pointer");
  LQ_REQUIRE(lq_linear_heads_accepts(x, w, in_dtype, K, ldx), "linear_heads: bfloat16 operands, K in 16s, rows on 8 bytes");
  LQ_REQUIRE(lq_ceil_div(N, 64) <= 65535, "linear_heads: too many columns");
  dim3 grid(lq_ceil_div(rows, 64), lq_ceil_div(N, 64), heads);
  const bool wide = K % 32 == 0 && ldx % 8 == 0 && ((uintptr_t)x | (uintptr_t)w) % 16 == 0, few = rows <= 16;
#define LQ_HEADS(FEW, STEP, T)                                                                                                        \
  linear_heads_kernel<FEW, STEP, T><<<grid, 256, 0, stream>>>((const bf16_t*)x, ldx, (const bf16_t*)w, (T*)out, ldo, rows, N, K, \
                                                              out_head_stride)
#define LQ_HEADS_T(T) (wide ? (few ? LQ_HEADS(true, 32, T) : LQ_HEADS(false, 32, T)) : (few ? LQ_HEADS(true, 16, T) : LQ_HEADS(false, 16, T)))
  if (out_dtype == LQ_F32) LQ_HEADS_T(float);
  else if (out_dtype == LQ_BF16) LQ_HEADS_T(bf16_t);
  else LQ_REQUIRE(false, "linear_heads: unknown dtype %d", out_dtype);
#undef LQ_HEADS_T
#undef LQ_HEADS
  LQ_CHECK_LAUNCH("linear_heads");
  return 0;
}

// Whether lq_latent_rows and lq_latent_query take a latent layer's sizes (in a bfloat16 run).
extern "C" int lq_latent_accepts(int dtype, int heads, int dim, int rot_dim, int kv_rank, int q_rank) {
  return dtype == LQ_BF16 && heads >= 1 && heads <= 65535 && dim >= 16 && dim % 16 == 0 && rot_dim >= 2 && rot_dim <= 1024 &&
         kv_rank >= 1 && kv_rank <= 256 * LATENT_PER && q_rank >= 1 && q_rank <= 256 * LATENT_PER &&
         (long long)heads * (dim + rot_dim) <= 0x3fffffff && (long long)heads * (kv_rank + rot_dim) <= 0x3fffffff;
}

// src float32 [rows, q_rank (+ kv_rank + rot_dim)], cos_sin float32 [rows, dims / 2, 2]; kcache null: no key or value of its own.
extern "C" int lq_latent_rows(const float* src, int lds_, int rows, int q_rank, int kv_rank, int rot_dim, const float* wq, const float* wkv,
                              float eps, const float* cos_sin, int dims, int interleaved, float magnitude, void* cq, int ldcq,
                              const int* row_pos, const int* row_seq, const int* seq_slot, const int* block_table, int bt_stride,
                              void* kcache, void* vcache, int block_size, hipStream_t stream) {
  const bool own = kcache != nullptr;
  LQ_REQUIRE(rows > 0 && lq_latent_accepts(LQ_BF16, 1, 16, rot_dim, kv_rank, q_rank), "latent_rows: rows %d, ranks %d and %d, %d rotated", rows,
             q_rank, kv_rank, rot_dim);
  LQ_REQUIRE(lds_ >= q_rank + (own ? kv_rank + rot_dim : 0) && ldcq >= q_rank, "latent_rows: a row stride is smaller than its row");
  LQ_REQUIRE(src && wq && cq && own == (vcache != nullptr), "latent_rows: null pointer");
  LQ_REQUIRE(!own || (wkv && cos_sin && dims >= 2 && dims % 2 == 0 && dims <= rot_dim && row_pos && row_seq && seq_slot && block_table &&
                      block_size > 0 && bt_stride > 0), "latent_rows: the cache needs the rows' places and angles");
  const LatentRows a = {lds_, q_rank, kv_rank, rot_dim, ldcq, eps, wq, wkv, {cos_sin, dims, interleaved, magnitude},
                        row_pos, row_seq, seq_slot, block_table, bt_stride, block_size};
  latent_rows_kernel<bf16_t><<<dim3(rows, own ? 2 : 1), 256, 0, stream>>>(src, (bf16_t*)cq, (bf16_t*)kcache, (bf16_t*)vcache, a);
  LQ_CHECK_LAUNCH("latent_rows");
  return 0;
}

// x float32 [rows, heads * dim + heads * rot_dim], w bfloat16 [heads, kv_rank, dim] dense, out bfloat16 [rows, heads * (kv_rank + rot_dim)]
extern "C" int lq_latent_query(const float* x, int ldx, const void* w, void* out, int ldo, int rows, int heads, int dim, int rot_dim,
                               int kv_rank, const float* cos_sin, int dims, int interleaved, float magnitude, hipStream_t stream) {
  LQ_REQUIRE(rows > 0 && lq_latent_accepts(LQ_BF16, heads, dim, rot_dim, kv_rank, 1), "latent_query: rows %d, %d heads of %d and %d, rank %d", rows,
             heads, dim, rot_dim, kv_rank);
  LQ_REQUIRE(ldx >= heads * (dim + rot_dim) && ldo >= heads * (kv_rank + rot_dim), "latent_query: a row stride is smaller than its row");
  LQ_REQUIRE(x && w && out && cos_sin && dims >= 2 && dims % 2 == 0 && dims <= rot_dim, "latent_query: null pointer, or %d rotated of %d", dims, rot_dim);
  LQ_REQUIRE(ldx % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 8 == 0, "latent_query: operands are not aligned");
  const dim3 grid(lq_ceil_div(rows, 64), lq_ceil_div(kv_rank, 64) + 1, heads);
  const bool wide = dim % 32 == 0 && (uintptr_t)w % 16 == 0;
  const auto kernel = rows <= 16 ? (wide ? latent_query_kernel<true, 32> : latent_query_kernel<true, 16>)
                                 : (wide ? latent_query_kernel<false, 32> : latent_query_kernel<false, 16>);
  kernel<<<grid, 256, 0, stream>>>(x, ldx, (const bf16_t*)w, (bf16_t*)out, ldo, rows, kv_rank, dim, rot_dim,
                                   Turn{cos_sin, dims, interleaved, magnitude});
  LQ_CHECK_LAUNCH("latent_query");
  return 0;
}
