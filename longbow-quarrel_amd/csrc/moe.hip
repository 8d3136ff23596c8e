// Kernels of a mixture of experts whose experts' matrices lie side by side: the router's choice and the experts'
// activation.  Router scores and weights are 32-bit.
#include "device_math.h"

namespace {

// One thread a row: s = sigmoid(z), the `top` largest win (the lower index on a tie); route[r, e] = the expert's
// weight (its score, or its share of the chosen scores), -1 for an expert that was not chosen.
// With `correction` the experts are chosen by s + correction[e]; the weights stay the scores s.  With `groups` > 1
// the experts form that many equal groups of neighbours; a group's mark is the sum of its two largest choice scores
// (of its one, in groups of one), and only experts of the `keep` groups with the largest marks (the lower index on a
// tie) can be chosen.  `softmax`: s = softmax(z) over all E outputs in the sigmoid's place.  `mark_max`: a group's mark
// is its largest choice score alone.  `renorm_eps` is added to the chosen scores' sum before the division.  The last
// `n_ident` of the E outputs are experts without tensors: their weights go to `ident` [rows, n_ident] (-1: not
// chosen) and `route` has the E - n_ident others.
__global__ __launch_bounds__(64) void moe_route_kernel(const float* __restrict__ z, int ldz, float* __restrict__ route,
                                                       int rows, int E, int top, int renorm,
                                                       const float* __restrict__ correction, int groups, int keep,
                                                       int softmax, int mark_max, float renorm_eps,
                                                       float* __restrict__ ident, int n_ident) {
  const int r = blockIdx.x * 64 + threadIdx.x;
  if (r >= rows) return;
  const float* zr = z + (long long)r * ldz;
  const int R = E - n_ident;  // experts with tensors
  float* out_real = route + (long long)r * R;
  float* out_ident = n_ident > 0 ? ident + (long long)r * n_ident : nullptr;
  auto out = [&](int e) -> float& { return e < R ? out_real[e] : out_ident[e - R]; };
  for (int e = 0; e < E; ++e) out(e) = -1.f;
  float zmax = -INFINITY, inv_sum = 1.f;
  if (softmax) {
    for (int e = 0; e < E; ++e) zmax = fmaxf(zmax, zr[e]);
    float sum = 0.f;
    for (int e = 0; e < E; ++e) sum += expf(zr[e] - zmax);
    inv_sum = 1.f / sum;
  }
  auto score = [&](int e) { return softmax ? expf(zr[e] - zmax) * inv_sum : 1.f / (1.f + expf(-zr[e])); };
  auto choice = [&](int e) { return correction != nullptr ? score(e) + correction[e] : score(e); };
  unsigned long long kept = ~0ull;  // bit g: group g may be chosen from
  const int per = groups > 1 ? E / groups : E;
  if (groups > 1 && keep < groups) {
    kept = 0ull;
    for (int n = 0; n < keep; ++n) {
      int best = -1;
      float bm = 0.f;
      for (int g = 0; g < groups; ++g) {
        if ((kept >> g) & 1ull) continue;
        float a = -INFINITY, b = -INFINITY;  // the group's two largest choice scores
        for (int e = g * per; e < (g + 1) * per; ++e) {
          const float v = choice(e);
          if (v > a) b = a, a = v;
          else if (v > b) b = v;
        }
        const float mark = per > 1 && !mark_max ? a + b : a;
        if (best < 0 || mark > bm) best = g, bm = mark;
      }
      if (best < 0) break;
      kept |= 1ull << best;
    }
  }
  float total = 0.f;
  for (int k = 0; k < top; ++k) {
    int best = -1;
    float bz = 0.f;
    for (int e = 0; e < E; ++e) {
      if (out(e) >= 0.f) continue;  // chosen already
      if (groups > 1 && !((kept >> (e / per)) & 1ull)) continue;
      const float v = choice(e);  // scores are compared, not logits: equal scores are a tie
      if (best < 0 || v > bz) best = e, bz = v;
    }
    if (best < 0) break;
    const float w = score(best);
    out(best) = w == w ? w : 0.f;
    total += out(best);
  }
  total += renorm_eps;
  if (renorm && total > 0.f)
    for (int e = 0; e < E; ++e)
      if (out(e) >= 0.f) out(e) /= total;
}

constexpr int ROUTE_PER = 16;  // outputs a lane at most in the kernels below

// The same choice with a wavefront a row, for up to 64 PER experts: lane l has the outputs l, l + 64, ...  A thread a row
// reads its logits one behind the other and works out every score again in each of its `top` searches: at 8 rows a chain
// of latencies on one wavefront, whatever the rest of the chip does.  Here the scores are made once, a search is a maximum
// over the lanes, and a group's mark is one lane's search in LDS.  Sums are added up in the order of the kernel above, so
// the weights are the same to the bit.
// A thread a row -> a wavefront a row, the same bits: 8 rows, 2 of 8 experts 8.1 -> 2.9 us; 8 rows, 4 of 16 in groups
// with a softmax 29 -> 5.6; 8 rows, 8 of 64 in groups 220 -> 7.1; 2635 rows of 16 35.7 -> 6.3; 17 rows of 1024 1414 -> 45.
struct RouteArgs {
  float* route;
  int E, top, renorm;
  const float* correction;
  int groups, keep, softmax, mark_max;
  float renorm_eps;
  float* ident;
  int n_ident;
};

// Row r, whose logits are z[0 .. E), by one wavefront; `mine`: E floats of LDS for the choice scores, where groups are marked.
template <int PER>
__device__ inline void route_row(const float* z, float* mine, int r, const RouteArgs& a) {
  const int lane = threadIdx.x & 63, E = a.E, top = a.top, renorm = a.renorm, groups = a.groups, keep = a.keep, n_ident = a.n_ident;
  const int softmax = a.softmax, mark_max = a.mark_max;
  const float renorm_eps = a.renorm_eps;
  const float* correction = a.correction;
  float *route = a.route, *ident = a.ident;
  float s[PER], v[PER];   // scores; what the choice goes by
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int e = lane + 64 * j;
    s[j] = e < E ? z[e] : -INFINITY;
  }
  if (softmax) {
    float zmax = -INFINITY, sum = 0.f;
#pragma unroll
    for (int j = 0; j < PER; ++j) zmax = fmaxf(zmax, s[j]);
    zmax = wave_max(zmax);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      s[j] = expf(s[j] - zmax);
      const int n = E - 64 * j < 64 ? E - 64 * j : 64;
      for (int i = 0; i < n; ++i) sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s[j]), i));
    }
    const float inv_sum = 1.f / sum;
#pragma unroll
    for (int j = 0; j < PER; ++j) s[j] *= inv_sum;
  } else {
#pragma unroll
    for (int j = 0; j < PER; ++j) s[j] = 1.f / (1.f + expf(-s[j]));
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int e = lane + 64 * j;
    v[j] = correction != nullptr && e < E ? s[j] + correction[e] : s[j];
  }
  // Of the lanes' values the largest, the lowest index among equals; a value that is no number counts only where it is
  // the first of the candidates (which bit j of `from` marks), and then wins.  -> its index, or -1
  auto pick = [&](const float* val, unsigned from, int n) {
    int first = -1;
    float most = -INFINITY;
#pragma unroll
    for (int j = PER - 1; j >= 0; --j) {
      if (j >= n) continue;
      const unsigned long long some = __ballot((from >> j) & 1u);
      if (some != 0ull) first = 64 * j + (int)__builtin_ctzll(some);
      if (((from >> j) & 1u) && val[j] > most) most = val[j];
    }
    if (first < 0) return -1;
    most = wave_max(most);
    int best = first;
    bool odd = false;
#pragma unroll
    for (int j = PER - 1; j >= 0; --j) {
      if (j >= n) continue;
      const unsigned long long same = __ballot(((from >> j) & 1u) && val[j] == most);
      if (same != 0ull) best = 64 * j + (int)__builtin_ctzll(same);
      odd = odd || __ballot(64 * j + lane == first && val[j] != val[j]) != 0ull;
    }
    return odd ? first : best;
  };
  unsigned from = 0;  // bit j: output lane + 64 j may still be chosen
#pragma unroll
  for (int j = 0; j < PER; ++j)
    if (lane + 64 * j < E) from |= 1u << j;
  if (groups > 1 && keep < groups) {
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (lane + 64 * j < E) mine[lane + 64 * j] = v[j];
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
    const int per = E / groups;
    float a = -INFINITY, b = -INFINITY;  // the two largest choice scores of group `lane`
    if (lane < groups)
      for (int i = 0; i < per; ++i) {
        const float x = mine[lane * per + i];
        if (x > a) b = a, a = x;
        else if (x > b) b = x;
      }
    float mark[PER];
    mark[0] = per > 1 && !mark_max ? a + b : a;
    unsigned left = lane < groups ? 1u : 0u;
    unsigned long long kept = 0ull;  // bit g: group g may be chosen from
    for (int n = 0; n < keep; ++n) {
      const int g = pick(mark, left, 1);
      if (g < 0) break;
      kept |= 1ull << g;
      if (lane == g) left = 0u;
    }
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (lane + 64 * j < E && !((kept >> ((lane + 64 * j) / per)) & 1ull)) from &= ~(1u << j);
  }
  float total = 0.f;
  unsigned chosen = 0;
  for (int k = 0; k < top; ++k) {
    const int best = pick(v, from, PER);
    if (best < 0) break;
    float w = 0.f;
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (best / 64 == j) w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s[j]), best % 64));
    total += w == w ? w : 0.f;
    if (lane == best % 64) from &= ~(1u << (best / 64)), chosen |= 1u << (best / 64);
  }
  total += renorm_eps;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int e = lane + 64 * j;
    if (e >= E) continue;
    float w = -1.f;
    if ((chosen >> j) & 1u) {
      w = s[j] == s[j] ? s[j] : 0.f;
      if (renorm && total > 0.f) w /= total;
    }
    const int R = E - n_ident;
    if (e < R) route[(long long)r * R + e] = w;
    else ident[(long long)r * n_ident + e - R] = w;
  }
}

template <int PER>
__global__ __launch_bounds__(256) void moe_route_lanes_kernel(const float* __restrict__ z, int ldz, int rows, RouteArgs a) {
  extern __shared__ float lds[];  // [4][E]
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r < rows) route_row<PER>(z + (long long)r * ldz, lds + (threadIdx.x >> 6) * a.E, r, a);  // (a wavefront shares nothing with the others)
}

// The `top` largest logits win (the lower index on a tie) and the weights are the softmax over these alone.  A wavefront a
// row: lane l has the logits l, l + 64, ...; every round finds the largest that is left.
template <int PER>
__device__ inline void route_row_chosen(const float* z, int r, const RouteArgs& a) {
  const int lane = threadIdx.x & 63, E = a.E, top = a.top;
  float* route = a.route;
  float v[PER], w[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int e = lane + 64 * j;
    v[j] = e < E ? z[e] : -INFINITY;
    if (v[j] != v[j]) v[j] = -INFINITY;
    w[j] = -1.f;
  }
  float first = 0.f, sum = 0.f;
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int at = 0x7fffffff;  // the best's index: among equals, and where nothing is a number, the lowest that is left
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int e = lane + 64 * j;
      if (e < E && w[j] < 0.f && (at == 0x7fffffff || v[j] > best)) best = v[j], at = e;
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float ob = __shfl_xor(best, off, LQ_WAVE);
      const int oa = __shfl_xor(at, off, LQ_WAVE);
      if (oa != 0x7fffffff && (at == 0x7fffffff || ob > best || (ob == best && oa < at))) best = ob, at = oa;
    }
    if (at == 0x7fffffff) break;
    if (k == 0) first = best;
    float share = expf(best - first);
    if (share != share) share = 0.f;
    sum += share;
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (lane + 64 * j == at) w[j] = share;
  }
  const float inv = sum > 0.f ? 1.f / sum : 0.f;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int e = lane + 64 * j;
    if (e < E) route[(long long)r * E + e] = w[j] < 0.f ? -1.f : w[j] * inv;
  }
}

__global__ __launch_bounds__(256) void moe_route_chosen_kernel(const float* __restrict__ z, int ldz, int rows, RouteArgs a) {
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r < rows) route_row_chosen<ROUTE_PER>(z + (long long)r * ldz, r, a);
}

// Few rows: the router's product and the choice in one launch, a workgroup a row.  Wavefront w makes logits w, w + 16, ... of the N
// (products of bfloat16, which are exact, in 32-bit sums), the first one chooses.  What bounds it is a launch's start and one trip for
// the operands, which the two launches that this stands for (a product of one workgroup, then a wavefront a row) both had: replayed
// steps of 8 rows of 2 048 over 8 experts take 2.5 us a layer less.
constexpr int ROUTER_MOST = 64, ROUTER_WAVES = 16;
__global__ __launch_bounds__(ROUTER_WAVES * 64) void moe_router_kernel(const bf16_t* __restrict__ h, int ldh, const bf16_t* __restrict__ w, int ldw,
                                                                       float* __restrict__ z, int ldz, int K, int N, RouteArgs a) {
  __shared__ float logits[ROUTER_MOST], choice[ROUTER_MOST];
  const int r = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bf16_t* x = h + (long long)r * ldh;
  for (int n = wave; n < N; n += ROUTER_WAVES) {
    const bf16_t* y = w + (long long)n * ldw;
    float sum[2] = {0.f, 0.f};
#pragma unroll 4
    for (int k = lane * 8; k < K; k += 512) {
      const uint4 p = *(const uint4*)(x + k), q = *(const uint4*)(y + k);
      const unsigned u[4] = {p.x, p.y, p.z, p.w}, v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sum[0] = fmaf(__uint_as_float(u[i] << 16), __uint_as_float(v[i] << 16), sum[0]);
        sum[1] = fmaf(__uint_as_float(u[i] & 0xffff0000u), __uint_as_float(v[i] & 0xffff0000u), sum[1]);
      }
    }
    const float all = wave_sum(sum[0] + sum[1]);
    if (lane == 0) logits[n] = all, z[(long long)r * ldz + n] = all;
  }
  __syncthreads();
  if (wave > 0) return;
  if (a.softmax == 2) route_row_chosen<1>(logits, r, a);
  else route_row<1>(logits, choice, r, a);
}

// out[r, :] += h[r, :] * (the sum of the row's chosen identity experts' weights); weights [rows, n] (-1: not chosen)
template <typename T>
__global__ __launch_bounds__(256) void moe_identity_kernel(const T* __restrict__ h, int ldh,
                                                           const float* __restrict__ weights, int n,
                                                           float* __restrict__ out, int ldo, int width) {
  const int r = blockIdx.x;
  float w = 0.f;
  for (int i = 0; i < n; ++i) {
    const float v = weights[(long long)r * n + i];
    if (v >= 0.f) w += v;
  }
  if (w == 0.f) return;
  for (int c = threadIdx.x; c < width; c += 256) out[(long long)r * ldo + c] += w * to_f32(h[(long long)r * ldh + c]);
}

// VEC (1 or 4) neighbouring entries
template <typename T, int VEC>
__device__ inline void store_run(T* o, const float (&v)[VEC]) {
  if constexpr (VEC == 4 && sizeof(T) == 2) {
    uint2 packed;
    packed.x = (uint32_t)f32_to_bf16(v[0]).bits | ((uint32_t)f32_to_bf16(v[1]).bits << 16);
    packed.y = (uint32_t)f32_to_bf16(v[2]).bits | ((uint32_t)f32_to_bf16(v[3]).bits << 16);
    *(uint2*)o = packed;
  } else if constexpr (VEC == 4) {
    *(float4*)o = make_float4(v[0], v[1], v[2], v[3]);
  } else {
    *o = from_f32<T>(v[0]);
  }
}

// gu [rows, E, 2, ff] (gate then up of every expert), route [rows, E]; out [rows, E, ff]:
// g = min(w gate, limit), u = clamp(w up, -limit, limit), y = g sigmoid(1.702 g) (u + 1) for a chosen expert (its
// weight w on what it read: `on_input`; otherwise w multiplies y), 0 for the others.  `plain_silu`: the expert is
// y = silu(gate) up without clamps.
template <typename T, int VEC>
__global__ __launch_bounds__(256) void moe_glu_kernel(const float* __restrict__ gu, long long ldg,
                                                      const float* __restrict__ route, T* __restrict__ out,
                                                      long long ldo, int E, int ff, float limit, int on_input,
                                                      int plain_silu) {
  const int r = blockIdx.y;
  const int i = (blockIdx.x * 256 + threadIdx.x) * VEC;  // VEC entries a thread, all of one expert
  if (i >= E * ff) return;
  const int e = i / ff, c = i - e * ff;
  const float w = route[(long long)r * E + e];
  float y[VEC], gate[VEC], up[VEC];
#pragma unroll
  for (int j = 0; j < VEC; ++j) y[j] = 0.f;
  if (w >= 0.f) {
    const float* p = gu + r * ldg + (long long)e * 2 * ff + c;
    if constexpr (VEC == 4) {
      const float4 a = *(const float4*)p, b = *(const float4*)(p + ff);
      gate[0] = a.x, gate[1] = a.y, gate[2] = a.z, gate[3] = a.w, up[0] = b.x, up[1] = b.y, up[2] = b.z, up[3] = b.w;
    } else {
      gate[0] = p[0], up[0] = p[ff];
    }
    const float s = on_input ? w : 1.f;
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      if (plain_silu) {
        const float g = gate[j] * s;
        y[j] = g / (1.f + expf(-g)) * (up[j] * s);
      } else {
        const float g = fminf(gate[j] * s, limit);
        const float u = fminf(fmaxf(up[j] * s, -limit), limit);
        y[j] = g / (1.f + expf(-1.702f * g)) * (u + 1.f);
      }
      if (!on_input) y[j] *= w;
    }
  }
  store_run<T, VEC>(out + r * ldo + i, y);
}

// The same for experts without a gate: u [rows, E ff + shared], out likewise: out = act(u) w for a chosen expert's entries,
// 0 for the others'; the last `shared` columns (an expert that every row uses) pass with weight one.  VEC entries a thread,
// all of one expert.
template <typename T, int VEC>
__global__ __launch_bounds__(256) void moe_act_kernel(const float* __restrict__ u, long long ldu, const float* __restrict__ route,
                                                      T* __restrict__ out, long long ldo, int E, int ff, int shared, int act) {
  const int r = blockIdx.y;
  const int i = (blockIdx.x * 256 + threadIdx.x) * VEC;
  if (i >= E * ff + shared) return;
  const float w = i < E * ff ? route[(long long)r * E + i / ff] : 1.f;
  float v[VEC];
#pragma unroll
  for (int j = 0; j < VEC; ++j) v[j] = 0.f;
  if (w >= 0.f) {
    if constexpr (VEC == 4) {
      const float4 q = *(const float4*)(u + r * ldu + i);
      v[0] = q.x, v[1] = q.y, v[2] = q.z, v[3] = q.w;
    } else {
      v[0] = u[r * ldu + i];
    }
#pragma unroll
    for (int j = 0; j < VEC; ++j) v[j] = activate(v[j], act) * w;
  }
  store_run<T, VEC>(out + r * ldo + i, v);
}

// ---- a step's rows sorted by expert ----------------------------------------------------------------------------------
constexpr int SORT_THREADS = 1024;  // (the walk over the rows is a chain of barriers)
// counts[e] = rows that chose expert e; one workgroup an expert.
__global__ __launch_bounds__(SORT_THREADS) void moe_count_kernel(const float* __restrict__ route, int rows, int E,
                                                        int* __restrict__ counts) {
  __shared__ float red[16];
  const int e = blockIdx.x;
  float n = 0.f;  // (counts of up to 2^24 rows are whole numbers in 32-bit floats)
  for (int r = threadIdx.x; r < rows; r += SORT_THREADS) n += route[(long long)r * E + e] >= 0.f ? 1.f : 0.f;
  n = block_sum(n, red);
  if (threadIdx.x == 0) counts[e] = (int)n;
}

// Expert e's rows, in ascending order, take the places offset(e) .. offset(e) + counts[e] - 1 of the sorted list
// (offset: the counts of the experts before it): order[place] = row, weight[place] = the row's weight for the expert,
// place_of[row, e] = place (-1 for an expert the row did not choose).  One workgroup an expert walks the rows in
// chunks of SORT_THREADS with a running count, so the order does not depend on timing.
__global__ __launch_bounds__(SORT_THREADS) void moe_place_kernel(const float* __restrict__ route, int rows, int E,
                                                        const int* __restrict__ counts, int* __restrict__ order,
                                                        float* __restrict__ weight, int* __restrict__ place_of, int places) {
  __shared__ int wave_n[SORT_THREADS / 64];
  __shared__ int base;
  const int e = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (threadIdx.x == 0) {
    int off = 0;
    for (int i = 0; i < e; ++i) off += counts[i];
    base = off;
  }
  __syncthreads();
  for (int r0 = 0; r0 < rows; r0 += SORT_THREADS) {
    const int r = r0 + threadIdx.x;
    const float w = r < rows ? route[(long long)r * E + e] : -1.f;
    const bool chosen = w >= 0.f;
    const unsigned long long mask = __ballot(chosen);
    const int before = __popcll(mask & ((1ull << lane) - 1ull));
    if (lane == 0) wave_n[wave] = __popcll(mask);
    __syncthreads();
    int at = base + before;
    for (int i = 0; i < wave; ++i) at += wave_n[i];
    if (chosen) order[at] = r, weight[at] = w;
    if (r < rows) place_of[(long long)r * E + e] = chosen ? at : -1;
    __syncthreads();
    if (threadIdx.x == 0) for (int i = 0; i < SORT_THREADS / 64; ++i) base += wave_n[i];
    __syncthreads();
  }
  if (e == E - 1)  // places that nobody takes name a row that there is, with no weight
    for (int at = base + threadIdx.x; at < places; at += SORT_THREADS) order[at] = 0, weight[at] = -1.f;
}

// dst[i, :] = src[order[i], :], rows of `width` units
template <typename U>
__global__ __launch_bounds__(256) void moe_gather_kernel(const U* __restrict__ src, long long ld, const int* __restrict__ order,
                                                         U* __restrict__ dst, int width) {
  const U* s = src + (long long)order[blockIdx.x] * ld;
  U* d = dst + (long long)blockIdx.x * width;
  for (int i = threadIdx.x; i < width; i += 256) d[i] = s[i];
}

// out[r, :] = the sum, over the experts that row r chose in ascending order, of ys[place_of[r, e], :]
template <int VEC>
__global__ __launch_bounds__(256) void moe_scatter_kernel(const float* __restrict__ ys, const int* __restrict__ place_of, int E,
                                                          float* __restrict__ out, int ldo, int width) {
  const int r = blockIdx.x;
  const int* places = place_of + (long long)r * E;
  for (int i = threadIdx.x * VEC; i < width; i += 256 * VEC) {
    float acc[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) acc[j] = 0.f;
    for (int e = 0; e < E; ++e) {
      const int at = places[e];
      if (at < 0) continue;
      const float* y = ys + (long long)at * width + i;
      if constexpr (VEC == 4) {
        const float4 q = *(const float4*)y;
        acc[0] += q.x, acc[1] += q.y, acc[2] += q.z, acc[3] += q.w;
      } else {
        acc[0] += y[0];
      }
    }
    store_run<float, VEC>(out + (long long)r * ldo + i, acc);
  }
}

}  // namespace

// `experts` counts every output of the router, the `n_ident` identity experts at its end included: route is
// [rows, experts - n_ident], ident [rows, n_ident] (null without identity experts).
// what the choice's options must be, whichever launch makes it
static int check_route(int rows, int experts, int top, int ldz, const float* correction, int groups, int keep, int softmax, float renorm_eps,
                       const float* ident, int n_ident) {
  LQ_REQUIRE(groups >= 0 && (groups <= 1 || (groups <= 64 && experts % groups == 0 && keep >= 1 && keep <= groups)),
             "moe_route: %d experts in %d groups of which %d are kept", experts, groups, keep);
  LQ_REQUIRE(rows > 0 && experts > 0 && top >= 1 && top <= experts && ldz >= experts, "moe_route: rows %d, %d of %d experts",
             rows, top, experts);
  LQ_REQUIRE(softmax >= 0 && softmax <= 2 && (softmax != 2 || (correction == nullptr && groups <= 1 && n_ident == 0)),
             "moe_route: a softmax over the chosen logits takes no correction, groups or identity experts");
  LQ_REQUIRE(n_ident >= 0 && n_ident < experts && (n_ident == 0 || ident != nullptr) && renorm_eps >= 0.f,
             "moe_route: %d identity experts of %d", n_ident, experts);
  return 0;
}

extern "C" int lq_moe_route(const float* z, int ldz, float* route, int rows, int experts, int top, int renormalize,
                            const float* correction, int groups, int keep, int softmax, int mark_max, float renorm_eps,
                            float* ident, int n_ident, hipStream_t stream) {
  const int rc = check_route(rows, experts, top, ldz, correction, groups, keep, softmax, renorm_eps, ident, n_ident);
  if (rc != 0) return rc;
  LQ_REQUIRE(z && route, "moe_route: null pointer");
  const RouteArgs a = {route, experts, top, renormalize, correction, groups, keep, softmax, mark_max, renorm_eps, ident, n_ident};
  if (softmax == 2) {
    LQ_REQUIRE(experts <= 64 * ROUTE_PER, "moe_route: %d experts (at most %d)", experts, 64 * ROUTE_PER);
    moe_route_chosen_kernel<<<lq_ceil_div(rows, 4), 256, 0, stream>>>(z, ldz, rows, a);
    LQ_CHECK_LAUNCH("moe_route(softmax over the chosen)");
    return 0;
  }
  // (up to 16 outputs a lane, as above; more would not stay in registers)
  const size_t lds = groups > 1 ? 4 * (size_t)experts * sizeof(float) : 0;
#define LQ_ROUTE(PER) moe_route_lanes_kernel<PER><<<lq_ceil_div(rows, 4), 256, lds, stream>>>(z, ldz, rows, a)
  if (experts <= 64) LQ_ROUTE(1);
  else if (experts <= 256) LQ_ROUTE(4);
  else if (experts <= 64 * ROUTE_PER) LQ_ROUTE(ROUTE_PER);
  else
    moe_route_kernel<<<lq_ceil_div(rows, 64), 64, 0, stream>>>(z, ldz, route, rows, experts, top, renormalize, correction,
                                                               groups, keep, softmax, mark_max, renorm_eps, ident, n_ident);
#undef LQ_ROUTE
  LQ_CHECK_LAUNCH("moe_route");
  return 0;
}

// Whether lq_moe_router takes the router's product [rows, K] x [N, K]^T and the choice together.
extern "C" int lq_moe_router_takes(int dtype, int rows, int K, int N) {
  return dtype == LQ_BF16 && rows >= 1 && rows <= 16 && K >= 8 && K % 8 == 0 && N >= 1 && N <= ROUTER_MOST;
}

// Whether that is faster than the product and the choice in a launch each.  Every row's workgroup reads the whole
// weight, at what one compute unit draws (and for more than 16 outputs in more than one round of its wavefronts); the product reads it
// with all of them, and from 9 rows on takes another kernel that is slower here.  Weights from memory, us, two launches -> one: 1 and 8 rows, 8 outputs of
// 2 048 5.6 -> 4.5 and 6.8 -> 4.8, 16 of 3 072 6.9 -> 5.5 and 7.8 -> 5.9, 32 of 1 536 6.5 -> 6.1 and 7.1 -> 6.6, but 32 of 2 048 7.1 -> 8.5 and 8.1 -> 8.7, 8 of
// 7 168 8.9 -> 10.5 and 10.9 -> 10.2, 64 of 2 048 7.9 -> 14.2; 9 and 16 rows, 16 of 7 168 16.7 -> 11.1 and 19.5 -> 11, 32 of 2 048 9.2 -> 8.6 and 10 -> 8.6, but 32 of
// 4 096 12 -> 12.7, 64 of 1 024 8.7 -> 10.
extern "C" int lq_moe_router_pays(int dtype, int rows, int K, int N) {
  if (!lq_moe_router_takes(dtype, rows, K, N) || N > 32) return 0;
  return (long long)N * K <= (rows <= 8 ? 49152 : N <= 16 ? 114688 : 65536);
}

// z[rows, N] = h . w^T, and lq_moe_route of z's first `experts` columns.
extern "C" int lq_moe_router(const void* h, int ldh, const void* w, int ldw, float* z, int ldz, float* route, int dtype, int rows, int K,
                             int N, int experts, int top, int renormalize, const float* correction, int groups, int keep, int softmax,
                             int mark_max, float renorm_eps, float* ident, int n_ident, hipStream_t stream) {
  LQ_REQUIRE(lq_moe_router_takes(dtype, rows, K, N) && N >= experts && ldz >= N, "moe_router: %d rows of %d, %d outputs are not taken", rows, K, N);
  const int rc = check_route(rows, experts, top, ldz, correction, groups, keep, softmax, renorm_eps, ident, n_ident);
  if (rc != 0) return rc;
  LQ_REQUIRE(h && w && z && route, "moe_router: null pointer");
  LQ_REQUIRE(ldh >= K && ldw >= K && ldh % 8 == 0 && ldw % 8 == 0 && ((uintptr_t)h | (uintptr_t)w) % 16 == 0, "moe_router: rows must lie on 16 bytes");
  const RouteArgs a = {route, experts, top, renormalize, correction, groups, keep, softmax, mark_max, renorm_eps, ident, n_ident};
  moe_router_kernel<<<rows, ROUTER_WAVES * 64, 0, stream>>>((const bf16_t*)h, ldh, (const bf16_t*)w, ldw, z, ldz, K, N, a);
  LQ_CHECK_LAUNCH("moe_router");
  return 0;
}

extern "C" int lq_moe_identity(const void* h, int dtype, int ldh, const float* weights, int n, float* out, int ldo, int rows,
                               int width, hipStream_t stream) {
  LQ_REQUIRE(rows > 0 && width > 0 && n > 0 && ldh >= width && ldo >= width, "moe_identity: rows %d, width %d, %d experts", rows,
             width, n);
  LQ_REQUIRE(h && weights && out, "moe_identity: null pointer");
  if (dtype == LQ_F32)
    moe_identity_kernel<float><<<rows, 256, 0, stream>>>((const float*)h, ldh, weights, n, out, ldo, width);
  else if (dtype == LQ_BF16)
    moe_identity_kernel<bf16_t><<<rows, 256, 0, stream>>>((const bf16_t*)h, ldh, weights, n, out, ldo, width);
  else LQ_REQUIRE(false, "moe_identity: unknown dtype %d", dtype);
  LQ_CHECK_LAUNCH("moe_identity");
  return 0;
}

extern "C" int lq_moe_glu(const float* gu, long long ldg, const float* route, void* out, int out_dtype, long long ldo,
                          int rows, int experts, int ff, float limit, int on_input, int plain_silu, hipStream_t stream) {
  LQ_REQUIRE(rows > 0 && experts > 0 && ff > 0 && (long long)experts * ff <= 0x7fffffff, "moe_glu: rows %d, experts %d, inner %d",
             rows, experts, ff);
  LQ_REQUIRE(ldg >= 2ll * experts * ff && ldo >= (long long)experts * ff, "moe_glu: a row stride is smaller than its row");
  LQ_REQUIRE(gu && route && out, "moe_glu: null pointer");
  LQ_REQUIRE(out_dtype == LQ_F32 || out_dtype == LQ_BF16, "moe_glu: unknown dtype %d", out_dtype);
  // four entries a thread where they lie in whole vectors
  const bool quads = ff % 4 == 0 && ldg % 4 == 0 && ldo % 4 == 0 && ((uintptr_t)gu & 15) == 0 &&
                     ((uintptr_t)out & (out_dtype == LQ_BF16 ? 7 : 15)) == 0;
  for (int r0 = 0; r0 < rows; r0 += 65535) {
    const int nr = rows - r0 < 65535 ? rows - r0 : 65535;
    dim3 grid((unsigned)lq_ceil_div64((long long)experts * ff, quads ? 1024 : 256), nr);
#define LQ_MOE_GLU(T, VEC)                                                                                        \
  moe_glu_kernel<T, VEC><<<grid, 256, 0, stream>>>(gu + r0 * ldg, ldg, route + (long long)r0 * experts,           \
                                                   (T*)out + r0 * ldo, ldo, experts, ff, limit, on_input, plain_silu)
    if (out_dtype == LQ_F32) {
      if (quads) LQ_MOE_GLU(float, 4);
      else LQ_MOE_GLU(float, 1);
    } else {
      if (quads) LQ_MOE_GLU(bf16_t, 4);
      else LQ_MOE_GLU(bf16_t, 1);
    }
#undef LQ_MOE_GLU
  }
  LQ_CHECK_LAUNCH("moe_glu");
  return 0;
}

// u and out [rows, experts * ff + shared]; route [rows, experts]; act: an activation's number (device_math.h)
extern "C" int lq_moe_act(const float* u, long long ldu, const float* route, void* out, int out_dtype, long long ldo, int rows,
                          int experts, int ff, int shared, int act, hipStream_t stream) {
  const long long n = (long long)experts * ff + shared;
  LQ_REQUIRE(rows > 0 && experts > 0 && ff > 0 && shared >= 0 && n <= 0x7fffff00, "moe_act: rows %d, experts %d, inner %d, shared %d",
             rows, experts, ff, shared);
  LQ_REQUIRE(ldu >= n && ldo >= n, "moe_act: a row stride is smaller than its row");
  LQ_REQUIRE(u && route && out, "moe_act: null pointer");
  LQ_REQUIRE(act >= ACT_SILU && act <= ACT_RELU2, "moe_act: unknown activation %d", act);
  LQ_REQUIRE(out_dtype == LQ_F32 || out_dtype == LQ_BF16, "moe_act: unknown dtype %d", out_dtype);
  const int el = out_dtype == LQ_F32 ? 4 : 2;
  const bool fours = ff % 4 == 0 && shared % 4 == 0 && ldu % 4 == 0 && ldo % 4 == 0 && (uintptr_t)u % 16 == 0 &&
                     (uintptr_t)out % (4 * el) == 0;
  for (int r0 = 0; r0 < rows; r0 += 65535) {
    const int nr = rows - r0 < 65535 ? rows - r0 : 65535;
    const dim3 grid((unsigned)lq_ceil_div64(n, fours ? 1024 : 256), nr);
#define LQ_MOE_ACT(T, VEC)                                                                                              \
  moe_act_kernel<T, VEC><<<grid, 256, 0, stream>>>(u + r0 * ldu, ldu, route + (long long)r0 * experts, (T*)out + r0 * ldo, \
                                                   ldo, experts, ff, shared, act)
    if (out_dtype == LQ_F32 && fours) LQ_MOE_ACT(float, 4);
    else if (out_dtype == LQ_F32) LQ_MOE_ACT(float, 1);
    else if (fours) LQ_MOE_ACT(bf16_t, 4);
    else LQ_MOE_ACT(bf16_t, 1);
#undef LQ_MOE_ACT
  }
  LQ_CHECK_LAUNCH("moe_act");
  return 0;
}

// route [rows, experts] (a weight, or -1): counts [experts], order and weight [pairs] (pairs: the chosen
// (row, expert) couples, expert by expert, rows ascending), place_of [rows, experts]
extern "C" int lq_moe_sort(const float* route, int rows, int experts, int* counts, int* order, float* weight, int* place_of,
                           int places, hipStream_t stream) {
  LQ_REQUIRE(places >= 0, "moe_sort: %d places", places);
  LQ_REQUIRE(rows > 0 && rows < (1 << 24) && experts > 0 && experts <= 65535, "moe_sort: rows %d, experts %d", rows, experts);
  LQ_REQUIRE(route && counts && order && weight && place_of, "moe_sort: null pointer");
  moe_count_kernel<<<experts, SORT_THREADS, 0, stream>>>(route, rows, experts, counts);
  LQ_CHECK_LAUNCH("moe_sort(count)");
  moe_place_kernel<<<experts, SORT_THREADS, 0, stream>>>(route, rows, experts, counts, order, weight, place_of, places);
  LQ_CHECK_LAUNCH("moe_sort(place)");
  return 0;
}

extern "C" int lq_moe_gather(const void* src, int dtype, int ld, const int* order, void* dst, int n, int width,
                             hipStream_t stream) {
  LQ_REQUIRE(n > 0 && width > 0 && ld >= width, "moe_gather: %d rows of %d (stride %d)", n, width, ld);
  LQ_REQUIRE(src && order && dst, "moe_gather: null pointer");
  LQ_REQUIRE(dtype == LQ_F32 || dtype == LQ_BF16, "moe_gather: unknown dtype %d", dtype);
  const int per = dtype == LQ_F32 ? 4 : 8;  // entries in 16 bytes
  if (width % per == 0 && ld % per == 0 && (((uintptr_t)src | (uintptr_t)dst) & 15) == 0)
    moe_gather_kernel<uint4><<<n, 256, 0, stream>>>((const uint4*)src, ld / per, order, (uint4*)dst, width / per);
  else if (dtype == LQ_F32) moe_gather_kernel<float><<<n, 256, 0, stream>>>((const float*)src, ld, order, (float*)dst, width);
  else moe_gather_kernel<bf16_t><<<n, 256, 0, stream>>>((const bf16_t*)src, ld, order, (bf16_t*)dst, width);
  LQ_CHECK_LAUNCH("moe_gather");
  return 0;
}

extern "C" int lq_moe_scatter(const float* ys, const int* place_of, int experts, float* out, int ldo, int rows, int width,
                              hipStream_t stream) {
  LQ_REQUIRE(rows > 0 && width > 0 && experts > 0 && ldo >= width, "moe_scatter: rows %d, width %d, experts %d", rows, width, experts);
  LQ_REQUIRE(ys && place_of && out, "moe_scatter: null pointer");
  if (width % 4 == 0 && ldo % 4 == 0 && (((uintptr_t)ys | (uintptr_t)out) & 15) == 0)
    moe_scatter_kernel<4><<<rows, 256, 0, stream>>>(ys, place_of, experts, out, ldo, width);
  else
    moe_scatter_kernel<1><<<rows, 256, 0, stream>>>(ys, place_of, experts, out, ldo, width);
  LQ_CHECK_LAUNCH("moe_scatter");
  return 0;
}
