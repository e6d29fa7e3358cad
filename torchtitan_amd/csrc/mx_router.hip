// Token-choice routing of an MoE layer from the router's float32 logits: scores, top-k choice, weights
// of the chosen experts and their gradient, and the maps from (token, choice) pairs to rows of the
// aligned expert groups.  Small integer and float work whose cost is launches and latency: one wave
// owns a token, its logits stay in registers, and what a sort would do is counted instead.
#include "mx_common.h"

namespace mx {

constexpr int kRouteThreads = 256;
constexpr int kRouteWaves = kRouteThreads / 64;
// Tokens of one workgroup: few enough that 16 384 tokens give every SIMD four waves to hide the
// serial chain of the k selections behind one another, many enough that the per-workgroup counts
// (experts x workgroups) stay small.
constexpr int kRouteTokens = 16;
constexpr int kRouteMaxExperts = 512;
constexpr int kRouteMaxTopK = 16;
static_assert(kRouteTokens * kRouteMaxTopK <= kRouteThreads, "one lane per pair of a workgroup");

// Reductions over the 64 lanes, result in all of them: four DPP steps inside rows of 16, then the
// four row results as scalars.
template <class F>
__device__ __forceinline__ uint32_t wave_reduce(uint32_t v, F&& f) {
  v = f(v, dpp<kQuadXor1>(v));
  v = f(v, dpp<kQuadXor2>(v));
  v = f(v, dpp<0x141>(v));  // row_half_mirror: the other quad of 8 lanes
  v = f(v, dpp<0x140>(v));  // row_mirror: the other 8 of 16 lanes
  const uint32_t a = __builtin_amdgcn_readlane(v, 0), b = __builtin_amdgcn_readlane(v, 16);
  const uint32_t c = __builtin_amdgcn_readlane(v, 32), d = __builtin_amdgcn_readlane(v, 48);
  return f(f(a, b), f(c, d));
}
__device__ __forceinline__ float wave_sum(float v) {
  return __uint_as_float(wave_reduce(__float_as_uint(v), [](uint32_t a, uint32_t b) {
    return __float_as_uint(__uint_as_float(a) + __uint_as_float(b));
  }));
}
__device__ __forceinline__ float wave_max(float v) {
  return __uint_as_float(wave_reduce(__float_as_uint(v), [](uint32_t a, uint32_t b) {
    return __float_as_uint(fmaxf(__uint_as_float(a), __uint_as_float(b)));
  }));
}

// A float as an unsigned number of the same order, a NaN of either sign above all as torch.topk has it; never 0,
// which marks a place that is taken.
__device__ __forceinline__ uint32_t order_key(float f) {
  if (f != f) return 0xFFFFFFFFu;
  const uint32_t u = __float_as_uint(f);
  const uint32_t k = u ^ ((u >> 31) ? 0xFFFFFFFFu : 0x80000000u);
  return k ? k : 1u;
}

// Scores of one token, lane l holding experts l, l + 64, ...: softmax or sigmoid in float32.
template <int VPL, bool SOFTMAX>
__device__ __forceinline__ void route_scores(const float* __restrict__ row, int experts, int lane, float (&s)[VPL]) {
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int e = lane + 64 * i;
    s[i] = e < experts ? row[e] : -__builtin_inff();
  }
  if (SOFTMAX) {
    float m = s[0];
#pragma unroll
    for (int i = 1; i < VPL; ++i) m = fmaxf(m, s[i]);
    m = wave_max(m);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      s[i] = expf(s[i] - m);
      sum += s[i];
    }
    sum = wave_sum(sum);
#pragma unroll
    for (int i = 0; i < VPL; ++i) s[i] = s[i] / sum;
  } else {
#pragma unroll
    for (int i = 0; i < VPL; ++i) s[i] = 1.0f / (1.0f + expf(-s[i]));
  }
}

// The k experts of largest score + bias (ties: the lowest number first) of every token in falling
// order, their weights -- the scores, normalised over the chosen ones if asked, times `scale` -- and
// per workgroup and expert how many pairs chose it: block_counts[e * blocks + b].
template <int VPL, bool SOFTMAX>
__global__ __launch_bounds__(kRouteThreads) void route_topk_kernel(
    const float* __restrict__ logits, int64_t tokens, int experts, const float* __restrict__ bias, int top_k,
    int norm, float scale, float* __restrict__ top, int64_t* __restrict__ selected,
    int32_t* __restrict__ block_counts) {
  __shared__ int32_t counts[kRouteMaxExperts];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int e = tid; e < experts; e += kRouteThreads) counts[e] = 0;
  __syncthreads();
  for (int j = wave; j < kRouteTokens; j += kRouteWaves) {
    const int64_t t = (int64_t)blockIdx.x * kRouteTokens + j;
    if (t >= tokens) break;
    float s[VPL];
    route_scores<VPL, SOFTMAX>(logits + t * experts, experts, lane, s);
    uint32_t key[VPL];
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      const int e = lane + 64 * i;
      key[i] = e < experts ? order_key(bias ? s[i] + bias[e] : s[i]) : 0u;
    }
    int mine = 0;       // lane c: the c-th choice ...
    float mine_s = 0.f;  // ... and its score
    for (int c = 0; c < top_k; ++c) {
      uint32_t best = key[0];
#pragma unroll
      for (int i = 1; i < VPL; ++i) best = max(best, key[i]);
      best = wave_reduce(best, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
      int winner = 0;
      float score = 0.f;
      bool found = false;
#pragma unroll
      for (int i = 0; i < VPL; ++i) {
        const uint64_t at = __builtin_amdgcn_ballot_w64(!found && key[i] == best);
        if (at) {
          const int l = __builtin_ctzll(at);
          winner = l + 64 * i;
          score = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(s[i]), l));
          if (lane == l) key[i] = 0u;
          found = true;
        }
      }
      if (lane == c) {
        mine = winner;
        mine_s = score;
      }
    }
    // summed as a tree: one after the other the weights of 8 of 128 experts are 6.5e-8 from float64, so 5.5e-8
    const float sum = norm ? wave_sum(mine_s) : 0.f;
    if (lane < top_k) {
      float w = norm ? mine_s / (sum + 1e-20f) : mine_s;
      w *= scale;
      top[t * top_k + lane] = w;
      selected[t * top_k + lane] = mine;
      atomicAdd(&counts[mine], 1);
    }
  }
  __syncthreads();
  for (int e = tid; e < experts; e += kRouteThreads) block_counts[(int64_t)e * gridDim.x + blockIdx.x] = counts[e];
}

// Gradient with respect to the logits: dense [tokens, experts] from that of the chosen weights.
template <int VPL, bool SOFTMAX>
__global__ __launch_bounds__(kRouteThreads) void route_topk_bwd_kernel(
    const float* __restrict__ logits, int64_t tokens, int experts, int top_k, int norm, float scale,
    const int64_t* __restrict__ selected, const float* __restrict__ dtop, float* __restrict__ dlogits) {
  const int lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * kRouteWaves + (threadIdx.x >> 6);
  if (t >= tokens) return;
  float s[VPL], ds[VPL];
  route_scores<VPL, SOFTMAX>(logits + t * experts, experts, lane, s);
#pragma unroll
  for (int i = 0; i < VPL; ++i) ds[i] = 0.f;
  // lane c: the c-th choice, its score and the gradient of its weight
  int e_c = 0;
  float g_c = 0.f, s_c = 0.f;
  if (lane < top_k) {
    e_c = (int)selected[t * top_k + lane];
    g_c = dtop[t * top_k + lane] * scale;
  }
  for (int c = 0; c < top_k; ++c) {
    const int e = __builtin_amdgcn_readlane(e_c, c);
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < VPL; ++i)
      if ((e >> 6) == i) v = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(s[i]), e & 63));
    if (lane == c) s_c = v;
  }
  if (norm) {  // w = s / S, S = sum of the chosen: dw/ds = g / S - (sum g s) / S^2
    const float total = wave_sum(s_c) + 1e-20f, dot = wave_sum(g_c * s_c);
    g_c = g_c / total - dot / (total * total);
  }
  for (int c = 0; c < top_k; ++c) {
    const int e = __builtin_amdgcn_readlane(e_c, c);
    const float g = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(g_c), c));
#pragma unroll
    for (int i = 0; i < VPL; ++i)
      if (e == lane + 64 * i) ds[i] = g;
  }
  float dot = 0.f;
  if (SOFTMAX) {
#pragma unroll
    for (int i = 0; i < VPL; ++i) dot += ds[i] * s[i];
    dot = wave_sum(dot);
  }
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int e = lane + 64 * i;
    if (e < experts) dlogits[t * experts + e] = SOFTMAX ? s[i] * (ds[i] - dot) : ds[i] * s[i] * (1.0f - s[i]);
  }
}

// One workgroup per expert: block_counts[e][.] to exclusive prefix sums, their total to counts[e].
__global__ __launch_bounds__(kRouteThreads) void route_scan_kernel(int32_t* __restrict__ block_counts, int blocks,
                                                                   int64_t* __restrict__ counts) {
  __shared__ int32_t part[kRouteThreads];
  int32_t* mine = block_counts + (int64_t)blockIdx.x * blocks;
  const int tid = threadIdx.x;
  const int per = (blocks + kRouteThreads - 1) / kRouteThreads;
  const int lo = min(tid * per, blocks), hi = min(lo + per, blocks);
  int32_t sum = 0;
  for (int i = lo; i < hi; ++i) sum += mine[i];
  part[tid] = sum;
  __syncthreads();
  for (int off = 1; off < kRouteThreads; off <<= 1) {
    const int32_t add = tid >= off ? part[tid - off] : 0;
    __syncthreads();
    part[tid] += add;
    __syncthreads();
  }
  int32_t run = part[tid] - sum;
  for (int i = lo; i < hi; ++i) {
    const int32_t c = mine[i];
    mine[i] = run;
    run += c;
  }
  if (tid == kRouteThreads - 1) counts[blockIdx.x] = part[tid];
}

// The plan of mx_moe_route_plan from the choices themselves: within a group the pairs keep the order of
// their tokens, so a pair's row is the group's start + pairs of earlier workgroups + pairs before
// it in its own.  The workgroups past the last token block clear the rows no pair owns.
__global__ __launch_bounds__(kRouteThreads) void route_fill_kernel(
    const int64_t* __restrict__ selected, const float* __restrict__ scores, int64_t pairs, int top_k, int experts,
    const int32_t* __restrict__ block_counts, int blocks, const int64_t* __restrict__ counts, int64_t max_len,
    int alignment, int32_t* __restrict__ m_offsets, int64_t* __restrict__ src_row, float* __restrict__ row_score,
    int64_t* __restrict__ pos) {
  __shared__ int32_t ends[kRouteMaxExperts];  // inclusive padded group ends
  __shared__ int32_t part[kRouteThreads];
  __shared__ int32_t chosen[kRouteThreads];
  const int tid = threadIdx.x;
  auto padded = [&](int e) -> int32_t {
    const int32_t c = (int32_t)counts[e];
    return ((c < alignment ? alignment : c) + alignment - 1) / alignment * alignment;
  };
  constexpr int kPer = kRouteMaxExperts / kRouteThreads;
  int32_t sum = 0;
#pragma unroll
  for (int i = 0; i < kPer; ++i)
    if (tid * kPer + i < experts) sum += padded(tid * kPer + i);
  part[tid] = sum;
  const int64_t base = (int64_t)blockIdx.x * (kRouteTokens * top_k);
  const int n = base < pairs ? (int)min((int64_t)kRouteTokens * top_k, pairs - base) : 0;
  if (tid < n) chosen[tid] = (int32_t)selected[base + tid];
  __syncthreads();
  for (int off = 1; off < kRouteThreads; off <<= 1) {
    const int32_t add = tid >= off ? part[tid - off] : 0;
    __syncthreads();
    part[tid] += add;
    __syncthreads();
  }
  int32_t run = part[tid] - sum;
#pragma unroll
  for (int i = 0; i < kPer; ++i)
    if (tid * kPer + i < experts) {
      run += padded(tid * kPer + i);
      ends[tid * kPer + i] = run;
    }
  __syncthreads();

  if ((int)blockIdx.x < blocks) {
    if (tid < n) {
      const int e = chosen[tid];
      int32_t rank = 0;
      for (int i = 0; i < tid; ++i) rank += chosen[i] == e;
      const int64_t p = (int64_t)(e ? ends[e - 1] : 0) + block_counts[(int64_t)e * blocks + blockIdx.x] + rank;
      const int64_t pair = base + tid;
      if (p < max_len) {
        src_row[p] = pair / top_k;
        row_score[p] = scores[pair];
      }
      pos[pair] = p;
    }
    return;
  }
  const int w = blockIdx.x - blocks, width = gridDim.x - blocks;
  if (w == 0)
    for (int e = tid; e < experts; e += kRouteThreads) m_offsets[e] = ends[e];
  for (int e = w; e < experts; e += width) {
    const int64_t from = (int64_t)(e ? ends[e - 1] : 0) + (int32_t)counts[e], to = ends[e];
    for (int64_t p = from + tid; p < to && p < max_len; p += kRouteThreads) {
      src_row[p] = -1;
      row_score[p] = 0.f;
    }
  }
  for (int64_t p = (int64_t)ends[experts - 1] + w * kRouteThreads + tid; p < max_len; p += width * kRouteThreads) {
    src_row[p] = -1;
    row_score[p] = 0.f;
  }
}

static inline int64_t route_blocks(int64_t tokens) { return (tokens + kRouteTokens - 1) / kRouteTokens; }

static int check_route(int64_t tokens, int64_t experts, int64_t top_k) {
  if (tokens < 0 || experts <= 0 || top_k <= 0 || top_k > experts) return MX_ERR_INVALID_ARG;
  if (experts > kRouteMaxExperts || top_k > kRouteMaxTopK || tokens * top_k > 0x7FFFFFFF) return MX_ERR_UNSUPPORTED;
  return MX_OK;
}

}  // namespace mx

using namespace mx;

#define MX_ROUTE_DISPATCH(KERNEL, GRID, ...)                                                                   \
  do {                                                                                                         \
    const dim3 grid_((unsigned)(GRID)), block_(kRouteThreads);                                                 \
    const int vpl_ = experts <= 64 ? 1 : experts <= 128 ? 2 : experts <= 256 ? 4 : 8;                          \
    if (softmax) {                                                                                             \
      if (vpl_ == 1) hipLaunchKernelGGL((KERNEL<1, true>), grid_, block_, 0, st, __VA_ARGS__);                 \
      else if (vpl_ == 2) hipLaunchKernelGGL((KERNEL<2, true>), grid_, block_, 0, st, __VA_ARGS__);            \
      else if (vpl_ == 4) hipLaunchKernelGGL((KERNEL<4, true>), grid_, block_, 0, st, __VA_ARGS__);            \
      else hipLaunchKernelGGL((KERNEL<8, true>), grid_, block_, 0, st, __VA_ARGS__);                           \
    } else {                                                                                                   \
      if (vpl_ == 1) hipLaunchKernelGGL((KERNEL<1, false>), grid_, block_, 0, st, __VA_ARGS__);                \
      else if (vpl_ == 2) hipLaunchKernelGGL((KERNEL<2, false>), grid_, block_, 0, st, __VA_ARGS__);           \
      else if (vpl_ == 4) hipLaunchKernelGGL((KERNEL<4, false>), grid_, block_, 0, st, __VA_ARGS__);           \
      else hipLaunchKernelGGL((KERNEL<8, false>), grid_, block_, 0, st, __VA_ARGS__);                          \
    }                                                                                                          \
  } while (0)

extern "C" int64_t mx_route_blocks(int64_t tokens) { return tokens < 0 ? -1 : route_blocks(tokens); }

extern "C" int mx_route_topk(const float* logits, int64_t tokens, int64_t experts, const float* bias, int64_t top_k,
                             int softmax, int norm, float scale, float* top_scores, int64_t* selected,
                             int64_t* counts, int32_t* block_counts, void* stream) {
  if (const int rc = check_route(tokens, experts, top_k)) return rc;
  if (!counts || (tokens > 0 && (!logits || !top_scores || !selected || !block_counts))) return MX_ERR_INVALID_ARG;
  hipStream_t st = (hipStream_t)stream;
  const int64_t blocks = route_blocks(tokens);
  if (tokens > 0)
    MX_ROUTE_DISPATCH(route_topk_kernel, blocks, logits, tokens, (int)experts, bias, (int)top_k, norm, scale, top_scores,
                      selected, block_counts);
  hipLaunchKernelGGL(route_scan_kernel, dim3((unsigned)experts), dim3(kRouteThreads), 0, st, block_counts, (int)blocks,
                     counts);
  return hipGetLastError() == hipSuccess ? MX_OK : MX_ERR_LAUNCH;
}

extern "C" int mx_route_topk_bwd(const float* logits, int64_t tokens, int64_t experts, int64_t top_k, int softmax,
                                 int norm, float scale, const int64_t* selected, const float* dtop, float* dlogits,
                                 void* stream) {
  if (const int rc = check_route(tokens, experts, top_k)) return rc;
  if (tokens == 0) return MX_OK;
  if (!logits || !selected || !dtop || !dlogits) return MX_ERR_INVALID_ARG;
  hipStream_t st = (hipStream_t)stream;
  MX_ROUTE_DISPATCH(route_topk_bwd_kernel, (tokens + kRouteWaves - 1) / kRouteWaves, logits, tokens, (int)experts,
                    (int)top_k, norm, scale, selected, dtop, dlogits);
  return hipGetLastError() == hipSuccess ? MX_OK : MX_ERR_LAUNCH;
}

extern "C" int mx_route_fill(const int64_t* selected, const float* scores, int64_t tokens, int64_t top_k,
                             int64_t experts, const int32_t* block_counts, const int64_t* counts,
                             int64_t max_len, int64_t alignment, int32_t* m_offsets, int64_t* src_row,
                             float* row_score, int64_t* pos, void* stream) {
  if (const int rc = check_route(tokens, experts, top_k)) return rc;
  if (max_len < 0 || alignment <= 0) return MX_ERR_INVALID_ARG;
  if (!counts || !m_offsets || (tokens > 0 && (!selected || !scores || !block_counts || !pos)) ||
      (max_len > 0 && (!src_row || !row_score)))
    return MX_ERR_INVALID_ARG;
  if (alignment > (1 << 20) || max_len > 0x7FFFFFFF) return MX_ERR_UNSUPPORTED;
  const int64_t blocks = route_blocks(tokens), cleaners = experts < 32 ? experts : 32;
  hipLaunchKernelGGL(route_fill_kernel, dim3((unsigned)(blocks + cleaners)), dim3(kRouteThreads), 0,
                     (hipStream_t)stream, selected, scores, tokens * top_k, (int)top_k, (int)experts, block_counts,
                     (int)blocks, counts, max_len, (int)alignment, m_offsets, src_row, row_score, pos);
  return hipGetLastError() == hipSuccess ? MX_OK : MX_ERR_LAUNCH;
}
