// Per-token log-probabilities of chosen tokens from bf16 logits, and their backward: the hot
// op of the policy-gradient loss around the model.  HBM-bound row streaming: the forward reads
// each logit once (online log-sum-exp in float32), the backward reads it once more and writes
// the bf16 gradient; no float32 copy of the logits and no [rows, vocab] log-softmax exist.
#include "mx_common.h"

namespace mx {

constexpr int kLpThreads = 256;
constexpr int kLpFwdThreads = 512, kLpFwdThreadsShort = 256;
constexpr int kLpUnroll = 4;
constexpr int kLpBwdUnroll = 2;

// Eight logits from any even address: rows of a vocabulary that is no multiple of 8 are read where
// they lie (the hardware takes 16-byte loads at any element; a copy of the logits to aligned rows
// would double their traffic).
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(2)));
__device__ __forceinline__ u32x4 lp_load8(const uint16_t* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(p));
}
__device__ __forceinline__ float lp_bf16(uint32_t lo16) { return __uint_as_float(lo16 << 16); }

// (max, sum of exp(x - max)) of two partial results; one whose max is -inf has met no number yet, and its
// sum is 0, or NaN if it has met a NaN.
__device__ __forceinline__ void lse_merge(float& m, float& s, float m2, float s2) {
  const float mm = fmaxf(m, m2);
  const float a = m == -__builtin_inff() ? s : s * __expf(m - mm);  // (exp(-inf - (-inf)) would be NaN)
  const float b = m2 == -__builtin_inff() ? s2 : s2 * __expf(m2 - mm);
  m = mm;
  s = a + b;
}

// lse[r] = log sum_v exp(x[r, v]); lp[r] = x[r, target[r]] - lse[r] (NaN if the target is outside
// [0, vocab)).
__device__ __forceinline__ void lp_finish(const uint16_t* row, int64_t vocab, int64_t t, float m, float s, float* lp,
                                          float* lse) {
  const float l = m + __logf(s);
  *lse = l;
  *lp = (t >= 0 && t < vocab) ? lp_bf16(row[t]) - l : __builtin_nanf("");
}

// One workgroup per row, or per `splits`-th part of a row, whose (max, sum) then goes to `partial`
// for token_logprob_merge_kernel.  HBM-bound: what counts is bytes in flight, so a lane asks for
// four 16-byte pieces before it uses the first, and rows are cut until the chip is full (a sample of
// a few hundred generated tokens has fewer rows than the chip has room for workgroups).
// 457 rows x 151 936: 52.6 us with one 256-lane workgroup per row and one piece in flight, 25.0 us now
// (5.5 TB/s); 16 rows: 54 before, 6.7 us in 12 parts each (16.0 uncut).
template <int THREADS, bool SPLIT>
__global__ __launch_bounds__(THREADS) void token_logprob_fwd_kernel(
    const uint16_t* __restrict__ logits, int64_t ld, int64_t vocab, const int64_t* __restrict__ target,
    float* __restrict__ lp, float* __restrict__ lse, int splits, float2* __restrict__ partial) {
  constexpr int kWaves = THREADS / 64;
  __shared__ float sm[kWaves], ss[kWaves];
  const int64_t r = SPLIT ? blockIdx.x / splits : blockIdx.x;
  const int part = SPLIT ? (int)(blockIdx.x - r * splits) : 0;
  const uint16_t* row = logits + r * ld;
  const int tid = threadIdx.x;
  float m = -__builtin_inff(), s = 0.f;
  const int64_t chunks = vocab / 8;
  const int64_t per = SPLIT ? (chunks + splits - 1) / splits : chunks;
  const int64_t lo = part * per, hi = lo + per < chunks ? lo + per : chunks;
  for (int64_t c = lo + tid; c < hi; c += THREADS * kLpUnroll) {
    u32x4 v[kLpUnroll];
#pragma unroll
    for (int u = 0; u < kLpUnroll; ++u) {
      const int64_t cu = c + u * THREADS;
      if (cu < hi) v[u] = lp_load8(row + cu * 8);
    }
#pragma unroll
    for (int u = 0; u < kLpUnroll; ++u) {
      if (c + u * THREADS >= hi) break;  // (no exponentials of nothing: 16384 rows x 8192 67 us with them, 50 without)
      const float x[8] = {lp_bf16(v[u].x & 0xFFFFu), lp_bf16(v[u].x >> 16), lp_bf16(v[u].y & 0xFFFFu),
                          lp_bf16(v[u].y >> 16),     lp_bf16(v[u].z & 0xFFFFu), lp_bf16(v[u].z >> 16),
                          lp_bf16(v[u].w & 0xFFFFu), lp_bf16(v[u].w >> 16)};
      float cm = x[0];
#pragma unroll
      for (int e = 1; e < 8; ++e) cm = fmaxf(cm, x[e]);
      if (cm > m) {  // rescale the running sum to the new maximum
        s = m == -__builtin_inff() ? s : s * __expf(m - cm);
        m = cm;
      }
      if (m != -__builtin_inff()) {
#pragma unroll
        for (int e = 0; e < 8; ++e) s += __expf(x[e] - m);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (x[e] != x[e]) s = x[e];
      }
    }
  }
  if (!SPLIT || part == splits - 1)
    for (int64_t i = chunks * 8 + tid; i < vocab; i += THREADS) {
      const float x = lp_bf16(row[i]);
      lse_merge(m, s, x, x == -__builtin_inff() ? 0.f : 1.f);
    }
  // across the workgroup: the maximum first, then one rescaling per lane and plain sums (merging
  // pairs step by step takes two exponentials a step and an eighth more time at 2000 rows x 8192)
  float top = m;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) top = fmaxf(top, __shfl_xor(top, off, 64));
  if ((tid & 63) == 0) sm[tid >> 6] = top;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kWaves; ++w) top = fmaxf(top, sm[w]);
  s = m == -__builtin_inff() ? s : s * __expf(m - top);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if ((tid & 63) == 0) ss[tid >> 6] = s;
  __syncthreads();
  if (tid == 0) {
    m = top;
    s = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s += ss[w];
    if constexpr (SPLIT)
      partial[blockIdx.x] = float2{m, s};
    else
      lp_finish(row, vocab, target[r], m, s, lp + r, lse + r);
  }
}

// The parts of every row put together, in order; one lane per row.
__global__ __launch_bounds__(64) void token_logprob_merge_kernel(const uint16_t* __restrict__ logits, int64_t ld,
                                                                 int64_t vocab, const int64_t* __restrict__ target,
                                                                 int64_t rows, int splits,
                                                                 const float2* __restrict__ partial,
                                                                 float* __restrict__ lp, float* __restrict__ lse) {
  const int64_t r = (int64_t)blockIdx.x * 64 + threadIdx.x;
  if (r >= rows) return;
  float m = -__builtin_inff(), s = 0.f;
  for (int p = 0; p < splits; ++p) {
    const float2 q = partial[r * splits + p];
    lse_merge(m, s, q.x, q.y);
  }
  lp_finish(logits + r * ld, vocab, target[r], m, s, lp + r, lse + r);
}

// dlogits[r, v] = g[r] * ((v == target[r]) - exp(x[r, v] - lse[r])) rounded to bf16.  HBM-bound; a
// workgroup takes kLpBwdUnroll pieces per lane of one row, all loads first.
__global__ __launch_bounds__(kLpThreads) void token_logprob_bwd_kernel(
    const uint16_t* __restrict__ logits, int64_t ld, int64_t vocab, const int64_t* __restrict__ target,
    const float* __restrict__ lse, const float* __restrict__ g, uint16_t* __restrict__ dlogits,
    int64_t ldd) {
  const int64_t r = blockIdx.y;
  const uint16_t* row = logits + r * ld;
  uint16_t* drow = dlogits + r * ldd;
  const float l = lse[r], gr = g[r];
  const int64_t t = target[r];
  const int64_t chunks = vocab / 8;
  auto grad = [&](float x, int64_t v) {
    const float p = __expf(x - l);
    const float d = gr * ((v == t ? 1.f : 0.f) - p);
    const uint32_t u = __float_as_uint(d);
    return (u & 0x7FFFFFFFu) > 0x7F800000u ? ((u >> 16) | 0x40u) : ((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
  };
  const int64_t c0 = (int64_t)blockIdx.x * (kLpThreads * kLpBwdUnroll) + threadIdx.x;
  u32x4 v[kLpBwdUnroll];
#pragma unroll
  for (int u = 0; u < kLpBwdUnroll; ++u) {
    const int64_t c = c0 + u * kLpThreads;
    if (c < chunks) v[u] = lp_load8(row + c * 8);
  }
#pragma unroll
  for (int u = 0; u < kLpBwdUnroll; ++u) {
    const int64_t c = c0 + u * kLpThreads;
    if (c >= chunks) break;
    const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      o[e] = grad(lp_bf16(w[e] & 0xFFFFu), c * 8 + 2 * e) | (grad(lp_bf16(w[e] >> 16), c * 8 + 2 * e + 1) << 16);
    __builtin_nontemporal_store(u32x4{o[0], o[1], o[2], o[3]}, reinterpret_cast<u32x4*>(drow + c * 8));
  }
  if (blockIdx.x == 0)
    for (int64_t i = chunks * 8 + threadIdx.x; i < vocab; i += kLpThreads)
      drow[i] = (uint16_t)grad(lp_bf16(row[i]), i);
}

}  // namespace mx

using namespace mx;

extern "C" int mx_token_logprob_fwd_split(const void* logits, int64_t rows, int64_t vocab, int64_t ld,
                                          const int64_t* target, float* logprob, float* lse, int64_t splits,
                                          float* partial, void* stream) {
  if (rows < 0 || vocab <= 0 || ld < vocab || splits < 1) return MX_ERR_INVALID_ARG;
  if (rows == 0) return MX_OK;
  if (!logits || !target || !logprob || !lse || (splits > 1 && !partial)) return MX_ERR_INVALID_ARG;
  if (((uintptr_t)logits & 1) || ((uintptr_t)target & 7) || ((uintptr_t)logprob & 3) || ((uintptr_t)lse & 3) ||
      ((uintptr_t)partial & 7))
    return MX_ERR_ALIGNMENT;
  if (rows > 0x7FFFFFFF || splits > 65535 || rows * splits > 0x7FFFFFFF) return MX_ERR_UNSUPPORTED;
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)(rows * splits)), block(kLpFwdThreads), small(kLpFwdThreadsShort);
  auto whole_rows = [&](auto kernel, dim3 lanes) {
    hipLaunchKernelGGL(kernel, grid, lanes, 0, st, (const uint16_t*)logits, ld, vocab, target, logprob, lse, 1, (float2*)nullptr);
  };
  if (splits == 1) {
    // Rows that 512 lanes read with four pieces in flight half empty, and more of them than the chip holds at
    // once: half the lanes, us, 512 / 256: 16384 rows x 8192 49.7 / 39.2, 2000 rows x 1000 5.2 / 3.7, x 8192
    // 8.4 / 7.6, x 12288 10.0 / 9.7; 4096 rows x 16000 21.3 / 22.6, x 32000 39.4 / 42.9; 16 rows x 8192 3.3 / 3.8
    if (vocab <= 12288 && rows > 512) whole_rows(token_logprob_fwd_kernel<kLpFwdThreadsShort, false>, small);
    else whole_rows(token_logprob_fwd_kernel<kLpFwdThreads, false>, block);
  } else {
    hipLaunchKernelGGL((token_logprob_fwd_kernel<kLpFwdThreads, true>), grid, block, 0, st, (const uint16_t*)logits, ld,
                       vocab, target, logprob, lse, (int)splits, (float2*)partial);
    hipLaunchKernelGGL(token_logprob_merge_kernel, dim3((unsigned)((rows + 63) / 64)), dim3(64), 0, st,
                       (const uint16_t*)logits, ld, vocab, target, rows, (int)splits, (const float2*)partial, logprob, lse);
  }
  return hipGetLastError() == hipSuccess ? MX_OK : MX_ERR_LAUNCH;
}

extern "C" int mx_token_logprob_fwd(const void* logits, int64_t rows, int64_t vocab, int64_t ld,
                                    const int64_t* target, float* logprob, float* lse, void* stream) {
  if (rows > 0 && vocab > 0 && ld >= vocab && logits && (ld % 8 || ((uintptr_t)logits & 15))) return MX_ERR_ALIGNMENT;
  return mx_token_logprob_fwd_split(logits, rows, vocab, ld, target, logprob, lse, 1, nullptr, stream);
}

extern "C" int mx_token_logprob_bwd_any(const void* logits, int64_t rows, int64_t vocab, int64_t ld,
                                        const int64_t* target, const float* lse, const float* grad_logprob,
                                        void* dlogits, int64_t ldd, void* stream) {
  if (rows < 0 || vocab <= 0 || ld < vocab || ldd < vocab) return MX_ERR_INVALID_ARG;
  if (rows == 0) return MX_OK;
  if (!logits || !target || !lse || !grad_logprob || !dlogits) return MX_ERR_INVALID_ARG;
  if (ldd % 8 || ((uintptr_t)logits & 1) || ((uintptr_t)dlogits & 15) || ((uintptr_t)target & 7) ||
      ((uintptr_t)lse & 3) || ((uintptr_t)grad_logprob & 3))
    return MX_ERR_ALIGNMENT;
  if (rows > 65535) return MX_ERR_UNSUPPORTED;  // one grid row per token row
  const int64_t chunks = vocab / 8, per = kLpThreads * kLpBwdUnroll;
  const int64_t gx = chunks > per ? (chunks + per - 1) / per : 1;
  if (gx > 0x7FFFFFFF) return MX_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(token_logprob_bwd_kernel, dim3((unsigned)gx, (unsigned)rows), dim3(kLpThreads), 0,
                     (hipStream_t)stream, (const uint16_t*)logits, ld, vocab, target, lse, grad_logprob,
                     (uint16_t*)dlogits, ldd);
  return hipGetLastError() == hipSuccess ? MX_OK : MX_ERR_LAUNCH;
}

extern "C" int mx_token_logprob_bwd(const void* logits, int64_t rows, int64_t vocab, int64_t ld,
                                    const int64_t* target, const float* lse, const float* grad_logprob,
                                    void* dlogits, int64_t ldd, void* stream) {
  if (rows > 0 && vocab > 0 && ld >= vocab && ldd >= vocab && logits && target && lse && grad_logprob && dlogits &&
      (ld % 8 || ((uintptr_t)logits & 15)))
    return MX_ERR_ALIGNMENT;
  return mx_token_logprob_bwd_any(logits, rows, vocab, ld, target, lse, grad_logprob, dlogits, ldd, stream);
}
