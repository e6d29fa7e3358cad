// Routed-token side of the MoE layer around the expert GEMMs: the weighted sum that brings the
// top-k expert outputs of a token back together, and the row dot products that give the
// gradient of the routing scores.  HBM-bound row streaming, float32 arithmetic in a fixed order.
#include <type_traits>

#include "mx_common.h"

namespace mx {

constexpr int kMoeThreads = 256;

__device__ __forceinline__ float bf16_bits_f32(uint32_t w_lo16) { return __uint_as_float(w_lo16 << 16); }

// float32 -> bf16 bits, round to nearest even, NaN kept quiet.
__device__ __forceinline__ uint32_t f32_bf16_bits(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (u >> 16) | 0x40u;
  return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

// a * b rounded to float32 on its own: the empty asm keeps the compiler from contracting the
// product into the addition that follows (one rounding instead of the stated two).
__device__ __forceinline__ float rounded_product(float a, float b) {
  float p = a * b;
  asm volatile("" : "+v"(p));
  return p;
}

// bf16(a + b) of two bf16 values, as a bf16 tensor addition forms it.
__device__ __forceinline__ float bf16_sum(uint32_t a16, uint32_t b16) {
  return bf16_bits_f32(f32_bf16_bits(bf16_bits_f32(a16) + bf16_bits_f32(b16)));
}

// The 8 bf16 values of one 16-byte piece, with y2 as bf16(y + y2).
template <bool TWO>
__device__ __forceinline__ void piece_f32(const u32x4& v, const u32x4& v2, float* x) {
  const uint32_t d[4] = {v.x, v.y, v.z, v.w}, d2[4] = {v2.x, v2.y, v2.z, v2.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    x[2 * e] = TWO ? bf16_sum(d[e] & 0xFFFFu, d2[e] & 0xFFFFu) : bf16_bits_f32(d[e] & 0xFFFFu);
    x[2 * e + 1] = TWO ? bf16_sum(d[e] >> 16, d2[e] >> 16) : bf16_bits_f32(d[e] >> 16);
  }
}

__device__ __forceinline__ u32x4 pack_piece(const float* acc) {
  u32x4 o;
  o.x = f32_bf16_bits(acc[0]) | (f32_bf16_bits(acc[1]) << 16);
  o.y = f32_bf16_bits(acc[2]) | (f32_bf16_bits(acc[3]) << 16);
  o.z = f32_bf16_bits(acc[4]) | (f32_bf16_bits(acc[5]) << 16);
  o.w = f32_bf16_bits(acc[6]) | (f32_bf16_bits(acc[7]) << 16);
  return o;
}

// out[t, :] = sum_j w[t, j] * y[pos[t, j], :]   (j = 0 .. k-1 in that order, float32, the product
// and the sum rounded separately; w == nullptr: plain sum).  A position outside [0, y_rows)
// contributes nothing.  With y2 (TWO), the rows summed are bf16(y + y2) (two matrices of one shape
// that a bf16 addition would have merged first).  One lane per 8 columns, grid-stride over
// (token, column chunk).  Bound by reading y: the rows of KU choices are asked for before the
// first is used (an out-of-range one reads row 0 and is dropped at its use); 16384 tokens, 8 choices,
// 2048 columns: 108 us, 5.6 TB/s (one row after the other: 128 us).
template <int KU, bool TWO>
__global__ __launch_bounds__(kMoeThreads) void moe_combine_kernel(
    const uint16_t* __restrict__ y, const uint16_t* __restrict__ y2, int64_t y_rows, int64_t ldy,
    const int64_t* __restrict__ pos,
    const float* __restrict__ w, int64_t tokens, int k, int64_t cols, uint16_t* __restrict__ out,
    int64_t ldo) {
  const int64_t chunks = cols / 8;
  const int64_t total = tokens * chunks;
  if (y_rows == 0) k = 0;
  for (int64_t i = (int64_t)blockIdx.x * kMoeThreads + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * kMoeThreads) {
    const int64_t t = i / chunks, c = (i - t * chunks) * 8;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int j0 = 0; j0 < k; j0 += KU) {
      u32x4 v[KU], v2[KU];
      bool in[KU];
#pragma unroll
      for (int j = 0; j < KU; ++j) {
        const int64_t r = pos[t * k + (j0 + j < k ? j0 + j : 0)];
        in[j] = j0 + j < k && r >= 0 && r < y_rows;
        const int64_t at = (in[j] ? r : 0) * ldy + c;
        v[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(y + at));
        if (TWO) v2[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(y2 + at));
      }
#pragma unroll
      for (int j = 0; j < KU; ++j) {
        if (!in[j]) continue;
        float x[8];
        piece_f32<TWO>(v[j], TWO ? v2[j] : v[j], x);
        const float s = w ? w[t * k + j0 + j] : 1.0f;  // 1 * x is x: the plain sum
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += rounded_product(s, x[e]);
      }
    }
    *reinterpret_cast<u32x4*>(out + t * ldo + c) = pack_piece(acc);
  }
}

// The weighted sum above and dots[t, j] = <y[pos[t, j], :], x[t, :]> (float32; 0 for a position
// outside y) from one read of y: in the backward of an MoE layer whose scores multiply the expert
// inputs, the rows that are summed into dx are those whose products with x are the scores' gradient.
// OUT = false leaves the sum out.  One wave per token, its lanes on 8-column pieces, the k <= KU
// rows of a piece in flight together; the dot products add the pieces and then the lanes in the
// order of moe_row_dot_kernel, so both give the same bits.  At the size above 125 us for what took
// 128 + 123 us as two kernels.
template <int KU, bool OUT>
__global__ __launch_bounds__(kMoeThreads) void moe_combine_dot_kernel(
    const uint16_t* __restrict__ y, int64_t y_rows, int64_t ldy, const int64_t* __restrict__ pos,
    const float* __restrict__ w, const uint16_t* __restrict__ x, int64_t ldx, int64_t tokens, int k,
    int64_t cols, uint16_t* __restrict__ out, int64_t ldo, float* __restrict__ dots) {
  const int lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * (kMoeThreads / 64) +
                    __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (t >= tokens) return;
  int64_t row[KU];
  float s[KU], dot[KU];
  bool in[KU];
#pragma unroll
  for (int j = 0; j < KU; ++j) {
    const int64_t at = t * k + (j < k ? j : 0);
    row[j] = pos[at];
    s[j] = OUT && w ? w[at] : 1.0f;
    in[j] = j < k && row[j] >= 0 && row[j] < y_rows;
    row[j] = (in[j] ? row[j] : 0) * ldy;
    dot[j] = 0.f;
  }
  for (int64_t c = lane * 8; c < cols; c += 64 * 8) {
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (y_rows > 0) {
      u32x4 v[KU];
#pragma unroll
      for (int j = 0; j < KU; ++j)
        v[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(y + row[j] + c));
      const u32x4 vx = *reinterpret_cast<const u32x4*>(x + t * ldx + c);
      float b[8];
      piece_f32<false>(vx, vx, b);
#pragma unroll
      for (int j = 0; j < KU; ++j) {
        if (!in[j]) continue;
        float a[8];
        piece_f32<false>(v[j], v[j], a);
#pragma unroll
        for (int e = 0; e < 8; ++e) dot[j] = __builtin_fmaf(a[e], b[e], dot[j]);
        if (OUT) {
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[e] += rounded_product(s[j], a[e]);
        }
      }
    }
    if (OUT) *reinterpret_cast<u32x4*>(out + t * ldo + c) = pack_piece(acc);
  }
#pragma unroll
  for (int j = 0; j < KU; ++j) {
    if (j >= k) break;
    float d = dot[j];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) d += __shfl_xor(d, off, 64);
    if (lane == 0) dots[t * k + j] = d;
  }
}

// out[i] = sum_d a[ia[i], d] * b[ib[i], d] in float32; a row index outside its matrix gives 0.
// With a2, a's rows are bf16(a + a2).  One wave per output: lanes stride over 8-column chunks,
// then a butterfly over the 64 lanes.
__global__ __launch_bounds__(kMoeThreads) void moe_row_dot_kernel(
    const uint16_t* __restrict__ a, const uint16_t* __restrict__ a2, int64_t a_rows, int64_t lda,
    const int64_t* __restrict__ ia,
    const uint16_t* __restrict__ b, int64_t b_rows, int64_t ldb, const int64_t* __restrict__ ib,
    int64_t n, int64_t cols, float* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  const int64_t wave = ((int64_t)blockIdx.x * kMoeThreads + threadIdx.x) >> 6;
  const int64_t waves = ((int64_t)gridDim.x * kMoeThreads) >> 6;
  for (int64_t i = wave; i < n; i += waves) {
    const int64_t ra = ia[i], rb = ib[i];
    float acc = 0.f;
    if (ra >= 0 && ra < a_rows && rb >= 0 && rb < b_rows) {
      for (int64_t c = lane * 8; c < cols; c += 64 * 8) {
        const u32x4 va = *reinterpret_cast<const u32x4*>(a + ra * lda + c);
        const u32x4 vb = *reinterpret_cast<const u32x4*>(b + rb * ldb + c);
        const uint32_t da[4] = {va.x, va.y, va.z, va.w}, db[4] = {vb.x, vb.y, vb.z, vb.w};
        float xa[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          xa[2 * e] = bf16_bits_f32(da[e] & 0xFFFFu);
          xa[2 * e + 1] = bf16_bits_f32(da[e] >> 16);
        }
        if (a2) {
          const u32x4 v2 = *reinterpret_cast<const u32x4*>(a2 + ra * lda + c);
          const uint32_t d2[4] = {v2.x, v2.y, v2.z, v2.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            xa[2 * e] = bf16_sum(da[e] & 0xFFFFu, d2[e] & 0xFFFFu);
            xa[2 * e + 1] = bf16_sum(da[e] >> 16, d2[e] >> 16);
          }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc = __builtin_fmaf(xa[2 * e], bf16_bits_f32(db[e] & 0xFFFFu), acc);
          acc = __builtin_fmaf(xa[2 * e + 1], bf16_bits_f32(db[e] >> 16), acc);
        }
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) out[i] = acc;
  }
}

static inline unsigned moe_grid(int64_t work_items) {
  const int64_t blocks = (work_items + kMoeThreads - 1) / kMoeThreads;
  const int64_t cap = 256 * 16;  // 16 workgroups per CU keep every CU streaming
  return (unsigned)(blocks < 1 ? 1 : (blocks > cap ? cap : blocks));
}

}  // namespace mx

using namespace mx;

extern "C" int mx_moe_combine(const void* y, const void* y2, int64_t y_rows, int64_t ldy,
                              const int64_t* pos,
                              const float* weights, int64_t tokens, int64_t top_k, int64_t cols,
                              void* out, int64_t ldo, void* stream) {
  if (y_rows < 0 || tokens < 0 || top_k < 0 || top_k > 1024 || cols < 0 || ldy < cols || ldo < cols)
    return MX_ERR_INVALID_ARG;
  if (tokens == 0 || cols == 0) return MX_OK;
  if (!out || (top_k > 0 && (!y || !pos))) return MX_ERR_INVALID_ARG;
  if (cols % 8 || ldy % 8 || ldo % 8 || ((uintptr_t)y & 15) || ((uintptr_t)y2 & 15) ||
      ((uintptr_t)out & 15) || ((uintptr_t)pos & 7) || ((uintptr_t)weights & 3))
    return MX_ERR_ALIGNMENT;
  const dim3 grid(moe_grid(tokens * (cols / 8)));
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kMoeThreads), 0, (hipStream_t)stream, (const uint16_t*)y,
                       (const uint16_t*)y2, y_rows, ldy, pos, weights, tokens, (int)top_k, cols,
                       (uint16_t*)out, ldo);
  };
  // As many rows together as leave fewest places empty in rounds of up to eight (of two matrices, four): a
  // place without a choice reads row 0 for nothing.  16384 tokens x 2048 with y2, 1 choice 36.2 us in rounds of
  // one, 56.6 of four; 9 choices unweighted 122 us in two rounds of five, 143 of eight.
  const int choices = top_k < 1 ? 1 : (int)top_k, most = y2 ? 4 : 8;
  const int rounds = (choices + most - 1) / most, unroll = (choices + rounds - 1) / rounds;
  auto pick = [&](auto two) {
    constexpr bool TWO = decltype(two)::value;
    if (unroll == 1) launch(moe_combine_kernel<1, TWO>);
    else if (unroll == 2) launch(moe_combine_kernel<2, TWO>);
    else if (unroll == 3) launch(moe_combine_kernel<3, TWO>);
    else if (unroll == 4) launch(moe_combine_kernel<4, TWO>);
    else if constexpr (!TWO) {
      if (unroll == 5) launch(moe_combine_kernel<5, false>);
      else if (unroll == 6) launch(moe_combine_kernel<6, false>);
      else if (unroll == 7) launch(moe_combine_kernel<7, false>);
      else launch(moe_combine_kernel<8, false>);
    }
  };
  if (y2) pick(std::true_type{});
  else pick(std::false_type{});
  return hipGetLastError() == hipSuccess ? MX_OK : MX_ERR_LAUNCH;
}

extern "C" int mx_moe_combine_dot(const void* y, int64_t y_rows, int64_t ldy, const int64_t* pos,
                                  const float* weights, const void* x, int64_t ldx, int64_t tokens,
                                  int64_t top_k, int64_t cols, void* out, int64_t ldo, float* dots,
                                  void* stream) {
  if (y_rows < 0 || tokens < 0 || top_k < 1 || top_k > 16 || cols < 0 || ldy < cols || ldx < cols ||
      (out && ldo < cols) || tokens > ((int64_t)1 << 32))
    return MX_ERR_INVALID_ARG;
  if (tokens == 0) return MX_OK;
  if (!dots || !pos || (cols > 0 && ((!y && y_rows > 0) || !x))) return MX_ERR_INVALID_ARG;
  if (cols % 8 || ldy % 8 || ldx % 8 || (out && ldo % 8) || ((uintptr_t)y & 15) || ((uintptr_t)x & 15) ||
      ((uintptr_t)out & 15) || ((uintptr_t)pos & 7) || ((uintptr_t)weights & 3) || ((uintptr_t)dots & 3))
    return MX_ERR_ALIGNMENT;
  const dim3 grid((unsigned)((tokens + kMoeThreads / 64 - 1) / (kMoeThreads / 64)));
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kMoeThreads), 0, (hipStream_t)stream, (const uint16_t*)y,
                       y_rows, ldy, pos, weights, (const uint16_t*)x, ldx, tokens, (int)top_k, cols,
                       (uint16_t*)out, ldo, dots);
  };
  auto pick = [&](auto with_out) {
    constexpr bool OUT = decltype(with_out)::value;
    if (top_k <= 1)
      launch(moe_combine_dot_kernel<1, OUT>);
    else if (top_k <= 2)
      launch(moe_combine_dot_kernel<2, OUT>);
    else if (top_k <= 4)
      launch(moe_combine_dot_kernel<4, OUT>);
    else if (top_k <= 8)
      launch(moe_combine_dot_kernel<8, OUT>);
    else
      launch(moe_combine_dot_kernel<16, OUT>);
  };
  if (out)
    pick(std::true_type{});
  else
    pick(std::false_type{});
  return hipGetLastError() == hipSuccess ? MX_OK : MX_ERR_LAUNCH;
}

extern "C" int mx_moe_row_dot(const void* a, const void* a2, int64_t a_rows, int64_t lda,
                              const int64_t* ia,
                              const void* b, int64_t b_rows, int64_t ldb, const int64_t* ib,
                              int64_t n, int64_t cols, float* out, void* stream) {
  if (a_rows < 0 || b_rows < 0 || n < 0 || cols < 0 || lda < cols || ldb < cols)
    return MX_ERR_INVALID_ARG;
  if (n == 0) return MX_OK;
  if (!a || !b || !ia || !ib || !out) return MX_ERR_INVALID_ARG;
  if (cols % 8 || lda % 8 || ldb % 8 || ((uintptr_t)a & 15) || ((uintptr_t)a2 & 15) ||
      ((uintptr_t)b & 15) ||
      ((uintptr_t)ia & 7) || ((uintptr_t)ib & 7) || ((uintptr_t)out & 3))
    return MX_ERR_ALIGNMENT;
  hipLaunchKernelGGL(moe_row_dot_kernel, dim3(moe_grid(n * 64)), dim3(kMoeThreads), 0,
                     (hipStream_t)stream, (const uint16_t*)a, (const uint16_t*)a2, a_rows, lda, ia,
                     (const uint16_t*)b,
                     b_rows, ldb, ib, n, cols, out);
  return hipGetLastError() == hipSuccess ? MX_OK : MX_ERR_LAUNCH;
}
