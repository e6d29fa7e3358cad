// The router's gate: logits = x W^T in float32 for bf16 x [tokens, dim] and W [experts, dim], and its
// backward.  The products are those of a float32 matmul: bf16 times bf16 is exact in float32, and a
// float32 operand (the logits' gradient) is cut into three bf16 parts that add up to it exactly.
//
// Few experts make these products reading x (and writing dx) once: 16384 tokens x 2048, 128 experts
// move 67 MB per pass, and the operations of the three-part products come to 10 us.  All operands are
// read straight into MFMA registers.  The order of the contraction is free and so is the assignment of
// rows and columns to a fragment's lanes, so a lane reads whole 16-byte pieces in any orientation:
// where the contraction runs along the rows of the stored matrix, eight rows of a piece are
// interleaved in registers into fragments for eight neighbouring columns.
//
// Measured at that size: logits 41 us, dx with the addition 41 us, weight gradient 36 us in two launches, where the
// float32 matmuls around conversions of x, W and dx and a separate addition took 75 + 98 + 141 + 100 us.
// With 8 experts 13, 25 and 26 us: the forward reads x at 5.4 TB/s, and what more experts add is W
// coming from the L2 for every 32 tokens and the three-part products.
#include <type_traits>

#include "mx_gemm_tile.h"

namespace mx {

int launch_splitk_reduce(const float* part, int slices, int64_t M, int64_t N, void* d, int64_t ldd, bool f32,
                         hipStream_t st);

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

constexpr int kGateMaxExperts = 128;
constexpr int kGateSlab = 128;  // columns of dim one wave of the backward works on

__device__ __forceinline__ v4f mfma_bf16(const u32x4& a, const u32x4& b, const v4f& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}

// Eight rows of an 8-column piece -> eight fragments, one per column, the rows along the contraction.
__device__ __forceinline__ void columns_of(const u32x4 (&rows)[8], u32x4 (&f)[8]) {
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      f[2 * q][p] = __builtin_amdgcn_perm(rows[2 * p + 1][q], rows[2 * p][q], 0x05040100u);
      f[2 * q + 1][p] = __builtin_amdgcn_perm(rows[2 * p + 1][q], rows[2 * p][q], 0x07060302u);
    }
}

// v = part[0] + part[1] + part[2], each of eight bits of mantissa: the upper half of v, of what is left
// and of what is left then.  An infinite v has no rest.
__device__ __forceinline__ void three_parts(const float (&v)[8], u32x4 (&part)[3]) {
  float a[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) a[e] = v[e];
#pragma unroll
  for (int s = 0; s < 3; ++s) {
#pragma unroll
    for (int p = 0; p < 4; ++p)
      part[s][p] = __builtin_amdgcn_perm(__float_as_uint(a[2 * p + 1]), __float_as_uint(a[2 * p]), 0x07060302u);
    if (s == 2) break;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float rest = a[e] - __uint_as_float(__float_as_uint(a[e]) & 0xFFFF0000u);
      a[e] = s == 0 && __builtin_amdgcn_classf(a[e], 0x204) ? 0.f : rest;
    }
  }
}

// logits[t, e] = <x[t], w[e]>.  A workgroup takes 16 MT tokens and all (up to 16 NT) experts; its four
// waves take turns along dim, 64 elements at a time (a row's 128-byte line), and add
// up through LDS at the end: four times shorter chains, which is what counts for few tokens, and W
// read once per 16 MT tokens from the L2.
// Per wave: the next step's x and the next half step's W are in flight while one is multiplied.
//
// SEGS > 1: the contraction in that many equal parts with a sum of its own each; workgroups begin with
// different parts, and the sums are added in one order, so that a token's logits do not depend on where it
// stands.
template <int MT, int NT, int SEGS>
__global__ __launch_bounds__(256, 2) void gate_fwd_kernel(const uint16_t* __restrict__ x, int64_t ldx,
                                                          const uint16_t* __restrict__ w, int64_t ldw,
                                                          int64_t tokens, int experts, int dim,
                                                          float* __restrict__ logits) {
  __shared__ v4f sums[SEGS][4][MT * NT][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, j = lane >> 4;
  const int64_t t0 = (int64_t)blockIdx.x * 16 * MT;
  const uint16_t *xr[MT], *wr[NT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int64_t t = t0 + 16 * m + i;
    xr[m] = x + (t < tokens ? t : tokens - 1) * ldx + 8 * j;
  }
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int e = 16 * n + i;
    wr[n] = w + (e < experts ? e : experts - 1) * ldw + 8 * j;
  }
  v4f acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = v4f{0.f, 0.f, 0.f, 0.f};
  const int steps = dim / 64, per = steps / SEGS;  // (SEGS > 1: per is a multiple of 8)
  int seg = SEGS > 1 ? (int)((blockIdx.x >> 3) % SEGS) : 0;
  const int turn = seg * per;
  auto at = [&](int s) { return 64 * (s + turn < steps ? s + turn : s + turn - steps); };
  u32x4 xa[2][MT], xb[2][MT], w0[NT], w1[NT];
  auto load_x = [&](int k, u32x4 (&xp)[2][MT]) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int m = 0; m < MT; ++m) xp[h][m] = *reinterpret_cast<const u32x4*>(xr[m] + k + 32 * h);
  };
  auto load_w = [&](int k, u32x4 (&wp)[NT]) {
#pragma unroll
    for (int n = 0; n < NT; ++n) wp[n] = *reinterpret_cast<const u32x4*>(wr[n] + k);
  };
  auto multiply = [&](const u32x4 (&xp)[MT], const u32x4 (&wp)[NT]) {
    __builtin_amdgcn_sched_barrier(0);  // the loads above stay above
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[m][n] = mfma_bf16(wp[n], xp[m], acc[m][n]);
    __builtin_amdgcn_sched_barrier(0);
  };
  // one 64-deep step out of xp, the next one's x on its way into xn
  auto step = [&](int s, const u32x4 (&xp)[2][MT], u32x4 (&xn)[2][MT]) {
    const int k = at(s), kn = at(s + 4 < steps ? s + 4 : s);
    load_w(k + 32, w1);
    load_x(kn, xn);
    multiply(xp[0], w0);
    load_w(kn, w0);
    multiply(xp[1], w1);
  };
  if (wave < steps) {
    load_x(at(wave), xa);
    load_w(at(wave), w0);
  }
  auto keep = [&]() {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        sums[seg][wave][m * NT + n][lane] = acc[m][n];
        acc[m][n] = v4f{0.f, 0.f, 0.f, 0.f};
      }
    seg = seg + 1 < SEGS ? seg + 1 : 0;
  };
  for (int s = wave, left = per; s < steps; s += 8) {
    step(s, xa, xb);
    if (s + 4 < steps) step(s + 4, xb, xa);
    if (SEGS > 1 && (left -= 8) == 0) {
      keep();
      left = per;
    }
  }
  if (SEGS == 1) keep();
  __syncthreads();
  // a lane holds experts 16n + 4j .. + 3 of token 16m + i
  for (int q = wave; q < MT * NT; q += 4) {
    v4f s = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < SEGS; ++g) {
      const v4f a = sums[g][0][q][lane], b = sums[g][1][q][lane], c = sums[g][2][q][lane], d = sums[g][3][q][lane];
      s = g == 0 ? (a + b) + (c + d) : s + ((a + b) + (c + d));
    }
    const int64_t t = t0 + 16 * (q / NT) + i;
    const int e = 16 * (q % NT) + 4 * j;
    if (t < tokens && e < experts) *reinterpret_cast<v4f*>(logits + t * experts + e) = s;
  }
}

// out[t, d] = bf16(sum_e g[t, e] w[e, d]), added to base[t, d] as a bf16 tensor addition forms it (base may be
// null).  A wave keeps the fragments of
// 128 columns of W for all experts (32 KS of them, zeros behind the last) and walks over 16-token tiles:
// W is read once per walk, g by every wave of columns (from the L2), base and out once.
template <int KS>
__global__ __launch_bounds__(256, 2) void gate_dx_kernel(const float* __restrict__ g, const uint16_t* __restrict__ w,
                                                         int64_t ldw, const uint16_t* __restrict__ base, int64_t ldb,
                                                         int64_t tokens, int experts, int dim, int tiles,
                                                         uint16_t* __restrict__ out) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, j = lane >> 4;
  const int d0 = (blockIdx.y * 4 + wave) * kGateSlab;
  if (d0 >= dim) return;
  // wf[.][f]: row i of the fragment is column d0 + 8 (4 (i % 4) + i / 4) + f, so that a lane's results of one
  // r are eight neighbouring columns, next to those of the other three lanes of its token
  const int piece = 4 * (i & 3) + (i >> 2);
  u32x4 wf[KS][8];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    u32x4 rows[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) rows[r] = u32x4{0, 0, 0, 0};
    const int e = 32 * ks + 8 * j;
    if (e < experts) {
#pragma unroll
      for (int r = 0; r < 8; ++r) rows[r] = *reinterpret_cast<const u32x4*>(w + (int64_t)(e + r) * ldw + d0 + 8 * piece);
    }
    columns_of(rows, wf[ks]);
  }
  for (int n = 0; n < tiles; ++n) {
    const int64_t t0 = ((int64_t)blockIdx.x * tiles + n) * 16;
    if (t0 >= tokens) break;
    const int64_t t = t0 + i, tc = t < tokens ? t : tokens - 1;
    v4f gv[KS][2];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int e = 32 * ks + 8 * j;
      gv[ks][0] = gv[ks][1] = v4f{0.f, 0.f, 0.f, 0.f};
      if (e < experts) {
        const v4f* p = reinterpret_cast<const v4f*>(g + tc * experts + e);
        gv[ks][0] = p[0];
        gv[ks][1] = p[1];
      }
    }
    v4f acc[8];
#pragma unroll
    for (int f = 0; f < 8; ++f) acc[f] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const float v[8] = {gv[ks][0].x, gv[ks][0].y, gv[ks][0].z, gv[ks][0].w,
                          gv[ks][1].x, gv[ks][1].y, gv[ks][1].z, gv[ks][1].w};
      u32x4 part[3];
      three_parts(v, part);
#pragma unroll
      for (int s = 2; s >= 0; --s)
#pragma unroll
        for (int f = 0; f < 8; ++f) acc[f] = mfma_bf16(wf[ks][f], part[s], acc[f]);
    }
    if (t < tokens) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = d0 + 8 * (4 * r + j);
        u32x4 o;
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = pack_bf16(acc[2 * q][r], acc[2 * q + 1][r]);
        if (base) {
          const u32x4 b = *reinterpret_cast<const u32x4*>(base + t * ldb + d);
#pragma unroll
          for (int q = 0; q < 4; ++q)
            o[q] = pack_bf16(__uint_as_float(o[q] << 16) + __uint_as_float(b[q] << 16),
                             __uint_as_float(o[q] & 0xFFFF0000u) + __uint_as_float(b[q] & 0xFFFF0000u));
        }
        *reinterpret_cast<u32x4*>(out + t * dim + d) = o;
      }
    }
  }
}

// part[z][e, d] = sum of g[t, e] x[t, d] over the tokens of slice z (a second launch adds the slices).  A wave
// takes 16 EF experts x 128 columns over `steps` 32-token steps, the four waves of a workgroup follow
// one another along the tokens and add up through LDS.
template <int EF>
__global__ __launch_bounds__(256, 2) void gate_dw_kernel(const float* __restrict__ g, const uint16_t* __restrict__ x,
                                                         int64_t ldx, int64_t tokens, int experts, int dim, int steps,
                                                         float* __restrict__ part) {
  __shared__ v4f sums[4][EF * 8][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, j = lane >> 4;
  const int e0 = blockIdx.y * 16 * EF + EF * i, d0 = blockIdx.x * kGateSlab;  // the lane's first expert
  const bool has_e = e0 < experts;
  const int64_t all = (tokens + 31) / 32, first = ((int64_t)blockIdx.z * 4 + wave) * steps;
  const int64_t last = first + steps < all ? first + steps : all;
  v4f acc[EF][8];
#pragma unroll
  for (int q = 0; q < EF; ++q)
#pragma unroll
    for (int f = 0; f < 8; ++f) acc[q][f] = v4f{0.f, 0.f, 0.f, 0.f};
  u32x4 xa[8], xb[8];
  float ga[8][EF], gb[8][EF];
  const bool whole_e = (int)(blockIdx.y + 1) * 16 * EF <= experts;
  auto load = [&](int64_t s, u32x4 (&xp)[8], float (&gp)[8][EF]) {
    if (whole_e && 32 * s + 32 <= tokens) {
      const uint16_t* xq = x + (32 * s + 8 * j) * ldx + d0 + 8 * i;
      const float* q = g + (32 * s + 8 * j) * experts + e0;
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        xp[r] = *reinterpret_cast<const u32x4*>(xq + r * ldx);
#pragma unroll
        for (int e = 0; e < EF; ++e) gp[r][e] = q[r * experts + e];
      }
      return;
    }
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int64_t t = 32 * s + 8 * j + r;
      const bool in = t < tokens;
      const int64_t tc = in ? t : tokens - 1;
      xp[r] = *reinterpret_cast<const u32x4*>(x + tc * ldx + d0 + 8 * i);
      const float* q = g + tc * experts + (has_e ? e0 : 0);
#pragma unroll
      for (int e = 0; e < EF; ++e) gp[r][e] = q[e];
      if (!in) xp[r] = u32x4{0, 0, 0, 0};
#pragma unroll
      for (int e = 0; e < EF; ++e) gp[r][e] = in && has_e ? gp[r][e] : 0.f;
    }
  };
  auto multiply = [&](const u32x4 (&xp)[8], const float (&gp)[8][EF]) {
    __builtin_amdgcn_sched_barrier(0);  // the loads above stay above
    u32x4 xf[8];
    columns_of(xp, xf);
#pragma unroll
    for (int e = 0; e < EF; ++e) {
      const float v[8] = {gp[0][e], gp[1][e], gp[2][e], gp[3][e], gp[4][e], gp[5][e], gp[6][e], gp[7][e]};
      u32x4 parts[3];
      three_parts(v, parts);
#pragma unroll
      for (int q = 2; q >= 0; --q)
#pragma unroll
        for (int f = 0; f < 8; ++f) acc[e][f] = mfma_bf16(parts[q], xf[f], acc[e][f]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  if (first < last) load(first, xa, ga);
  for (int64_t s = first; s < last; s += 2) {
    load(s + 1 < last ? s + 1 : s, xb, gb);
    multiply(xa, ga);
    if (s + 1 >= last) break;
    load(s + 2 < last ? s + 2 : s, xa, ga);
    multiply(xb, gb);
  }
  // a lane holds, in acc[e][f][r], expert EF (4j + r) + e of the block's and column d0 + 8i + f
  float* dst = part + (int64_t)blockIdx.z * experts * dim;
#pragma unroll
  for (int e = 0; e < EF; ++e)
#pragma unroll
    for (int f = 0; f < 8; ++f) sums[wave][e * 8 + f][lane] = acc[e][f];
  __syncthreads();
  for (int q = wave; q < 4 * EF; q += 4) {
    const int e = q / 4, r = q % 4, row = blockIdx.y * 16 * EF + EF * (4 * j + r) + e;
    float v[8];
#pragma unroll
    for (int f = 0; f < 8; ++f) {
      auto at = [&](int s) { return reinterpret_cast<const float*>(&sums[s][e * 8 + f][lane])[r]; };
      v[f] = (at(0) + at(1)) + (at(2) + at(3));
    }
    if (row < experts) {
      v4f* o = reinterpret_cast<v4f*>(dst + (int64_t)row * dim + d0 + 8 * i);
      o[0] = v4f{v[0], v[1], v[2], v[3]};
      o[1] = v4f{v[4], v[5], v[6], v[7]};
    }
  }
}

static bool gate_shape_ok(int64_t tokens, int64_t experts, int64_t dim) {
  return tokens >= 0 && tokens < ((int64_t)1 << 31) && experts >= 8 && experts <= kGateMaxExperts && experts % 8 == 0 &&
         dim >= kGateSlab && dim % kGateSlab == 0 && dim < ((int64_t)1 << 24);
}

// Experts per wave of the weight gradient, in 16s, and token slices (workgroups of four waves): two waves
// per SIMD of the chip where there are tokens for it.
static int gate_dw_frags(int64_t experts) { return experts <= 16 ? 1 : 2; }
static int64_t gate_dw_slices(int64_t tokens, int64_t experts, int64_t dim) {
  const int64_t tile = 16 * gate_dw_frags(experts), tiles = (dim / kGateSlab) * ((experts + tile - 1) / tile);
  const int64_t steps = (tokens + 31) / 32, most = (steps + 3) / 4;
  int64_t z = 512 / tiles;
  z = z < 1 ? 1 : z;
  return z < most ? z : (most < 1 ? 1 : most);
}

}  // namespace mx

using namespace mx;

extern "C" int mx_gate_logits(const void* x, int64_t ldx, const void* w, int64_t ldw, int64_t tokens, int64_t experts,
                              int64_t dim, float* logits, void* stream) {
  if (!gate_shape_ok(tokens, experts, dim) || ldx < dim || ldw < dim) return MX_ERR_INVALID_ARG;
  if (tokens == 0) return MX_OK;
  if (!x || !w || !logits) return MX_ERR_INVALID_ARG;
  if (ldx % 8 || ldw % 8 || ((uintptr_t)x & 15) || ((uintptr_t)w & 15) || ((uintptr_t)logits & 15)) return MX_ERR_ALIGNMENT;
  auto launch = [&](auto kernel, int mt) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)((tokens + 16 * mt - 1) / (16 * mt))), dim3(256), 0, (hipStream_t)stream,
                       (const uint16_t*)x, ldx, (const uint16_t*)w, ldw, tokens, (int)experts, (int)dim, logits);
  };
  // 32 tokens per workgroup halve the reads of W; 16 while that leaves CUs without work.  Rows a multiple of
  // 4 KB apart lie on the same channels of the L2: there half of the workgroups begin with the second half
  // of the contraction.  16384 x 4096, us, in order / in halves: 8 experts 35.2 / 22.1, 32 38.8 / 31.5,
  // 64 51.3 / 46.3; 128 76.9 / 76.9 and at 2048 41.5 / 42.5 (W's reads count for more, and a CU has room for one
  // workgroup with twice the sums), so in order.
  const bool halves = dim % 2048 == 0, few = tokens <= 16 * 256;
  auto pick = [&](auto nt) {
    constexpr int NT = decltype(nt)::value;
    if constexpr (NT <= 4) {
      if (halves) return few ? launch(gate_fwd_kernel<1, NT, 2>, 1) : launch(gate_fwd_kernel<2, NT, 2>, 2);
    }
    few ? launch(gate_fwd_kernel<1, NT, 1>, 1) : launch(gate_fwd_kernel<2, NT, 1>, 2);
  };
  if (experts <= 16) pick(std::integral_constant<int, 1>{});
  else if (experts <= 32) pick(std::integral_constant<int, 2>{});
  else if (experts <= 64) pick(std::integral_constant<int, 4>{});
  else pick(std::integral_constant<int, 8>{});
  return hipGetLastError() == hipSuccess ? MX_OK : MX_ERR_LAUNCH;
}

extern "C" int mx_gate_dx(const float* g, const void* w, int64_t ldw, const void* base, int64_t ldb, int64_t tokens,
                          int64_t experts, int64_t dim, void* out, void* stream) {
  if (!gate_shape_ok(tokens, experts, dim) || ldw < dim || (base && ldb < dim)) return MX_ERR_INVALID_ARG;
  if (tokens == 0) return MX_OK;
  if (!g || !w || !out) return MX_ERR_INVALID_ARG;
  if (ldw % 8 || (base && ldb % 8) || ((uintptr_t)g & 15) || ((uintptr_t)w & 15) || ((uintptr_t)base & 15) ||
      ((uintptr_t)out & 15))
    return MX_ERR_ALIGNMENT;
  const int64_t tiles = (tokens + 15) / 16, slabs = dim / kGateSlab;
  int64_t per_wave = tiles * slabs / 2048;  // two waves per SIMD, as the registers allow
  per_wave = per_wave < 1 ? 1 : (per_wave > 16 ? 16 : per_wave);
  const dim3 grid((unsigned)((tiles + per_wave - 1) / per_wave), (unsigned)((slabs + 3) / 4));
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, (hipStream_t)stream, g, (const uint16_t*)w, ldw,
                       (const uint16_t*)base, ldb, tokens, (int)experts, (int)dim, (int)per_wave, (uint16_t*)out);
  };
  if (experts <= 32) launch(gate_dx_kernel<1>);
  else if (experts <= 64) launch(gate_dx_kernel<2>);
  else launch(gate_dx_kernel<4>);
  return hipGetLastError() == hipSuccess ? MX_OK : MX_ERR_LAUNCH;
}

extern "C" int64_t mx_gate_dw_workspace(int64_t tokens, int64_t experts, int64_t dim) {
  return gate_shape_ok(tokens, experts, dim) ? gate_dw_slices(tokens, experts, dim) * experts * dim * 4 : 0;
}

extern "C" int mx_gate_dw(const float* g, const void* x, int64_t ldx, int64_t tokens, int64_t experts, int64_t dim,
                          void* workspace, void* dw, void* stream) {
  if (!gate_shape_ok(tokens, experts, dim) || tokens == 0 || ldx < dim) return MX_ERR_INVALID_ARG;
  if (!g || !x || !workspace || !dw) return MX_ERR_INVALID_ARG;
  if (ldx % 8 || ((uintptr_t)g & 15) || ((uintptr_t)x & 15) || ((uintptr_t)workspace & 15) || ((uintptr_t)dw & 15))
    return MX_ERR_ALIGNMENT;
  const int frags = gate_dw_frags(experts);
  const int64_t slices = gate_dw_slices(tokens, experts, dim), steps = ((tokens + 31) / 32 + 4 * slices - 1) / (4 * slices);
  const dim3 grid((unsigned)(dim / kGateSlab), (unsigned)((experts + 16 * frags - 1) / (16 * frags)), (unsigned)slices);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, (hipStream_t)stream, g, (const uint16_t*)x, ldx, tokens, (int)experts,
                       (int)dim, (int)steps, (float*)workspace);
  };
  if (frags == 1) launch(gate_dw_kernel<1>);
  else launch(gate_dw_kernel<2>);
  if (hipGetLastError() != hipSuccess) return MX_ERR_LAUNCH;
  return launch_splitk_reduce((const float*)workspace, (int)slices, experts, dim, dw, dim, false, (hipStream_t)stream);
}
