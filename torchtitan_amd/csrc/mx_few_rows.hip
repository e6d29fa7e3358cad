// Products of a few rows: D[M, N] = mx(x)[M, K] * deq(W)[N, K]^T for M <= 64 (a generator's or an evaluation's
// handful of tokens), x cast already or, up to 32 rows, in bf16 and cast on the way in.
//
// Bound by latency: a weight's bytes take 2 us of HBM time (2048 x 6144), but 128 x 128 tiles make 48
// workgroups of them, each walking the whole contraction with two steps in flight.  Here a workgroup
// takes 16 to 64 columns of the output and its eight waves take turns along the contraction, fragments
// straight from memory into registers (a workgroup reads nothing twice, LDS has nothing to share), the next
// step's on their way while one is multiplied; the eight partial sums meet in LDS.  Codes of 16 / 64
// rows, us, 128 x 128 tiles and now: 2048 x 6144 13.1 / 14.3, 6.6 / 9.7; 4096 x 4096 23.5 / 24.4, 7.3 / 13.1;
// 14336 x 4096 83 / 84, 20 / 39.  bf16 rows are cast in registers, with the codes and scales of the
// casts, and save the launch in front: 16 rows 9.6, 10.7 and 26 us.
#include "mx_gemm_tile.h"

namespace mx {

constexpr int kFewWaves = 8;
constexpr int64_t kFewRowsMax = 32;  // of bf16: every workgroup casts them anew

struct FewArgs {
  const void* x;            // bf16 [M, K] or codes [M, K up to 128]
  const uint8_t* x_scales;  // codes: MFMA order
  const uint8_t *w[2], *w_scales[2];
  uint16_t* d[2];
  int64_t M, N, K, ldx, ldw, ldd;  // ldx in elements of x
};

// 16 values of a block's half into codes.
template <int MODE>
__device__ __forceinline__ v4i few_codes(const u32x4 (&v)[2], uint32_t sb) {
  const uint32_t w[8] = {v[0].x, v[0].y, v[0].z, v[0].w, v[1].x, v[1].y, v[1].z, v[1].w};
  v4i out;
  if (sb != 255) {
    const float mult = scale_multiplier<MODE>(sb);
#pragma unroll
    for (int d = 0; d < 4; ++d) out[d] = (int)cvt2<true>(w[2 * d + 1], mult, cvt2<false>(w[2 * d], mult, 0));
  } else {
#pragma unroll
    for (int d = 0; d < 4; ++d) out[d] = (int)(nan_block_codes2(w[2 * d]) | (nan_block_codes2(w[2 * d + 1]) << 16));
  }
  return out;
}

__device__ __forceinline__ uint32_t few_amax(const u32x4 (&v)[2]) {
  uint32_t m = 0;
#pragma unroll
  for (int h = 0; h < 2; ++h)
    m = pk_max_u16(m, pk_max_u16(pk_max_u16(v[h].x & 0x7FFF7FFFu, v[h].y & 0x7FFF7FFFu),
                                 pk_max_u16(v[h].z & 0x7FFF7FFFu, v[h].w & 0x7FFF7FFFu)));
  return max(m & 0xFFFFu, m >> 16);
}

template <int MODE, int MT, int NT, bool CODES>
__global__ __launch_bounds__(64 * kFewWaves) void few_rows_kernel(FewArgs p) {
  __shared__ v4f sums[kFewWaves][MT * NT][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, lj = lane >> 4;
  const int64_t n0 = (int64_t)blockIdx.x * (16 * NT);
  const int which = blockIdx.y;
  const int steps = (int)((p.K + 127) / 128);
  // MFMA-order scale of (row 16 m + li of a 128-row group, block lj of step s): byte m / 2 of a dword
  auto scale_at = [&](int m) { return ((lj & 1) * 32 + 16 * (m & 1) + li) * 4 + (m >> 1) + (lj >> 1) * 256; };
  // the lane's share of a 128-deep step: bytes 16 lj .. + 15 and 64 + 16 lj .. + 15 of its row
  const uint8_t *wr[NT], *ws[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int64_t row = min(n0 + 16 * n + li, p.N - 1), tile = min(n0 + 16 * n, (p.N - 1) & ~(int64_t)15);
    wr[n] = p.w[which] + row * p.ldw + 16 * lj;
    ws[n] = p.w_scales[which] + (((tile >> 7) * steps * 2) << 8) + scale_at((int)(tile & 127) >> 4);
  }

  struct Step {
    v4i w[NT][2];
    uint32_t ws[NT], xs[MT];
    u32x4 x[MT][CODES ? 1 : 2][2];  // [row tile][half][16 bytes]; codes: both halves in [0]
  };
  auto load = [&](int s, Step& r) {
    const int64_t k = (int64_t)s * 128;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      r.w[n][0] = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(wr[n] + k));
      r.w[n][1] = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(wr[n] + k + 64));
      r.ws[n] = ws[n][(int64_t)s * 512];
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int64_t t = 16 * m + li < p.M ? 16 * m + li : p.M - 1;  // rows beyond are not stored
      if constexpr (CODES) {
        const uint8_t* xr = (const uint8_t*)p.x + t * p.ldx + k + 16 * lj;
        r.x[m][0][0] = *reinterpret_cast<const u32x4*>(xr);
        r.x[m][0][1] = *reinterpret_cast<const u32x4*>(xr + 64);
        r.xs[m] = p.x_scales[(int64_t)s * 512 + scale_at(m)];
      } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int64_t c = k + 64 * h + 16 * lj;
          const uint16_t* xr = (const uint16_t*)p.x + t * p.ldx + c;
          r.x[m][h][0] = r.x[m][h][1] = u32x4{0, 0, 0, 0};
          if (c < p.K) {  // K is a multiple of 32: all 16 values or none
            r.x[m][h][0] = *reinterpret_cast<const u32x4*>(xr);
            r.x[m][h][1] = *reinterpret_cast<const u32x4*>(xr + 8);
          }
        }
      }
    }
  };
  v4f acc[MT * NT];
#pragma unroll
  for (int m = 0; m < MT * NT; ++m) acc[m] = v4f{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const Step& r) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      v4i lo, hi;
      uint32_t sc;
      if constexpr (CODES) {
        lo = __builtin_bit_cast(v4i, r.x[m][0][0]);
        hi = __builtin_bit_cast(v4i, r.x[m][0][1]);
        sc = r.xs[m];
      } else {
        // blocks 0 and 2 lie in lanes lj = 0, 1 (first and second half), blocks 1 and 3 in lj = 2, 3;
        // the instruction takes the scale of block b from lane group b
        uint32_t top = few_amax(r.x[m][0]) | (few_amax(r.x[m][1]) << 16);
        top = pk_max_u16(top, (uint32_t)__shfl_xor((int)top, 16));
        const uint32_t s0 = scale_byte<MODE>(top & 0xFFFFu), s1 = scale_byte<MODE>(top >> 16);
        lo = few_codes<MODE>(r.x[m][0], s0);
        hi = few_codes<MODE>(r.x[m][1], s1);
        const uint32_t other = (uint32_t)__shfl_xor((int)(lj == 1 ? s1 : s0), 48);
        sc = lj == 0 ? s0 : lj == 3 ? s1 : other;
      }
      const v8i xf = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const v8i wf = {r.w[n][0].x, r.w[n][0].y, r.w[n][0].z, r.w[n][0].w, r.w[n][1].x, r.w[n][1].y, r.w[n][1].z, r.w[n][1].w};
        acc[m * NT + n] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf, xf, acc[m * NT + n], 0, 0, 0, (int)r.ws[n],
                                                                           0, (int)sc);
      }
    }
  };
  Step now, next;
  if (wave < steps) load(wave, now);
  // (one copy of the step: a launch this short feels its instructions being fetched)
#pragma unroll 1
  for (int s = wave; s < steps; s += kFewWaves) {
    load(min(s + kFewWaves, steps - 1), next);
    multiply(now);
    now = next;
  }
#pragma unroll
  for (int q = 0; q < MT * NT; ++q) sums[wave][q][lane] = acc[q];
  __syncthreads();
  for (int q = wave; q < MT * NT; q += kFewWaves) {
    v4f s = sums[0][q][lane];
#pragma unroll
    for (int i = 1; i < kFewWaves; ++i) s += sums[i][q][lane];
    // the lane holds columns n0 + 16 n + 4 lj .. + 3 of row 16 m + li
    const int64_t r = 16 * (q / NT) + li, c = n0 + 16 * (q % NT) + 4 * lj;
    if (r >= p.M || c >= p.N) continue;
    uint16_t* dst = p.d[which] + r * p.ldd + c;
    const u32x2 out = {pack_bf16(s.x, s.y), pack_bf16(s.z, s.w)};
    if (c + 3 < p.N && ((uintptr_t)dst & 7) == 0) {
      *reinterpret_cast<u32x2*>(dst) = out;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (c + i < p.N) dst[i] = (uint16_t)(out[i >> 1] >> (16 * (i & 1)));
    }
  }
}

template <int MODE, int NT, bool CODES>
static int launch_few_nt(const FewArgs& p, int products, hipStream_t st) {
  const int64_t tiles = (p.N + 16 * NT - 1) / (16 * NT);
  if (tiles > 0x7FFFFFFF || (p.K + 127) / 128 > (1 << 20)) return MX_ERR_UNSUPPORTED;
  const dim3 grid((unsigned)tiles, (unsigned)products), block(64 * kFewWaves);
  if (p.M <= 16) hipLaunchKernelGGL((few_rows_kernel<MODE, 1, NT, CODES>), grid, block, 0, st, p);
  else if (p.M <= 32) hipLaunchKernelGGL((few_rows_kernel<MODE, 2, NT, CODES>), grid, block, 0, st, p);
  else if constexpr (!CODES) return MX_ERR_UNSUPPORTED;
  else hipLaunchKernelGGL((few_rows_kernel<MODE, 4, NT, CODES>), grid, block, 0, st, p);
  return hipGetLastError() == hipSuccess ? MX_OK : MX_ERR_LAUNCH;
}

// The fewest columns that leave no more workgroups than CUs: a second round costs more than wider workgroups, which
// read x less often, and narrower ones have the shorter chains.  us at 2048 deep (4096 deep moves alike) by columns
// per workgroup 16 / 32 / 64, from codes of 16 and of 64 rows, from 16 rows of bf16:
//    4096 columns    5.1 /  6.6 /  9.5     7.8 /  9.1 / 12.4     7.7 /  9.6 / 13.1
//    5120            7.3 /  6.6 /  9.6    12.9 /  9.4 / 12.7    11.9 /  9.7 / 13.3
//    8192            7.4 /  6.8 /  9.7    12.8 /  9.9 / 13.1    12.1 /  9.8 / 13.4
//   10240            9.6 / 10.2 /  9.8    18.4 / 16.3 / 13.2    16.2 / 16.0 / 13.6
//   16384           12.1 / 10.5 / 10.2    23.9 / 16.9 / 13.4    21.3 / 16.6 / 14.0
template <int MODE, bool CODES>
static int launch_few(const FewArgs& p, int products, hipStream_t st) {
  constexpr int64_t kCus = 256;
  const int64_t columns = p.N * products;
  if (columns <= 16 * kCus) return launch_few_nt<MODE, 1, CODES>(p, products, st);
  if (columns <= 32 * kCus) return launch_few_nt<MODE, 2, CODES>(p, products, st);
  return launch_few_nt<MODE, 4, CODES>(p, products, st);
}

// For mx_gemm_nt's dispatch: operands already checked, K and both pitches multiples of 128 and 16.
int launch_few_rows_codes(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                          const uint8_t* b_scales, void* d, int64_t M, int64_t N, int64_t K, int64_t ldk, int64_t ldd,
                          hipStream_t st) {
  const FewArgs p{a_codes, a_scales, {b_codes, nullptr}, {b_scales, nullptr}, {(uint16_t*)d, nullptr}, M, N, K, ldk, ldk, ldd};
  return launch_few<MX_SCALE_FLOOR, true>(p, 1, st);
}

}  // namespace mx

using namespace mx;

extern "C" int mx_few_rows(const void* x, int64_t M, int64_t K, int64_t ldx, const uint8_t* w_codes,
                           const uint8_t* w_scales, const uint8_t* w2_codes, const uint8_t* w2_scales, int64_t N,
                           int64_t ldw, void* d, void* d2, int64_t ldd, int scale_mode, void* stream) {
  if (M < 0 || N < 0 || K <= 0 || ldx < K || ldd < N || (scale_mode != MX_SCALE_FLOOR && scale_mode != MX_SCALE_RCEIL))
    return MX_ERR_INVALID_ARG;
  if (M > kFewRowsMax) return MX_ERR_UNSUPPORTED;
  if (M == 0 || N == 0) return MX_OK;
  if (!x || !w_codes || !w_scales || !d || !w2_codes != !w2_scales || !w2_codes != !d2) return MX_ERR_INVALID_ARG;
  if (ldw < (K + 127) / 128 * 128) return MX_ERR_INVALID_ARG;
  if (K % 32 || ldx % 8 || ldw % 16 || ((uintptr_t)x & 15) || ((uintptr_t)w_codes & 15) || ((uintptr_t)w2_codes & 15) ||
      ((uintptr_t)d & 1) || ((uintptr_t)d2 & 1))
    return MX_ERR_ALIGNMENT;
  const FewArgs p{x, nullptr, {w_codes, w2_codes}, {w_scales, w2_scales}, {(uint16_t*)d, (uint16_t*)d2}, M, N, K, ldx, ldw, ldd};
  const int products = w2_codes ? 2 : 1;
  return scale_mode == MX_SCALE_FLOOR ? launch_few<MX_SCALE_FLOOR, false>(p, products, (hipStream_t)stream)
                                      : launch_few<MX_SCALE_RCEIL, false>(p, products, (hipStream_t)stream);
}
