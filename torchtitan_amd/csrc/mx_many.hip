// Row-wise cast and dequantization of a list of tensors in one launch: what a trainer hands to a
// generator is every converted weight of the model, and a layer's seven weights are 2 to 25 MB each --
// launches of 5 us whose first and last waves leave most of the chip idle.  Scales are row-major, so
// with dense rows of whole 32-element blocks a tensor is one flat run of blocks whatever its shape.
// HBM-bound: 3.03 bytes per element to cast (5.03 from float32), 3.03 to dequantize.
// The seven weights of a 2048 / 6144 layer (44 M elements): casts and scale re-layout 55 + 22 us in
// fourteen launches and dequantization 52 us in seven before, 28.4 and 29.1 us in one launch each
// (4.7 and 4.6 TB/s; 41 us with 16 codes per lane, whose two 16-byte stores each fill half lines).
#include "mx_common.h"

namespace mx {

constexpr int kManyThreads = 256;
constexpr int kManyUnroll = 4;      // pieces of 8 elements per lane
constexpr int kManyTensors = 48;    // of one launch (the table travels as a kernel argument)

struct ManyEntry {
  const void* src;   // cast: bf16 or float32 values; dequantization: codes
  uint8_t* codes;    // cast: codes out
  uint8_t* scales;   // cast: scales out; dequantization: scales in
  uint16_t* out;     // dequantization: bf16 out
  int64_t pieces;    // of 8 elements
  uint32_t first;    // first workgroup of this tensor
  uint32_t f32;      // cast: the values are float32
};
struct ManyTable {
  ManyEntry e[kManyTensors];
};

__device__ __forceinline__ int many_find(const ManyTable& t, int n) {
  int lo = 0, hi = n;  // the last entry whose first workgroup is not behind this one
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (t.e[mid].first <= blockIdx.x) lo = mid; else hi = mid;
  }
  return lo;
}

// float32 -> bf16 bits as a tensor conversion rounds: to nearest even, any NaN to the one quiet NaN.
__device__ __forceinline__ uint32_t many_bf16(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7FFFFFFFu) > 0x7F800000u) return 0x7FC0u;
  return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

template <int MODE>
__global__ __launch_bounds__(kManyThreads) void cast_rows_many_kernel(ManyTable table, int n) {
  const ManyEntry q = table.e[many_find(table, n)];
  const int64_t base = (int64_t)(blockIdx.x - q.first) * (kManyThreads * kManyUnroll) + threadIdx.x;
  u32x4 v[kManyUnroll];
#pragma unroll
  for (int k = 0; k < kManyUnroll; ++k) {
    const int64_t c = base + (int64_t)k * kManyThreads;
    v[k] = u32x4{0, 0, 0, 0};
    if (c < q.pieces) {
      if (q.f32) {
        const u32x4* p = reinterpret_cast<const u32x4*>(q.src) + c * 2;
        const u32x4 a = __builtin_nontemporal_load(p), b = __builtin_nontemporal_load(p + 1);
        auto two = [](uint32_t lo, uint32_t hi) {
          return many_bf16(__uint_as_float(lo)) | (many_bf16(__uint_as_float(hi)) << 16);
        };
        v[k] = u32x4{two(a.x, a.y), two(a.z, a.w), two(b.x, b.y), two(b.z, b.w)};
      } else {
        v[k] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(q.src) + c);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < kManyUnroll; ++k) {
    const int64_t c = base + (int64_t)k * kManyThreads;
    const u32x4 w = v[k];
    uint32_t m = pk_max_u16(pk_max_u16(w.x & 0x7FFF7FFFu, w.y & 0x7FFF7FFFu),
                            pk_max_u16(w.z & 0x7FFF7FFFu, w.w & 0x7FFF7FFFu));
    m = max(m & 0xFFFFu, m >> 16);
    m = max(m, dpp<kQuadXor1>(m));  // a block of 32 is the four pieces of a quad
    m = max(m, dpp<kQuadXor2>(m));
    const uint32_t sb = scale_byte<MODE>(m);
    const float mult = scale_multiplier<MODE>(sb);
    u32x2 out;
    if (sb != 255) {
      out.x = cvt2<true>(w.y, mult, cvt2<false>(w.x, mult, 0));
      out.y = cvt2<true>(w.w, mult, cvt2<false>(w.z, mult, 0));
    } else {
      out.x = nan_block_codes2(w.x) | (nan_block_codes2(w.y) << 16);
      out.y = nan_block_codes2(w.z) | (nan_block_codes2(w.w) << 16);
    }
    if (c < q.pieces) {
      __builtin_nontemporal_store(out, reinterpret_cast<u32x2*>(q.codes) + c);
      if ((threadIdx.x & 3) == 0) q.scales[c >> 2] = (uint8_t)sb;
    }
  }
}

// bf16 bits of code * 2^(scale byte - 127); exact except below bf16's normal range.
__device__ __forceinline__ uint32_t many_value(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (u >> 16) | 0x40u;
  return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

// (8 codes per lane and piece: the 16-byte stores of a wave are then one contiguous kilobyte)
__global__ __launch_bounds__(kManyThreads) void dequant_many_kernel(ManyTable table, int n) {
  const ManyEntry q = table.e[many_find(table, n)];
  const int64_t base = (int64_t)(blockIdx.x - q.first) * (kManyThreads * kManyUnroll) + threadIdx.x;
  u32x2 v[kManyUnroll];
  uint32_t sb[kManyUnroll];
#pragma unroll
  for (int k = 0; k < kManyUnroll; ++k) {
    const int64_t c = base + (int64_t)k * kManyThreads;
    if (c < q.pieces) {
      v[k] = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(q.src) + c);
      sb[k] = q.scales[c >> 2];
    }
  }
#pragma unroll
  for (int k = 0; k < kManyUnroll; ++k) {
    const int64_t c = base + (int64_t)k * kManyThreads;
    if (c >= q.pieces) break;
    const float s = sb[k] == 255u ? __uint_as_float(0x7FC00000u)
                                  : sb[k] == 0u ? __uint_as_float(0x00400000u) : __uint_as_float(sb[k] << 23);
    const uint32_t w[2] = {v[k].x, v[k].y};
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float f0 = __builtin_amdgcn_cvt_f32_fp8((int)w[e], 0) * s;
      const float f1 = __builtin_amdgcn_cvt_f32_fp8((int)w[e], 1) * s;
      const float f2 = __builtin_amdgcn_cvt_f32_fp8((int)w[e], 2) * s;
      const float f3 = __builtin_amdgcn_cvt_f32_fp8((int)w[e], 3) * s;
      o[2 * e] = many_value(f0) | (many_value(f1) << 16);
      o[2 * e + 1] = many_value(f2) | (many_value(f3) << 16);
    }
    __builtin_nontemporal_store(u32x4{o[0], o[1], o[2], o[3]}, reinterpret_cast<u32x4*>(q.out) + c);
  }
}

// Fills tables of up to kManyTensors non-empty tensors and launches each: `fill(i, entry)` sets what the
// kernel reads.
template <class Fill, class Launch>
static int many_launches(int64_t n, const int64_t* elems, Fill&& fill, Launch&& launch) {
  ManyTable table;
  int used = 0;
  int64_t blocks = 0;
  auto flush = [&]() -> int {
    if (used == 0) return MX_OK;
    launch(table, used, (unsigned)blocks);
    used = 0;
    blocks = 0;
    return hipGetLastError() == hipSuccess ? MX_OK : MX_ERR_LAUNCH;
  };
  for (int64_t i = 0; i < n; ++i) {
    if (elems[i] == 0) continue;
    const int64_t pieces = elems[i] / 8, per = kManyThreads * kManyUnroll;
    const int64_t mine = (pieces + per - 1) / per;
    if (mine > 0x7FFFFFFF) return MX_ERR_UNSUPPORTED;
    if (used == kManyTensors || blocks + mine > 0x7FFFFFFF)
      if (const int rc = flush()) return rc;
    ManyEntry e{};
    e.pieces = pieces;
    e.first = (uint32_t)blocks;
    fill(i, e);
    table.e[used++] = e;
    blocks += mine;
  }
  return flush();
}

}  // namespace mx

using namespace mx;

extern "C" int mx_cast_rows_many(int64_t n, const void* const* x, const int64_t* elems, const int32_t* is_f32,
                                 uint8_t* const* codes, uint8_t* const* scales, int scale_mode, void* stream) {
  if (n < 0 || (scale_mode != MX_SCALE_FLOOR && scale_mode != MX_SCALE_RCEIL)) return MX_ERR_INVALID_ARG;
  if (n > 0 && (!x || !elems || !is_f32 || !codes || !scales)) return MX_ERR_INVALID_ARG;
  for (int64_t i = 0; i < n; ++i) {
    if (elems[i] < 0 || (elems[i] > 0 && (!x[i] || !codes[i] || !scales[i]))) return MX_ERR_INVALID_ARG;
    if (elems[i] % 32 || ((uintptr_t)x[i] & 15) || ((uintptr_t)codes[i] & 7)) return MX_ERR_ALIGNMENT;
  }
  return many_launches(
      n, elems,
      [&](int64_t i, ManyEntry& e) {
        e.src = x[i];
        e.codes = codes[i];
        e.scales = scales[i];
        e.f32 = is_f32[i] != 0;
      },
      [&](const ManyTable& t, int used, unsigned blocks) {
        if (scale_mode == MX_SCALE_FLOOR)
          hipLaunchKernelGGL(cast_rows_many_kernel<MX_SCALE_FLOOR>, dim3(blocks), dim3(kManyThreads), 0,
                             (hipStream_t)stream, t, used);
        else
          hipLaunchKernelGGL(cast_rows_many_kernel<MX_SCALE_RCEIL>, dim3(blocks), dim3(kManyThreads), 0,
                             (hipStream_t)stream, t, used);
      });
}

extern "C" int mx_dequant_many(int64_t n, const uint8_t* const* codes, const uint8_t* const* scales,
                               const int64_t* elems, void* const* out, void* stream) {
  if (n < 0 || (n > 0 && (!codes || !scales || !elems || !out))) return MX_ERR_INVALID_ARG;
  for (int64_t i = 0; i < n; ++i) {
    if (elems[i] < 0 || (elems[i] > 0 && (!codes[i] || !scales[i] || !out[i]))) return MX_ERR_INVALID_ARG;
    if (elems[i] % 32 || ((uintptr_t)codes[i] & 15) || ((uintptr_t)out[i] & 15)) return MX_ERR_ALIGNMENT;
  }
  return many_launches(
      n, elems,
      [&](int64_t i, ManyEntry& e) {
        e.src = codes[i];
        e.scales = const_cast<uint8_t*>(scales[i]);
        e.out = (uint16_t*)out[i];
      },
      [&](const ManyTable& t, int used, unsigned blocks) {
        hipLaunchKernelGGL(dequant_many_kernel, dim3(blocks), dim3(kManyThreads), 0, (hipStream_t)stream, t, used);
      });
}
