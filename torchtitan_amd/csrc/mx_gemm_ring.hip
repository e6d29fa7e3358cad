// MXFP8 products of few tiles: one tile of 64 TA x 64 TB per workgroup, and as many 128-deep blocks of its operands in
// flight as the LDS holds.
//
//   D[M,N] = deq(A)[M,K] * deq(B)[N,K]^T, fp32 accumulate, bf16 (or bf16 values as float32) out.
//
// A product of some hundred rows has too few 256-wide tiles for the CUs, and each of them waits for its operands: a block
// takes 0.5 to 0.75 us where its MFMAs take 0.2 to 0.4.  Here the tiles are small, so that more CUs have one, and a ring
// of eight (64 x 64) or six (128 x 64) blocks hides the latency: a block takes 0.24 and 0.35 us on few CUs, 0.28 and 0.44
// with a tile on each.  That is about 580 and 840 cycles, of which the fragment reads fill 256 and 384 of the LDS's (32 and 48 KB
// at 128 B): what bounds it is the chain of a block, barrier, reads and their latency, MFMAs and waits, which nothing
// else on the CU overlaps, and with many CUs what they get out of the L2.  us on the GPU, before and now: 256 x 1024, K 2048 14.0 and 8.1; 512 x 1024, K 1024 9.7 and 6.8; 200 x 2560, K 4096 23.4 and 13.1;
// 768 x 1024, K 4096 23.4 and 13.4; 128 x 10240, K 3072 19.7 and 14.7.  (128 x 128 tiles with four blocks gain nothing over
// the persistent kernel anywhere: 14.2 us in the first of these.)
//
// Same LDS rows, swizzle, MFMA and operand layout as the persistent kernel (mx_gemm32.hip), and the same order of sums:
// one chain of 128-deep blocks per output, so that the choice between them does not change a bit.  Four waves in 2 x 2
// own half of either edge.  Per block one barrier: it says that the next block has landed (each wave has waited for
// its own copies) and that the current one's place is free (each has its fragments in registers).  Copies, reads of the
// next block's fragments and the MFMAs of this one's then run side by side.
#include "mx_gemm_tile.h"

namespace mx {

constexpr int kRingLds = 160 * 1024;

template <int TA, int TB>
struct RingLds {
  static constexpr int kA = 64 * TA * kBK, kCodes = 64 * (TA + TB) * kBK;
  static constexpr int kBlock = kCodes + 2048;  // + scales: a 128-row group of A, zeros, one of B, zeros (512 B each)
  static constexpr int kStages = kRingLds / kBlock < 8 ? kRingLds / kBlock : 8;
  static constexpr int kCopies = 2 * (TA + TB) + 1;  // of a block and wave
  static constexpr int kBytes = kStages * kBlock;
  static_assert((kStages - 1) * kCopies <= 63, "the wait counter has six bits");
};

template <int TA, int TB>
__global__ __launch_bounds__(256, 1) void gemm_ring_kernel(RingArgs p) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  using Lds = RingLds<TA, TB>;
  constexpr int S = Lds::kStages, TM = 2 * TA, TN = 2 * TB;
  const int64_t tiles_m1 = (p.M + 64 * TA - 1) / (64 * TA), tiles_n1 = (p.N + 64 * TB - 1) / (64 * TB);
  int64_t tm, tn;
  if (!map_tile(p.two == 2 ? 2 * tiles_m1 : tiles_m1, p.two == 1 ? 2 * tiles_n1 : tiles_n1, tm, tn)) return;
  const uint8_t *a_codes = p.a_codes, *a_scales = p.a_scales, *b_codes = p.b_codes, *b_scales = p.b_scales;
  void* d = p.d;
  if (p.two == 1 && tn >= tiles_n1) {
    tn -= tiles_n1;
    b_codes = p.b2_codes;
    b_scales = p.b2_scales;
    d = p.d2;
  }
  if (p.two == 2 && tm >= tiles_m1) {
    tm -= tiles_m1;
    a_codes = p.a2_codes;
    a_scales = p.a2_scales;
    d = p.d2;
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1, li = lane & 15, lj = lane >> 4;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_void_t*)smem;
  const uint32_t ld = (uint32_t)p.ldk;
  const int64_t m0 = tm * 64 * TA, n0 = tn * 64 * TB, ks_n = p.K / 64;
  const uint32_t blocks = (uint32_t)(p.K / kBK), total = p.pair ? 2 * blocks : blocks;

  // ---- copies: the persistent kernel's units of 8 rows x 128 B, see there
  const uint32_t c_even = (lane & 7) ^ ((lane >> 3) & 2);
  const uint32_t v_even = (uint32_t)(lane >> 3) * ld + c_even * 16;
  // waves 0, 1 copy the scales of A's 128-row group, 2 and 3 those of B's (each twice the same bytes); upper lanes: zeros
  const uint32_t v_scale = lane < 32 ? (uint32_t)lane * 16 : 0x80000000u;
  const uint32_t scale_dst = Lds::kCodes + (uint32_t)(wave >> 1) * 1024u;
  const uint8_t *a_from = a_codes + m0 * p.ldk, *b_from = b_codes + n0 * p.ldk;
  const int64_t s_from = wave < 2 ? (m0 >> 7) * ks_n * 256 : (n0 >> 7) * ks_n * 256;
  const uint8_t* s_of = (wave < 2 ? a_scales : b_scales) + s_from;
  const uint8_t *a2_from = p.pair ? p.a2_codes + m0 * p.ldk : a_from, *b2_from = p.pair ? p.b2_codes + n0 * p.ldk : b_from;
  const uint8_t* s2_of = p.pair ? (wave < 2 ? p.a2_scales : p.b2_scales) + s_from : s_of;
  uint32_t next = 0;  // block to be copied
  // (without branches: a block's MFMAs are to stay among its reads and copies)
  auto issue = [&](uint32_t slot) {
    const uint32_t sbase = lds_base + slot * Lds::kBlock;
    const bool second = next >= blocks;  // of a pair's two operand sets
    const uint32_t kb = second ? next - blocks : next;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(second ? a2_from : a_from, (p.M - m0) * p.ldk);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(second ? b2_from : b_from, (p.N - n0) * p.ldk);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(second ? s2_of : s_of, ks_n * 256);
    // behind the last block every lane reads out of range: the waits count the same copies throughout
    const uint32_t none = next >= total ? 0x80000000u : 0u;
    const uint32_t v0 = v_even | none, v1 = v0 ^ 64, vs = v_scale | none, k0 = none ? 0 : kb * kBK;
    static_for<0, 2 * TA>([&](auto q_) {
      constexpr int q = decltype(q_)::value;
      const uint32_t unit = wave * 2 * TA + q;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void_t*)(uintptr_t)(sbase + unit * 1024), 16, (q & 1) ? v1 : v0,
                                               unit * 8 * ld + k0, 0, 0);
    });
    static_for<0, 2 * TB>([&](auto q_) {
      constexpr int q = decltype(q_)::value;
      const uint32_t unit = wave * 2 * TB + q;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void_t*)(uintptr_t)(sbase + Lds::kA + unit * 1024), 16,
                                               (q & 1) ? v1 : v0, unit * 8 * ld + k0, 0, 0);
    });
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void_t*)(uintptr_t)(sbase + scale_dst), 16, vs, k0 * 4, 0, 0);
    ++next;
  };

  // ---- fragments.  The reads are assembly that the compiler's wait counts do not see (for reads that it sees it would
  // wait until every copy in flight has landed); `landed` is what the MFMAs depend on.
  struct Frags {
    v8i a[TM], b[TN];
    uint32_t sa[2], sb[2];
  };
  const uint32_t sw = (li & 2) | ((li & 8) >> 1);
  const uint32_t fa = (wm * 32 * TA + li) * kBK + ((lj ^ sw) << 4);
  const uint32_t fb = Lds::kA + (wn * 32 * TB + li) * kBK + ((lj ^ sw) << 4);
  const uint32_t fs = Lds::kCodes + (uint32_t)(lj >> 1) * 256 + (uint32_t)((lj & 1) * 32 + li) * 4;
  // the wave's first 32-row block in its 128-row scale group
  const uint32_t sh_a = 8 * (((uint32_t)(m0 >> 5) & 3) + wm * TA), sh_b = 8 * (((uint32_t)(n0 >> 5) & 3) + wn * TB);
  auto read_half = [&](v8i& to, uint32_t at, auto t_, auto hi_) {
    constexpr int t = decltype(t_)::value;
    v4i v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(t * 2048));
    if constexpr (decltype(hi_)::value) {
      to[4] = v.x; to[5] = v.y; to[6] = v.z; to[7] = v.w;
    } else {
      to[0] = v.x; to[1] = v.y; to[2] = v.z; to[3] = v.w;
    }
  };
  auto read_scales = [&](uint32_t& to, uint32_t at, auto off_) {
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(to) : "v"(at), "n"(decltype(off_)::value));
  };
  auto read = [&](Frags& f, uint32_t slot) {
    const uint32_t sbase = lds_base + slot * Lds::kBlock;
    read_scales(f.sa[0], sbase + fs, std::integral_constant<int, 0>{});
    read_scales(f.sa[1], sbase + fs, std::integral_constant<int, 64>{});
    read_scales(f.sb[0], sbase + fs, std::integral_constant<int, 1024>{});
    read_scales(f.sb[1], sbase + fs, std::integral_constant<int, 1024 + 64>{});
    static_for<0, TN>([&](auto t_) {
      read_half(f.b[decltype(t_)::value], sbase + fb, t_, std::false_type{});
      read_half(f.b[decltype(t_)::value], (sbase + fb) ^ 64u, t_, std::true_type{});
    });
    static_for<0, TM>([&](auto t_) {
      read_half(f.a[decltype(t_)::value], sbase + fa, t_, std::false_type{});
      read_half(f.a[decltype(t_)::value], (sbase + fa) ^ 64u, t_, std::true_type{});
    });
  };
  auto landed = [&](Frags& f) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    for (auto& x : f.a) asm volatile("" : "+v"(x));
    for (auto& x : f.b) asm volatile("" : "+v"(x));
    asm volatile("" : "+v"(f.sa[0]), "+v"(f.sa[1]), "+v"(f.sb[0]), "+v"(f.sb[1]));
    f.sa[0] >>= sh_a; f.sa[1] >>= sh_a;
    f.sb[0] >>= sh_b; f.sb[1] >>= sh_b;
  };

  v4f acc[TM][TN];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) acc[m][n] = v4f{0.f, 0.f, 0.f, 0.f};

  uint32_t slot = 0;  // of the block being computed
  auto after = [](uint32_t s) -> uint32_t { return s + 1 == S ? 0 : s + 1; };
  auto step = [&](Frags& cur, Frags& nxt) {
    // the next block has landed: all but the copies of the S - 2 blocks behind it
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * Lds::kCopies) : "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    read(nxt, after(slot));
    issue(slot);
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, TM>([&](auto m_) {
      constexpr int m = decltype(m_)::value;
      static_for<0, TN>([&](auto n_) {
        constexpr int n = decltype(n_)::value;
        mfma16_asm<(n >> 1), (m >> 1), false>(acc[m][n], cur.b[n], cur.a[m], cur.sb[n & 1], cur.sa[m & 1]);
      });
    });
    __builtin_amdgcn_sched_barrier(0);
    landed(nxt);
    slot = after(slot);
  };

#pragma unroll 1
  for (uint32_t i = 0; i < S; ++i) issue(i);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 1) * Lds::kCopies) : "memory");
  __builtin_amdgcn_s_barrier();
  Frags f0, f1;
  read(f0, 0);
  landed(f0);
  uint32_t s = 0;
  for (; s + 2 <= total; s += 2) {
    step(f0, f1);
    step(f1, f0);
  }
  if (s < total) step(f0, f1);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the copies behind the last block
  // The compiler does not know the assembly above for MFMAs: what reads the accumulators waits for the last one's passes,
  // and comes from here, so that no copy out of them is placed ahead of the wait.
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) asm volatile("" : "+a"(acc[m][n]));

  // ---- out: a lane holds row 16 m + li, columns 16 n + 4 lj .. + 3 of sub-tile (m, n)
  const int size = p.f32 ? 4 : 2;
  const uint32_t ldd_b = (uint32_t)p.ldd * size;
  const __amdgpu_buffer_rsrc_t rd = make_rsrc((uint8_t*)d + (m0 * p.ldd + n0) * size,
                                              (p.M - m0 < 64 * TA ? p.M - m0 : 64 * TA) * (int64_t)ldd_b);
  const uint32_t cols_left = p.N - n0 < 64 * TB ? (uint32_t)(p.N - n0) : 64 * TB;
  static_for<0, TM * TN>([&](auto i_) {
    constexpr int m = decltype(i_)::value / TN, n = decltype(i_)::value % TN;
    const uint32_t row = wm * 32 * TA + m * 16 + li, col = wn * 32 * TB + n * 16 + 4 * lj;
    const uint32_t v = col < cols_left ? row * ldd_b + col * size : 0x80000000u;
    const v4f a = acc[m][n];
    const u32x2 w = {pack_bf16(a.x, a.y), pack_bf16(a.z, a.w)};
    if (p.f32)
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{w.x << 16, w.x & 0xFFFF0000u, w.y << 16, w.y & 0xFFFF0000u}, rd, v, 0, 0);
    else
      __builtin_amdgcn_raw_buffer_store_b64(w, rd, v, 0, 0);
  });
}

template <int TA, int TB>
static bool configure_ring() {
  static std::atomic<bool> configured[kMaxDevices];
  return raise_lds_limit(reinterpret_cast<const void*>(gemm_ring_kernel<TA, TB>), RingLds<TA, TB>::kBytes, configured);
}
bool prepare_ring() { return configure_ring<1, 1>() && configure_ring<2, 1>(); }
bool prepare_dense();

template <int TA, int TB>
static int launch_ring_tile(const RingArgs& p, hipStream_t st) {
  if (!prepare_dense()) return MX_ERR_LAUNCH;
  const int64_t nb = ((p.M + 64 * TA - 1) / (64 * TA)) * ((p.N + 64 * TB - 1) / (64 * TB)) * (p.two ? 2 : 1);
  const int64_t grid = (nb + 7) / 8 * 8;
  if (grid > 0x7FFFFFFF) return MX_ERR_UNSUPPORTED;
  hipLaunchKernelGGL((gemm_ring_kernel<TA, TB>), dim3((unsigned)grid), dim3(256), (RingLds<TA, TB>::kBytes), st, p);
  return hipGetLastError() == hipSuccess ? MX_OK : MX_ERR_LAUNCH;
}
int launch_ring(const RingArgs& p, int ta, int tb, hipStream_t st) {
  if (ta == 1 && tb == 1) return launch_ring_tile<1, 1>(p, st);
  if (ta == 2 && tb == 1) return launch_ring_tile<2, 1>(p, st);
  return MX_ERR_UNSUPPORTED;
}

}  // namespace mx
