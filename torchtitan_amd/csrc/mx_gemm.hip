// Dense MXFP8 GEMM entry point: D[M,N] = deq(A)[M,K] * deq(B)[N,K]^T (bf16 out).
#include <mutex>

#include "mx_gemm_tile.h"

namespace mx {

struct DenseArgs {
  const uint8_t* a_codes;
  const uint8_t* a_scales;
  const uint8_t* b_codes;
  const uint8_t* b_scales;
  uint16_t* d;
  int64_t M, N, K, ldd;
  int64_t ldk;  // bytes between operand rows (>= K)
};

template <int BM, int BN, bool F32 = false>
__global__ __launch_bounds__(256, 1) void gemm_nt_kernel(DenseArgs p) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  using Tile = GemmTile<BM, BN, false, false>;
  const int64_t tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN;
  int64_t tm, tn;
  if (!map_tile(tiles_m, tiles_n, tm, tn)) return;
  const int64_t ks_n = (p.K / 32 + 1) / 2;
  Operand A{p.a_codes + tm * BM * p.ldk, p.ldk, p.M - tm * BM,
            p.a_scales + tm * (BM / 128) * ks_n * 256, ks_n};
  Operand B{p.b_codes + tn * BN * p.ldk, p.ldk, p.N - tn * BN,
            p.b_scales + tn * (BN / 128) * ks_n * 256, ks_n};
  Tile::template run<F32>(smem, A, B, 0, p.K, p.d + ((tm * BM * p.ldd + tn * BN) << (F32 ? 1 : 0)), p.ldd);
}

template <int BM, int BN, bool F32 = false>
static bool configure_dense() {
  static std::atomic<bool> configured[kMaxDevices];  // a per-function, per-device setting
  return raise_lds_limit(reinterpret_cast<const void*>(gemm_nt_kernel<BM, BN, F32>), GemmTile<BM, BN, false, false>::kLdsBytes,
                         configured);
}
// Raises the LDS limit of every kernel on tiles that a dense product of any shape and form may run on, in front of the
// first such launch on a GPU: limits are not to be raised under graph capture, and which tile a captured shape takes
// is not the caller's business.
bool prepare_dense32();
bool prepare_ring();
bool prepare_dense() {
  static std::atomic<bool> prepared[kMaxDevices];
  const int dev = current_device();
  if (dev < 0) return false;
  if (!prepared[dev].load(std::memory_order_acquire)) {
    if (!prepare_dense32() || !prepare_ring() || !configure_dense<128, 128>() || !configure_dense<256, 256>() ||
        !configure_dense<128, 128, true>())
      return false;
    prepared[dev].store(true, std::memory_order_release);
  }
  return true;
}

template <int BM, int BN, bool F32 = false>
static int launch_dense(const DenseArgs& p, hipStream_t st) {
  using Tile = GemmTile<BM, BN, false, false>;
  auto kern = gemm_nt_kernel<BM, BN, F32>;
  if (!prepare_dense()) return MX_ERR_LAUNCH;
  const int64_t nb = ((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
  const int64_t grid = (nb + 7) / 8 * 8;
  if (grid > 0x7FFFFFFF) return MX_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), Tile::kLdsBytes, st, p);
  return hipGetLastError() == hipSuccess ? MX_OK : MX_ERR_LAUNCH;
}

}  // namespace mx

using namespace mx;

namespace mx {
int launch_gemm_nt32(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                     const uint8_t* b_scales, void* d, int64_t M, int64_t N, int64_t K,
                     int64_t ldk, int64_t ldd, bool f32, hipStream_t st);
int launch_few_rows_codes(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                          const uint8_t* b_scales, void* d, int64_t M, int64_t N, int64_t K, int64_t ldk, int64_t ldd,
                          hipStream_t st);
GemmPlan plan_dense(int64_t M, int64_t N, int64_t K, bool may_split);
GemmPlan plan_ring(int64_t M, int64_t N, int64_t blocks, int products);
int launch_ring(const RingArgs& p, int ta, int tb, hipStream_t st);
int launch_gemm_nt32_splitk(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                            const uint8_t* b_scales, void* d, int64_t M, int64_t N, int64_t K,
                            int64_t ldk, int64_t ldd, const GemmPlan& plan, void* workspace, bool f32,
                            hipStream_t st);
}
// Test hooks (include/mxfp8_debug.h), process-wide.
// 0: pick by shape; 1 / 2: the 16x16x128 tile kernel with 256x256 / 128x128 tiles for every
// shape; 3: the persistent kernel wherever it is legal (comparison runs and tests)
static std::atomic<int> force_kernel{0};
extern "C" void mx_debug_force_kernel(int which) { force_kernel = which; }
namespace mx { void set_debug_grid(int g); }
extern "C" void mx_debug_set_grid(int g) { mx::set_debug_grid(g); }
extern "C" int mx_debug_lds_limits_raised(void) { return mx::lds_limits_raised; }
namespace mx { void set_debug_tile(int ta, int tb, int slices); }
extern "C" void mx_debug_set_tile(int ta, int tb, int slices) { mx::set_debug_tile(ta, tb, slices); }
#ifdef MX_TIMING_BUILD
namespace mx { void set_debug_prof(uint64_t* buf); }
// device buffer of 256*4*8 uint64 receiving per-wave cycle counts; nullptr switches timing off
extern "C" void mx_debug_set_prof(void* buf) { mx::set_debug_prof((uint64_t*)buf); }
#endif

static int check_dense(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                       const uint8_t* b_scales, const void* d, int64_t M, int64_t N, int64_t K,
                       int64_t ldd) {
  if (M < 0 || N < 0 || K < 0 || ldd < N) return MX_ERR_INVALID_ARG;
  if (M == 0 || N == 0) return MX_OK;
  if (!a_codes || !a_scales || !b_codes || !b_scales || !d) return MX_ERR_INVALID_ARG;
  if (K % 32 || K == 0) return MX_ERR_ALIGNMENT;  // K == 0 would need a zero fill: not a linear
  if (((uintptr_t)a_codes & 15) || ((uintptr_t)b_codes & 15) || ((uintptr_t)a_scales & 3) ||
      ((uintptr_t)b_scales & 3) || ((uintptr_t)d & 1) || (K % 16))
    return MX_ERR_ALIGNMENT;
  if (256 * K > 0x7FFFFFFFll) return MX_ERR_UNSUPPORTED;
  return MX_OK;
}

// What the persistent kernel (mx_gemm32.hip) needs beyond the general checks.
static bool persistent_ok(const void* d, int64_t N, int64_t K, int64_t ldd, int64_t ldk = 0) {
  if (ldk == 0) ldk = K;
  return !(K % 128 || ldk % 128 || (uint64_t)ldk * 256 > 0x7FFFFFFFull || N % 8 || ldd % 8 || ((uintptr_t)d & 15) ||
           (uint64_t)ldd * 512 > 0x7FFFFFFFull);
}

// Few rows: a workgroup for every 16 columns and more, its waves along the contraction, while its widest
// workgroups fit the CUs in one round: 64 rows 2048 -> 16384 13.6 us, 16.4 on tiles; 20480 25.1 and 16.9,
// 151936 127.8 and 86.8.
static bool few_rows_shape(int64_t M, int64_t N, int64_t K) { return M <= 64 && K % 128 == 0 && N <= 16384; }

// mx_gemm_nt with operand rows `ldk` bytes apart (ldk >= K, a multiple of 16).
static int gemm_nt_pitched(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                           const uint8_t* b_scales, void* d, int64_t M, int64_t N, int64_t K, int64_t ldk,
                           int64_t ldd, void* stream) {
  const int rc = check_dense(a_codes, a_scales, b_codes, b_scales, d, M, N, K, ldd);
  if (rc != MX_OK || M == 0 || N == 0) return rc;
  if (ldk < K) return MX_ERR_INVALID_ARG;
  if (ldk % 16) return MX_ERR_ALIGNMENT;
  if (256 * ldk > 0x7FFFFFFFll) return MX_ERR_UNSUPPORTED;
  DenseArgs p{a_codes, a_scales, b_codes, b_scales, (uint16_t*)d, M, N, K, ldd, ldk};
  hipStream_t st = (hipStream_t)stream;
  if (few_rows_shape(M, N, K) && force_kernel == 0)
    return launch_few_rows_codes(a_codes, a_scales, b_codes, b_scales, d, M, N, K, ldk, ldd, st);
  if (N <= 128 || (M <= 128 && force_kernel != 0) || force_kernel == 2) return launch_dense<128, 128>(p, st);
  if (force_kernel == 0) {
    if (!persistent_ok(d, N, K, ldd, ldk)) {
      // (few 256 x 256 tiles: four times as many 128 x 128 ones finish sooner)
      int num_cus = current_device_cus();
      if (num_cus == 0) num_cus = 256;
      const int64_t tiles256 = ((M + 255) / 256) * ((N + 255) / 256);
      if (M <= 128 || tiles256 * 8 <= (int64_t)num_cus * 3) return launch_dense<128, 128>(p, st);
      return launch_dense<256, 256>(p, st);
    }
    const GemmPlan plan = plan_dense(M, N, K, false);
    if (plan.ta == 0) return launch_dense<128, 128>(p, st);
    if (plan.ring())
      return launch_ring({a_codes, a_scales, b_codes, b_scales, nullptr, nullptr, nullptr, nullptr, d, nullptr, M, N, K, ldk, ldd,
                          0, 0, 0}, plan.ta, plan.tb, st);
  }
  if (force_kernel == 1 || !persistent_ok(d, N, K, ldd, ldk)) return launch_dense<256, 256>(p, st);
  return launch_gemm_nt32(a_codes, a_scales, b_codes, b_scales, d, M, N, K, ldk, ldd, false, st);
}

extern "C" int mx_gemm_nt(const uint8_t* a_codes, const uint8_t* a_scales,
                          const uint8_t* b_codes, const uint8_t* b_scales, void* d, int64_t M,
                          int64_t N, int64_t K, int64_t ldd, void* stream) {
  return gemm_nt_pitched(a_codes, a_scales, b_codes, b_scales, d, M, N, K, K, ldd, stream);
}

namespace mx {
int launch_gemm_nt32_pair(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                          const uint8_t* b_scales, const uint8_t* a2_codes, const uint8_t* a2_scales,
                          const uint8_t* b2_codes, const uint8_t* b2_scales, void* d, int64_t M,
                          int64_t N, int64_t K, int64_t ldk, int64_t ldd, hipStream_t st);
GemmPlan plan_pair(int64_t M, int64_t N, int64_t K);
int launch_gemm_nt32_pair_splitk(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                                 const uint8_t* b_scales, const uint8_t* a2_codes, const uint8_t* a2_scales,
                                 const uint8_t* b2_codes, const uint8_t* b2_scales, void* d, int64_t M, int64_t N,
                                 int64_t K, int64_t ldk, int64_t ldd, const GemmPlan& plan, void* workspace,
                                 hipStream_t st);
}

// The forms over two operand sets exist for the persistent kernel only, dense rows (ldk == K) or
// pitched: other shapes are the caller's two GEMMs (and an add).
extern "C" int mx_gemm_nt_pair_ld(const uint8_t* a_codes, const uint8_t* a_scales,
                                  const uint8_t* b_codes, const uint8_t* b_scales,
                                  const uint8_t* a2_codes, const uint8_t* a2_scales,
                                  const uint8_t* b2_codes, const uint8_t* b2_scales, void* d,
                                  int64_t M, int64_t N, int64_t K, int64_t ldk, int64_t ldd,
                                  void* stream) {
  int rc = check_dense(a_codes, a_scales, b_codes, b_scales, d, M, N, K, ldd);
  if (rc == MX_OK) rc = check_dense(a2_codes, a2_scales, b2_codes, b2_scales, d, M, N, K, ldd);
  if (rc != MX_OK || M == 0 || N == 0) return rc;
  if (ldk < K) return MX_ERR_INVALID_ARG;
  if (M <= 128 || N <= 128 || !persistent_ok(d, N, K, ldd, ldk) || force_kernel == 1 || force_kernel == 2)
    return MX_ERR_UNSUPPORTED;
  const GemmPlan plan = force_kernel == 0 ? plan_ring(M, N, 2 * (K / 128), 1) : GemmPlan{0, 0, 1};
  if (plan.ring())
    return launch_ring({a_codes, a_scales, b_codes, b_scales, a2_codes, a2_scales, b2_codes, b2_scales, d, nullptr, M, N, K, ldk,
                        ldd, 0, 1, 0}, plan.ta, plan.tb, (hipStream_t)stream);
  return launch_gemm_nt32_pair(a_codes, a_scales, b_codes, b_scales, a2_codes, a2_scales, b2_codes,
                               b2_scales, d, M, N, K, ldk, ldd, (hipStream_t)stream);
}

extern "C" int64_t mx_gemm_nt_pair_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 128 || N <= 128 || K <= 0 || N % 8 || (uint64_t)N * 1024 > 0x7FFFFFFFull) return 0;
  const GemmPlan plan = plan_pair(M, N, K);
  return plan.slices > 1 ? (int64_t)plan.slices * M * N * 4 : 0;
}

extern "C" int mx_gemm_nt_pair_ws(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                                  const uint8_t* b_scales, const uint8_t* a2_codes, const uint8_t* a2_scales,
                                  const uint8_t* b2_codes, const uint8_t* b2_scales, void* d, int64_t M, int64_t N,
                                  int64_t K, int64_t ldk, int64_t ldd, void* workspace, int64_t workspace_bytes,
                                  void* stream) {
  int rc = check_dense(a_codes, a_scales, b_codes, b_scales, d, M, N, K, ldd);
  if (rc == MX_OK) rc = check_dense(a2_codes, a2_scales, b2_codes, b2_scales, d, M, N, K, ldd);
  if (rc != MX_OK || M == 0 || N == 0) return rc;
  if (ldk < K) return MX_ERR_INVALID_ARG;
  const int64_t need = force_kernel == 0 && persistent_ok(d, N, K, ldd, ldk) ? mx_gemm_nt_pair_workspace_bytes(M, N, K) : 0;
  if (need == 0 || !workspace || workspace_bytes < need || ((uintptr_t)workspace & 15))
    return mx_gemm_nt_pair_ld(a_codes, a_scales, b_codes, b_scales, a2_codes, a2_scales, b2_codes, b2_scales, d, M, N, K,
                              ldk, ldd, stream);
  return launch_gemm_nt32_pair_splitk(a_codes, a_scales, b_codes, b_scales, a2_codes, a2_scales, b2_codes, b2_scales, d, M, N,
                                      K, ldk, ldd, plan_pair(M, N, K), workspace, (hipStream_t)stream);
}

extern "C" int mx_gemm_nt_pair(const uint8_t* a_codes, const uint8_t* a_scales,
                               const uint8_t* b_codes, const uint8_t* b_scales,
                               const uint8_t* a2_codes, const uint8_t* a2_scales,
                               const uint8_t* b2_codes, const uint8_t* b2_scales, void* d,
                               int64_t M, int64_t N, int64_t K, int64_t ldd, void* stream) {
  return mx_gemm_nt_pair_ld(a_codes, a_scales, b_codes, b_scales, a2_codes, a2_scales, b2_codes, b2_scales, d,
                            M, N, K, K, ldd, stream);
}

namespace mx {
int launch_gemm_nt32_two_b(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                           const uint8_t* b_scales, const uint8_t* b2_codes, const uint8_t* b2_scales,
                           void* d, void* d2, int64_t M, int64_t N, int64_t K, int64_t ldk, int64_t ldd,
                           hipStream_t st);
int launch_gemm_nt32_two_a(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* a2_codes,
                           const uint8_t* a2_scales, const uint8_t* b_codes, const uint8_t* b_scales,
                           void* d, void* d2, int64_t M, int64_t N, int64_t K, int64_t ldk, int64_t ldd,
                           hipStream_t st);
}

// Two products that share an operand, one launch of the persistent kernel; other shapes are the
// caller's two mx_gemm_nt calls.
extern "C" int mx_gemm_nt_shared_a_ld(const uint8_t* a_codes, const uint8_t* a_scales,
                                      const uint8_t* b_codes, const uint8_t* b_scales,
                                      const uint8_t* b2_codes, const uint8_t* b2_scales, void* d,
                                      void* d2, int64_t M, int64_t N, int64_t K, int64_t ldk,
                                      int64_t ldd, void* stream) {
  int rc = check_dense(a_codes, a_scales, b_codes, b_scales, d, M, N, K, ldd);
  if (rc == MX_OK) rc = check_dense(a_codes, a_scales, b2_codes, b2_scales, d2, M, N, K, ldd);
  if (rc != MX_OK || M == 0 || N == 0) return rc;
  if (ldk < K) return MX_ERR_INVALID_ARG;
  if (M <= 128 || N <= 128 || !persistent_ok(d, N, K, ldd, ldk) || !persistent_ok(d2, N, K, ldd, ldk) ||
      force_kernel == 1 || force_kernel == 2)
    return MX_ERR_UNSUPPORTED;
  const GemmPlan plan = force_kernel == 0 ? plan_ring(M, N, K / 128, 2) : GemmPlan{0, 0, 1};
  if (plan.ring())
    return launch_ring({a_codes, a_scales, b_codes, b_scales, nullptr, nullptr, b2_codes, b2_scales, d, d2, M, N, K, ldk, ldd, 1,
                        0, 0}, plan.ta, plan.tb, (hipStream_t)stream);
  return launch_gemm_nt32_two_b(a_codes, a_scales, b_codes, b_scales, b2_codes, b2_scales, d, d2, M, N,
                                K, ldk, ldd, (hipStream_t)stream);
}

namespace mx {
bool plan_gated(int64_t M, int64_t N, int64_t K);
int launch_gemm_nt32_gated(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes, const uint8_t* b_scales,
                           const uint8_t* b2_codes, const uint8_t* b2_scales, uint8_t* codes, uint8_t* scales, int64_t M,
                           int64_t N, int64_t K, int64_t ldk, int64_t ld_codes, int scale_mode, hipStream_t st);
}

extern "C" int mx_gemm_nt_swiglu_planned(int64_t M, int64_t N, int64_t K) {
  return M > 128 && N > 128 && K > 0 && N % 8 == 0 && K % 128 == 0 && force_kernel == 0 && plan_gated(M, N, K);
}

extern "C" int mx_gemm_nt_swiglu_ld(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                                    const uint8_t* b_scales, const uint8_t* b2_codes, const uint8_t* b2_scales,
                                    uint8_t* codes, int64_t ld_codes, uint8_t* scales, int64_t M, int64_t N, int64_t K,
                                    int64_t ldk, int scale_mode, void* stream) {
  int rc = check_dense(a_codes, a_scales, b_codes, b_scales, codes, M, N, K, N);
  if (rc == MX_OK) rc = check_dense(a_codes, a_scales, b2_codes, b2_scales, codes, M, N, K, N);
  if (rc != MX_OK || M == 0 || N == 0) return rc;
  if (ldk < K || ld_codes < (N + 127) / 128 * 128 || !scales || (scale_mode != MX_SCALE_FLOOR && scale_mode != MX_SCALE_RCEIL))
    return MX_ERR_INVALID_ARG;
  if (ld_codes % 16 || ((uintptr_t)codes & 15) || ((uintptr_t)scales & 3)) return MX_ERR_ALIGNMENT;
  if (M <= 128 || N <= 128 || K % 128 || ldk % 128 || (uint64_t)ldk * 256 > 0x7FFFFFFFull || N % 8 ||
      (uint64_t)ld_codes * 256 > 0x7FFFFFFFull)
    return MX_ERR_UNSUPPORTED;
  return launch_gemm_nt32_gated(a_codes, a_scales, b_codes, b_scales, b2_codes, b2_scales, codes, scales, M, N, K, ldk, ld_codes,
                                scale_mode, (hipStream_t)stream);
}

extern "C" int mx_gemm_nt_shared_a(const uint8_t* a_codes, const uint8_t* a_scales,
                                   const uint8_t* b_codes, const uint8_t* b_scales,
                                   const uint8_t* b2_codes, const uint8_t* b2_scales, void* d,
                                   void* d2, int64_t M, int64_t N, int64_t K, int64_t ldd,
                                   void* stream) {
  return mx_gemm_nt_shared_a_ld(a_codes, a_scales, b_codes, b_scales, b2_codes, b2_scales, d, d2, M, N, K, K,
                                ldd, stream);
}

extern "C" int mx_gemm_nt_shared_b_ld(const uint8_t* a_codes, const uint8_t* a_scales,
                                      const uint8_t* a2_codes, const uint8_t* a2_scales,
                                      const uint8_t* b_codes, const uint8_t* b_scales, void* d,
                                      void* d2, int64_t M, int64_t N, int64_t K, int64_t ldk,
                                      int64_t ldd, void* stream) {
  int rc = check_dense(a_codes, a_scales, b_codes, b_scales, d, M, N, K, ldd);
  if (rc == MX_OK) rc = check_dense(a2_codes, a2_scales, b_codes, b_scales, d2, M, N, K, ldd);
  if (rc != MX_OK || M == 0 || N == 0) return rc;
  if (ldk < K) return MX_ERR_INVALID_ARG;
  if (M <= 128 || N <= 128 || !persistent_ok(d, N, K, ldd, ldk) || !persistent_ok(d2, N, K, ldd, ldk) ||
      force_kernel == 1 || force_kernel == 2)
    return MX_ERR_UNSUPPORTED;
  const GemmPlan plan = force_kernel == 0 ? plan_ring(M, N, K / 128, 2) : GemmPlan{0, 0, 1};
  if (plan.ring())
    return launch_ring({a_codes, a_scales, b_codes, b_scales, a2_codes, a2_scales, nullptr, nullptr, d, d2, M, N, K, ldk, ldd, 2,
                        0, 0}, plan.ta, plan.tb, (hipStream_t)stream);
  return launch_gemm_nt32_two_a(a_codes, a_scales, a2_codes, a2_scales, b_codes, b_scales, d, d2, M, N,
                                K, ldk, ldd, (hipStream_t)stream);
}

extern "C" int mx_gemm_nt_shared_b(const uint8_t* a_codes, const uint8_t* a_scales,
                                   const uint8_t* a2_codes, const uint8_t* a2_scales,
                                   const uint8_t* b_codes, const uint8_t* b_scales, void* d,
                                   void* d2, int64_t M, int64_t N, int64_t K, int64_t ldd,
                                   void* stream) {
  return mx_gemm_nt_shared_b_ld(a_codes, a_scales, a2_codes, a2_scales, b_codes, b_scales, d, d2, M, N, K, K,
                                ldd, stream);
}

// How the shape is split along K by a caller that lends memory for the partial sums (slices == 1: not).
static GemmPlan split_plan(int64_t M, int64_t N, int64_t K) {
  constexpr GemmPlan kNone{0, 0, 1};
  if (M <= 0 || N <= 128 || K <= 0 || N % 8 || (uint64_t)N * 1024 > 0x7FFFFFFFull) return kNone;
  // Few rows run on their own kernel up to here; behind it slices on tiles are ahead although they
  // are summed by a second launch (16 x 4096: K 8192 12.8 us, 16.2 in eight slices, K 14336 19.9 and
  // 20.1; 64 x 4096: K 4096 13.4 and 14.8, K 8192 23.7 and 17.2, K 14336 38 and 22; 64 x 14336, K 4096
  // 24 and 20).
  if (few_rows_shape(M, N, K) && ((M + 15) / 16 * 16) * K <= 270000ll * 8192 / (N > 8192 ? N : 8192)) return kNone;
  return plan_dense(M, N, K, true);
}
static int64_t split_bytes(const GemmPlan& plan, int64_t M, int64_t N) {
  return plan.slices > 1 ? (int64_t)plan.slices * M * N * 4 : 0;
}

extern "C" int64_t mx_gemm_nt_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  return split_bytes(split_plan(M, N, K), M, N);
}

extern "C" int mx_gemm_nt_ld(const uint8_t* a_codes, const uint8_t* a_scales,
                             const uint8_t* b_codes, const uint8_t* b_scales, void* d, int64_t M,
                             int64_t N, int64_t K, int64_t ldk, int64_t ldd, void* workspace,
                             int64_t workspace_bytes, void* stream) {
  const int rc = check_dense(a_codes, a_scales, b_codes, b_scales, d, M, N, K, ldd);
  if (rc != MX_OK || M == 0 || N == 0) return rc;
  if (ldk < K) return MX_ERR_INVALID_ARG;
  GemmPlan plan{0, 0, 1};
  if (workspace && force_kernel == 0 && persistent_ok(d, N, K, ldd, ldk)) plan = split_plan(M, N, K);
  if (plan.slices == 1 || workspace_bytes < split_bytes(plan, M, N) || ((uintptr_t)workspace & 15))
    return gemm_nt_pitched(a_codes, a_scales, b_codes, b_scales, d, M, N, K, ldk, ldd, stream);
  return launch_gemm_nt32_splitk(a_codes, a_scales, b_codes, b_scales, d, M, N, K, ldk, ldd,
                                 plan, workspace, false, (hipStream_t)stream);
}

extern "C" int mx_gemm_nt_f32_ld(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                                 const uint8_t* b_scales, float* d, int64_t M, int64_t N, int64_t K, int64_t ldk,
                                 int64_t ldd, void* workspace, int64_t workspace_bytes, void* stream) {
  const int rc = check_dense(a_codes, a_scales, b_codes, b_scales, d, M, N, K, ldd);
  if (rc != MX_OK || M == 0 || N == 0) return rc;
  if (ldk < K) return MX_ERR_INVALID_ARG;
  // (the descriptor of a tile's output spans 256 rows of 4-byte values)
  if (M <= 64 || N <= 128 || !persistent_ok(d, N, K, ldd, ldk) || (uint64_t)ldd * 1024 > 0x7FFFFFFFull)
    return MX_ERR_UNSUPPORTED;
  hipStream_t st = (hipStream_t)stream;
  if (workspace && force_kernel == 0 && !((uintptr_t)workspace & 15)) {
    const GemmPlan plan = split_plan(M, N, K);
    if (plan.slices > 1 && workspace_bytes >= split_bytes(plan, M, N))
      return launch_gemm_nt32_splitk(a_codes, a_scales, b_codes, b_scales, d, M, N, K, ldk, ldd, plan, workspace, true, st);
  }
  const GemmPlan plan = force_kernel == 0 ? plan_dense(M, N, K, false) : GemmPlan{4, 4, 1};
  if (plan.ring())
    return launch_ring({a_codes, a_scales, b_codes, b_scales, nullptr, nullptr, nullptr, nullptr, d, nullptr, M, N, K, ldk, ldd,
                        0, 0, 1}, plan.ta, plan.tb, st);
  if (force_kernel == 1 || force_kernel == 2 || plan.ta == 0)
    return launch_dense<128, 128, true>(DenseArgs{a_codes, a_scales, b_codes, b_scales, (uint16_t*)d, M, N, K, ldd, ldk}, st);
  return launch_gemm_nt32(a_codes, a_scales, b_codes, b_scales, d, M, N, K, ldk, ldd, true, st);
}

extern "C" int mx_gemm_nt_ws(const uint8_t* a_codes, const uint8_t* a_scales,
                             const uint8_t* b_codes, const uint8_t* b_scales, void* d, int64_t M,
                             int64_t N, int64_t K, int64_t ldd, void* workspace,
                             int64_t workspace_bytes, void* stream) {
  return mx_gemm_nt_ld(a_codes, a_scales, b_codes, b_scales, d, M, N, K, K, ldd, workspace, workspace_bytes,
                       stream);
}

// ---- the split GEMM for callers that cannot allocate -------------------------------------------
// The float32 partial tiles of the split along K live in a file-scope device array instead of a
// caller-provided workspace.  Every GPU holds its own copy of the array at its own address until
// the process ends; the address is looked up once per device and is what the kernels receive.
constexpr int64_t kScratchBytes = 64ll << 20;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

static void* scratch_ptr[kMaxDevices];  // device address of `scratch` per GPU, nullptr: not looked up yet
static std::mutex scratch_mutex;

// Device address of this GPU's scratch array (nullptr: the lookup failed).
static void* scratch_of_current_device() {
  const int dev = current_device();
  if (dev < 0) return nullptr;
  std::lock_guard<std::mutex> lock(scratch_mutex);
  if (!scratch_ptr[dev]) {
    if (!prepare_dense()) return nullptr;
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
    scratch_ptr[dev] = ptr;
  }
  return scratch_ptr[dev];
}

extern "C" int64_t mx_gemm_nt_static_max_bytes(void) { return kScratchBytes; }

extern "C" int mx_gemm_nt_static(const uint8_t* a_codes, const uint8_t* a_scales,
                                 const uint8_t* b_codes, const uint8_t* b_scales, void* d,
                                 int64_t M, int64_t N, int64_t K, int64_t ldd, void* stream) {
  const int rc = check_dense(a_codes, a_scales, b_codes, b_scales, d, M, N, K, ldd);
  if (rc != MX_OK || M == 0 || N == 0) return rc;
  // the size check stands on the shape alone, whatever the test hooks say
  const GemmPlan plan = split_plan(M, N, K);
  if (split_bytes(plan, M, N) > kScratchBytes && persistent_ok(d, N, K, ldd)) return MX_ERR_SCRATCH_TOO_SMALL;
  void* ws = scratch_of_current_device();
  if (plan.slices == 1 || force_kernel != 0 || !persistent_ok(d, N, K, ldd))  // not split: no scratch involved
    return mx_gemm_nt(a_codes, a_scales, b_codes, b_scales, d, M, N, K, ldd, stream);
  if (!ws) return MX_ERR_LAUNCH;
  return launch_gemm_nt32_splitk(a_codes, a_scales, b_codes, b_scales, d, M, N, K, K, ldd,
                                 plan, ws, false, (hipStream_t)stream);
}
