// MXFP8 GEMM for large shapes, dense and grouped: persistent 256x256 tiles (dense also 192x256,
// 256x192, 128x256 and 256x128) on the scaled fp8 MFMA v_mfma_scale_f32_16x16x128_f8f6f4.
//
//   D[M,N] (bf16) = deq(A)[M,K] * deq(B)[N,K]^T, fp32 accumulate.
//
// One workgroup (4 waves, 2x2, 128x128 each = 256 accumulator registers per lane) per CU walks
// a list of output tiles; the K loops of all its tiles form one flat stream of 128-deep
// blocks, so the loads of the next tile's first blocks are already in flight while a tile is
// written out.
//
// (Numbers here and below are those of the 256x256 tile where nothing else is said: a wave owns half of
// either edge of any tile, Lds32 and BlockPlan have what follows from that.)
//
// Global -> LDS moves whole 128-byte rows (buffer_load_dwordx4 ... lds, 8 rows per instruction:
// full cache lines, which the texture path delivers about twice as fast as 64-byte pieces), so
// the ring holds two 128-deep blocks of 64 KB codes + 2 KB scales (128x256 and 256x128 tiles: three of
// 48 + 2 KB).  Two barriers per block: one
// releases the ring block whose last fragments have just been read (its refill starts there,
// spread thinly because the copy path is the scarce resource), one makes sure the next block
// has landed.
//
// Which MFMA.  The 16x16x128 and the 32x32x64 form both do 2048 flop per cycle and SIMD and read
// the same operand bytes per flop; the 16x16x128 one reads and writes a quarter of the
// accumulator registers per instruction.  Under the chip's power limit that is worth 9 % of
// sustained rate on the same operand bits with nothing else running, and was worth 6-10 % of
// shader clock inside this kernel against 2-3 % more cycles when the K loop moved to it (64 MFMA
// slots of 32 cycles per block leave less room behind each MFMA for the block's LDS reads and
// copies than 32 slots of 64 cycles).
//   A block is 64 MFMAs, one per 16x16 sub-tile, in four quarters over four fragment sets (two
//   64-row halves of A, two of B) that are refilled in place as soon as their last MFMA has been
//   issued; see block_steps for the slot plan.  Operand layout (measured): lane (i = l & 15,
//   j = l >> 4) holds row i, K bytes [16j, 16j+16) in registers 0-3 and [64+16j, 64+16j+16) in
//   registers 4-7; the scale of 32-element block b is taken from lane group b.  With the first
//   operand = B rows and the second = A rows, a lane ends up with D[row = l & 15][col = 4j + 0..3].
// Fragment reads are conflict-free under the b128 pass grouping.
//
// MX_ABL_NO_DMA / MX_ABL_NO_READ / MX_ABL_STORE_ROWS / MX_ABL_NO_EPILOGUE (never defined in the
// product build) drop the copies, the fragment reads, part of the output stores or the whole
// epilogue from the steady state, to time what is left; MX_ABL_SAME_PANEL makes all dense tiles
// read the same twelve operand panels (MX_ABL_SAME_A / MX_ABL_SAME_B: the same A / B panels only), so
// that every read beyond the L2 finds its line in the memory-side cache; MX_ABL_ROW_PAD=n reads the
// rows of a tile n bytes further apart than they lie (what a padded row pitch would do to the
// spread of a block's lines over the cache channels); MX_ABL_TR_READ issues every fragment read as
// two ds_read_b64_tr_b8 (what a K loop over operands stored K-strided would issue); MX_ABL_DMA_OOB
// issues every copy with all lanes out of range (the instructions and their LDS writes stay, the
// fetches go).  Results are then meaningless.
#include "mx_gemm_tile.h"

namespace mx {

constexpr int kT32 = 256;                        // tile edge (M and N)
constexpr int kK32 = 64;                         // K per compute step
constexpr int kKB = 128;                         // K per ring block (= one cache line per row)
constexpr int kCodes32 = 2 * kT32 * kKB;         // A rows then B rows, 256 of 128 B each
constexpr int kBlock32 = kCodes32 + 3072;        // + scales: groups A0, A1, B0, B1, A2 (+ 512 unused) x 2 steps x 256 B
constexpr int kRing32 = 2 * kBlock32;            // 134 KB
constexpr int kPatch32 = 6656;                   // per wave: 4608 B output patch + 2 KB of records / tables
constexpr int kPatchUsed = 4608;
constexpr int kPatchPitch = 144;                 // bytes per staged row: 128 + 16, keeps b128 accesses spread
constexpr uint32_t kRecordsPerPatch = (kPatch32 - kPatchUsed) / 64;
constexpr uint32_t kMaxTileRecords = 3 * kRecordsPerPatch;  // grouped modes: tile records a workgroup keeps in LDS
static_assert(kRing32 + 4 * kPatch32 == 160 * 1024, "the kernel's LDS map fills the CU's 160 KB");

// What a launch works on.  One kernel serves three problems that differ only in how a linear
// tile number maps to operand rows, K range and output address:
//   kDense        D[M,N] = A[M,K] B[N,K]^T
//   kGrouped2d3d  rows of A in groups (inclusive ends offs[g], all multiples of 32), group g
//                 against B[g][N,K]; rows from offs[G-1] to M are written as zeros
//   kGrouped2d2d  D[g][M,N] = A[M, lo_g:hi_g] B[N, lo_g:hi_g]^T, K = row length of A and B
//   kSplitK       as kGrouped2d2d with G equal slices of the K blocks worked out in the kernel
//                 and float32 output: D[g][M,N] are partial sums for a reduction pass
enum Gemm32Mode { kDense = 0, kGrouped2d3d = 1, kGrouped2d2d = 2, kSplitK = 3 };
struct Gemm32Args {
  const uint8_t* a_codes;
  const uint8_t* a_scales;
  const uint8_t* b_codes;
  const uint8_t* b_scales;
  uint16_t* d;
  int64_t M, N, K, ldd;
  const int32_t* offs;  // grouped modes: inclusive cumulative group sizes, on the device
  int64_t G;
  int32_t tn0, tn_cnt;  // grouped modes: this launch covers tile columns [tn0, tn0 + tn_cnt)
  uint64_t* prof;  // timing build only: per wave {vmcnt wait, barrier wait, step body} cycles
  // PAIR kernels: a second operand set of the same shapes; D = A B^T + A2 B2^T in one pass, every
  // output tile running the K blocks of the first set and then those of the second before it is
  // written out (dx = da W1 + db W3 of a SwiGLU block's backward)
  const uint8_t* a2_codes = nullptr;
  const uint8_t* a2_scales = nullptr;
  const uint8_t* b2_codes = nullptr;
  const uint8_t* b2_scales = nullptr;
  // Two products that share one operand in one launch (not with PAIR).  kTwoB: D = A B^T and
  // D2 = A B2^T, the tile columns of the second product numbered behind those of the first
  // (h1 = x W1^T and h3 = x W3^T of a SwiGLU block: every A panel is fetched for both).  kTwoA:
  // D = A B^T and D2 = A2 B^T, the tile rows of the second behind those of the first (the weight
  // gradients dW1 = d(h1)^T x and dW3 = d(h3)^T x).
  int32_t two = 0;
  uint16_t* d2 = nullptr;
  // kDense, kSplitK: bytes between the rows of A and of B (both operands' rows are K bytes long
  // and may lie further apart, by a multiple of 128); 0 = K
  int64_t ldk = 0;
  // kGrouped2d3d: output rows without the groups' padding.  Group g's first d_offs[g] -
  // d_offs[g-1] rows are written to rows [d_offs[g-1], d_offs[g]) of D (inclusive ends, on the
  // device), the rest of its rows nowhere; rows [d_offs[G-1], d_rows) of D are written as zeros
  // as far as A has rows behind its last group.  nullptr: D has A's rows.
  const int32_t* d_offs = nullptr;
  int64_t d_rows = 0;
  // kSplitK: 2 = the sum of two products (a2 .. b2 as for PAIR), each cut into G / 2 slices
  int32_t sets = 1;
  // GATE: how the gated product is scaled (d its codes, ldd bytes between their rows, d2 their scales)
  int32_t scale_mode = 0;
};
enum Gemm32Two { kTwoNone = 0, kTwoB = 1, kTwoA = 2 };

// Where one 256x256 tile lives.
struct Tile32 {
  const uint8_t *a, *b;    // first operand row of the tile, at the first K byte of its range
  const uint8_t *sa, *sb;  // scales of the tile's first 128-row group at its first 64-deep step
  uint16_t* d;
  int64_t rows_a, rows_b;  // valid rows from the tile's origin (may exceed 256; <= 0: none)
  int32_t rows_d;          // Gemm32Args::d_offs given: rows of the tile that D has (0..256)
  uint32_t koff;           // first K byte of the range inside an operand row (kGrouped2d2d)
  uint32_t nblocks;        // 128-deep K blocks, at least 1
  bool empty;              // no K range (an empty group, rows behind the last group, or poison):
                           // one block of out-of-range reads, i.e. zeros, stands in for it
  bool poison;             // grouped modes: the group ends break the alignment contract
  uint32_t rot;            // kGrouped2d3d: 32-row blocks between the tile's first row and the start of
                           // its 128-row scale group (0..3): the A scale bytes are turned by as much
  uint32_t odd;            // 192-row tiles: bit 0 / 1: the tile begins in the middle of a 128-row scale
                           // group of A / of B
  uint32_t tm, tn;         // GATE: its row and column
  uint32_t head, tail;     // kGrouped2d2d: the K range starts `head` 32-deep blocks into its first
                           // 128-deep block and ends `tail` of them into its last (0: at its end)
};

// Tile order: 8-tall column-major panels, so tiles that run together share A and B panels.
// 32-bit arithmetic: the tile count of any supported shape is far below 2^31.
__device__ __forceinline__ void tile_coords(uint32_t t, uint32_t tiles_m, uint32_t tiles_n,
                                            uint32_t& tm, uint32_t& tn) {
  constexpr uint32_t kGroupM = 8;
  const uint32_t width = kGroupM * tiles_n;
  const uint32_t group = t / width;
  const uint32_t first_m = group * kGroupM;
  const uint32_t gsz = tiles_m - first_m < kGroupM ? tiles_m - first_m : kGroupM;
  const uint32_t in = t - group * width;
  tn = in / gsz;
  tm = first_m + (in - tn * gsz);
}

// LDS accesses the compiler must not see (see the fragment reads in the kernel)
template <int OFF>
__device__ __forceinline__ void lds_write_b128_hidden(uint32_t addr, v4i v) {
  asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(addr), "v"(v), "n"(OFF) : "memory");
}
template <int OFF>
__device__ __forceinline__ v4i lds_read_b128_hidden(uint32_t addr) {
  v4i v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
  return v;
}
__device__ __forceinline__ v4i pin(v4i v) {
  asm volatile("" : "+v"(v));
  return v;
}

// One accumulator register into a VGPR, where the caller says (as assembly: the compiler's own
// copies out of the accumulator file are all placed at the top of the epilogue).
template <int E, class V>
__device__ __forceinline__ float acc_read(const V& c) {
  float x;
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(c[E]));
  return x;
}

// The LDS map of a tile of 64 TA x 64 TB: a ring of 128-deep blocks (A rows, B rows, scales of groups A0,
// A1, B0, B1, A2 of 512 B each) and four waves' output patches.  128 x 256 and 256 x 128 tiles leave
// room for a third block: theirs is 1024 MFMA cycles, less than it takes the copies from issue
// to landing, so with one block of lead the matrix cores wait (16384 x 14336, K 4096 829 -> 778 us on
// 128 x 256, 888 -> 837 on 256 x 128; 4096 x 2048, K 2 x 6144 80 -> 76).  Their patches stage 16 rows
// instead of 32.  (The two slots of a ring of two stay numbered 0 and 1: offsets that grow by a block
// cost a dozen more additions between the MFMAs and 1 % of a long launch.)
template <int TA, int TB>
struct Lds32 {
  static constexpr int kStages = TA + TB <= 6 ? 3 : 2;
  static constexpr int kA = 64 * TA * kKB, kCodes = 64 * (TA + TB) * kKB;
  static constexpr int kBlock = kCodes + (kStages == 3 ? 2048 : 3072);
  static constexpr int kRing = kStages * kBlock;
  static constexpr int kPatchRows = kStages == 3 ? 16 : 32;
  static constexpr int kPatch = kStages == 3 ? kPatchRows * kPatchPitch : kPatch32;
  static constexpr int kBytes = kRing + 4 * kPatch;
  static_assert(kBytes <= 160 * 1024);
};
static_assert(Lds32<4, 4>::kRing == kRing32 && Lds32<4, 4>::kBlock == kBlock32, "the grouped modes' tables lie behind it");

// Two fragment sets a side, whole 128-deep blocks: a[h][t] is sub-tile TA h + t of the wave's 32 TA rows of
// A (16 rows each), b[h][t] likewise for B; the scale dwords of the block being computed (one for the even
// and one for the odd sub-tiles) and those of the next.
template <int TA, int TB>
struct Frags16 {
  v8i a[2][TA];
  v8i b[2][TB];
  uint32_t sa[2], sb[2];
  uint32_t san[2], sbn[2];
  uint32_t sa_hi[2], sb_hi[2];  // as san, sbn, of the next 128-row group (see next_scales)
};

// When a K block's LDS reads and copies are issued: everything is counted in MFMA slots of the
// block, 4 * TA * TB of them in four quarters (see block_steps).
template <int TA, int TB>
struct BlockPlan {
  static constexpr int kQ = TA * TB;                 // MFMAs of a quarter
  static constexpr int kCopies = 2 * (TA + TB) + 1;  // copies of a block and wave
  // quarter 0: the last sub-tile of a[0] (2 reads), then b[1] (2 TB): so many behind each MFMA
  static constexpr int kReads0 = 2 + 2 * TB;
  static constexpr int kQuota0 = TA == 4 && TB == 4 ? 1 : TA > 2 ? 2 : 3;
  // the ring block is released in front of the last sub-tile of a[0], whose data and b[1]'s must have arrived;
  // with two sub-tiles that is too soon after the reads, and quarter 1 begins first
  static constexpr int kRelease = TA > 2 ? TB * (TA - 1) : kQ;
  static constexpr int kFirstCopy = kRelease + 1;
  static constexpr int copy_slot(int j) { return kFirstCopy + j * (4 * kQ - kFirstCopy) / kCopies; }
  static constexpr int copy_of(int slot) {  // the copy behind this slot's MFMA (-1: none)
    for (int j = 0; j < kCopies; ++j)
      if (copy_slot(j) == slot) return j;
    return -1;
  }
  static constexpr int copies_before(int slot) {
    int n = 0;
    for (int j = 0; j < kCopies; ++j) n += copy_slot(j) < slot;
    return n;
  }
  // quarter 2: b[0] of the next block and three scale dwords, in the slots without a copy where
  // there are enough of those, else evenly
  static constexpr int kReads2 = 2 * TB + 3;
  static constexpr bool kFree2 = kQ - (copies_before(3 * kQ) - copies_before(2 * kQ)) >= kReads2;
  static constexpr int first2(int i) {  // reads of the quarter issued before slot i of it
    if (!kFree2) return (i * kReads2 + kQ - 1) / kQ;
    const int n = i - (copies_before(2 * kQ + i) - copies_before(2 * kQ));
    return n < kReads2 ? n : kReads2;
  }
  // quarter 3: reads 0 .. 2 TA - 1 are a[1]'s, 2 TA + j is read j of a[0], whose sub-tile j / 2 is
  // free behind the first MFMA of the sub-tile after it.  Entry k of the plan, in issue order.
  static constexpr int kReads3 = 2 * TA + 2 * (TA - 1);
  static constexpr int kQuota3 = TA * TB >= 2 + kReads3 || (TA == 2 && TB == 4) ? 1 : 2;
  struct Plan3 {
    int slot[kReads3], what[kReads3];
  };
  static constexpr Plan3 plan3() {
    Plan3 p{};
    int k = 0, a1 = 0, a0 = 0;
    for (int s = 0; s < kQ; ++s)
      for (int q = 0; q < kQuota3; ++q) {
        const bool have0 = a0 < 2 * (TA - 1) && s >= TB * (a0 / 2 + 1);
        if (!have0 && a1 == 2 * TA) continue;
        p.slot[k] = s;
        p.what[k++] = have0 ? 2 * TA + a0++ : a1++;
      }
    return p;
  }
  static constexpr int after_a0(int t) {  // reads of quarter 3 issued after those of a[0][t]
    const Plan3 p = plan3();
    for (int k = 0; k < kReads3; ++k)
      if (p.what[k] == 2 * TA + 2 * t + 1) return kReads3 - 1 - k;
    return 0;
  }
  static constexpr int before0(int slot) { return kQuota0 * slot < kReads0 ? kQuota0 * slot : kReads0; }
};

// A wave's columns of the tile: sub-tile n begins at column first + 16 n for n < 4 and at
// second + 16 (n - 4) from there on.  192 wide (TB = 3), the waves share the middle 64 columns and
// wave 1 takes its own 64 first, so that both write whole 128-byte lines of them.
template <int TB>
__device__ __forceinline__ constexpr uint32_t wave_col(uint32_t wn, int n) {
  if constexpr (TB == 4) return wn * 128 + 16 * n;
  if constexpr (TB == 2) return wn * 64 + 16 * n;
  return n < 4 ? wn * 128 + 16 * n : 64 + wn * 32 + 16 * (n - 4);
}

// OUT32 (kDense, one product): D is float32, its values rounded to bf16 first, as a conversion of a bf16 result
// would give them; ldd counts floats.  (Instances of their own: a branch in front of the bf16 epilogue
// made 147456 x 2048, K 2048 forward and backward 1.6 % slower.)
// GATE (kDense, 256 x 256): G = silu(A B^T) * (A B2^T), every step rounded to bf16 as the tensor operations round, leaves
// as the row-wise MXFP8 operand of the next product: of a forward without gradients nothing else is read again.  A
// tile is 256 rows of 128 columns of G: a wave's sub-tiles 0 .. 3 come from B, 4 .. 7 from the same rows of B2, so that a lane
// holds both factors of its values; waves 0 and 2 copy B's rows into the ring, 1 and 3 those of B2.  What the
// gate adds to the epilogue (8 K vector instructions a wave, matrix cores idle; 5 to 6.7 us a round over two products on the
// same tiles with their stores) is less than the 8 bytes a value that are not written and read again, and the launch: 512 x
// 14336, K 4096 59.7 us in two launches, 55.2 in this one; 1024 x 14336 108 and 102 (plan_gated for where it is not).
template <int MODE, bool PROF, bool PAIR = false, int TA = 4, int TB = 4, bool OUT32 = false, bool GATE = false>
__global__ __launch_bounds__(256, 1) void gemm_nt32_kernel(Gemm32Args p) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  static_assert(!GATE || (MODE == kDense && TA == 4 && TB == 4 && !PAIR && !OUT32));
  static_assert((TA == 4 && TB == 4) || MODE == kDense || MODE == kSplitK, "grouped tiles are 256 x 256");
  using Plan = BlockPlan<TA, TB>;
  using Frags = Frags16<TA, TB>;
  using Lds = Lds32<TA, TB>;
  constexpr int kEA = 64 * TA, kEB = GATE ? 128 : 64 * TB;  // tile edges
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 15, lj = lane >> 4;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_void_t*)smem;  // LDS byte address of the ring
  const uint32_t K = (uint32_t)p.K;  // bytes per operand row; a multiple of 128 for this kernel
#ifndef MX_ABL_ROW_PAD  // timing ablation: the rows of a tile are read this many bytes further apart than they lie
#define MX_ABL_ROW_PAD 0
#endif
  // Kp: bytes from one operand row to the next.  A pitch that is not a multiple of 4 KB spreads the
  // lines a block's copies fetch together (one K block of 512 rows) over the channels of the L2.
  const uint32_t Kp = ((MODE == kDense || MODE == kSplitK) && p.ldk ? (uint32_t)p.ldk : K) + MX_ABL_ROW_PAD;
  const int64_t Kt = (MODE == kDense || MODE == kSplitK) && p.ldk ? p.ldk : p.K;  // ... as the tile origins use it
  const uint32_t ks_n = K / kK32;    // 64-deep steps per 128-row scale group
  // tile rows / columns of one product, and of the launch (p.two: the second product's tile
  // columns or rows come behind the first's; grouped launches cover columns [tn0, tn0 + tn_cnt))
  const uint32_t tiles_n1 = (uint32_t)((p.N + kEB - 1) / kEB), tiles_m1 = (uint32_t)((p.M + kEA - 1) / kEA);
  const uint32_t tiles_n = MODE == kDense ? (p.two == kTwoB ? 2 * tiles_n1 : tiles_n1) : (uint32_t)p.tn_cnt;
  const uint32_t tiles_m = p.two == kTwoA ? 2 * tiles_m1 : tiles_m1;
  const uint32_t tn0 = MODE == kDense ? 0u : (uint32_t)p.tn0;
  const uint32_t G = (uint32_t)p.G;

  // ---- tile count.  kGrouped2d3d: group g has ceil(rows_g / 256) x tiles_n tiles; the first
  //      tile number of every group (G + 2 entries, the last group being the zero rows behind
  //      offs[G-1]) is kept in the 2 KB that wave 0's output patch leaves unused.
  bool poison = false;
  bool dealt = false;  // kGrouped2d2d: tiles dealt by length (below) instead of in tile order
  constexpr uint32_t kMaxDealt = (kPatch32 - kPatchUsed) / 4;  // two uint16 per group in wave 0's spare patch LDS
  constexpr uint32_t kMinDealt = 32;   // fewer groups than that cannot be spread evenly over 8 XCDs
  uint32_t nb;
  // "any thread saw a bad group end", through a word of wave 1's spare patch bytes (the
  // kernel's whole 160 KB are dynamic LDS: a library reduction would ask for more)
  auto any_bad = [&](int bad) -> bool {
    uint32_t* flag = reinterpret_cast<uint32_t*>(smem + kRing32 + kPatch32 + kPatchUsed);
    if (tid == 0) *flag = 0;
    __syncthreads();
    if (bad) atomicOr(flag, 1u);
    __syncthreads();
    return *flag != 0;
  };
  if constexpr (MODE == kDense) {
    nb = tiles_m * tiles_n;
  } else if constexpr (MODE == kSplitK) {
    nb = G * tiles_m * tiles_n;
  } else if constexpr (MODE == kGrouped2d2d) {
    nb = G * tiles_m * tiles_n;
    // group lengths in K blocks, kept for the dealing below (up to kMaxDealt groups)
    uint16_t* g_blocks = reinterpret_cast<uint16_t*>(smem + kRing32 + kPatchUsed);
    int bad = 0;
    for (uint32_t g = tid; g < G; g += 256) {
      const int32_t hi = p.offs[g], lo = g ? p.offs[g - 1] : 0;
      bad |= (hi & 31) | (hi < lo) | (hi > (int64_t)K) | (lo < 0);
      if (G <= kMaxDealt && G >= kMinDealt) {
        const int64_t len = hi > lo ? (((int64_t)hi + 127) >> 7) - (lo >> 7) : 0;
        g_blocks[g] = (uint16_t)(len > 0xFFFF ? 0xFFFF : len);
      }
    }
    poison = any_bad(bad);
    dealt = !poison && G <= kMaxDealt && G >= kMinDealt;
    if (dealt) {
      // position of every group in the order of falling length (ties by index): G^2 / 256
      // comparisons per thread, far below one tile's worth of time
      uint16_t* g_sorted = g_blocks + kMaxDealt;
      for (uint32_t g = tid; g < G; g += 256) {
        const uint32_t mine = g_blocks[g];
        uint32_t rank = 0;
        for (uint32_t h = 0; h < G; ++h) {
          const uint32_t o = g_blocks[h];
          rank += (o > mine) | ((o == mine) & (h < g));
        }
        g_sorted[rank] = (uint16_t)g;
      }
      __syncthreads();
    }
  } else {
    uint32_t* first = reinterpret_cast<uint32_t*>(smem + kRing32 + kPatchUsed);
    int bad = 0;
    for (uint32_t g = tid; g <= G; g += 256) {
      const int64_t lo = g ? p.offs[g - 1] : 0, hi = g < G ? (int64_t)p.offs[g] : p.M;
      bad |= (g < G && (hi & 31)) | (hi < lo) | (hi > p.M) | (lo < 0);
      const int64_t rows = hi > lo ? hi - lo : 0;
      first[g + 1] = (uint32_t)((rows + kT32 - 1) / kT32) * tiles_n;
    }
    poison = any_bad(bad);
    if (tid < 64) {  // inclusive prefix sum of first[1 .. G+1] by wave 0, 10 entries per lane
      uint32_t sum = 0;
      for (uint32_t g = 1 + (uint32_t)tid * 10; g < 11 + (uint32_t)tid * 10 && g <= G + 1; ++g) sum += first[g];
      uint32_t incl = sum;
      for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(incl, d);
        if (tid >= d) incl += o;
      }
      uint32_t run = incl - sum;
      for (uint32_t g = 1 + (uint32_t)tid * 10; g < 11 + (uint32_t)tid * 10 && g <= G + 1; ++g) {
        run += first[g];
        first[g] = run;
      }
      if (tid == 0) first[0] = 0;
    }
    __syncthreads();
    nb = first[G + 1];
    if (poison) nb = tiles_m * tiles_n;  // then: NaN over all of D
  }

  // ---- this workgroup's tile list: XCD x (= blockIdx % 8) owns one contiguous run of tiles,
  //      its workgroups take them round-robin, so the XCD's CUs work on neighbouring tiles
  const uint32_t wgs_per_xcd = gridDim.x / 8;
  const uint32_t xcd = blockIdx.x % 8, idx = blockIdx.x / 8;
  const uint32_t per_xcd = (nb + 7) / 8;
  const uint32_t t_lo = xcd * per_xcd + idx;
  const uint32_t t_hi = (xcd + 1) * per_xcd < nb ? (xcd + 1) * per_xcd : nb;
  uint32_t n_my = t_lo < t_hi ? (t_hi - t_lo + wgs_per_xcd - 1) / wgs_per_xcd : 0;
  // kGrouped2d2d with uneven groups: a tile's time goes with its group's length, so tiles taken
  // in tile order leave the workgroups with sums that differ by a fifth and more.  Instead the
  // groups, in order of falling length, are dealt to the XCDs back and forth (j-th group of XCD
  // x = position 8j + x or 8j + 7 - x), which keeps the tiles of a group, and their operand
  // panels, inside one L2; and the tiles of an XCD's groups, still in that order, are dealt to
  // its workgroups back and forth in the same way: every workgroup gets one tile from each band
  // of neighbouring lengths.
  auto snake = [](uint32_t band, uint32_t k, uint32_t width) -> uint32_t {
    return (band & 1) ? width - 1 - k : k;
  };
  const uint32_t per_g2 = tiles_m * tiles_n;  // tiles of one group
  if (MODE == kGrouped2d2d && dealt) {
    const uint32_t full = G / 8, rest = G % 8;
    const uint32_t groups_x = full + (snake(full, xcd, 8) < rest ? 1 : 0);
    const uint32_t tiles_x = groups_x * per_g2;
    const uint32_t bands = tiles_x / wgs_per_xcd, tail = tiles_x % wgs_per_xcd;
    n_my = bands + (snake(bands, idx, wgs_per_xcd) < tail ? 1 : 0);
  }
  if (n_my == 0) return;
  if (PAIR) n_my *= 2;  // from here on n_my counts segments: two per output tile
  if (MODE != kDense && n_my > kMaxTileRecords) {
    // More tiles than records: the host splits launches so that this cannot happen.  Should it
    // ever, the tiles that have a record are written as NaN rather than left as they were.
    n_my = kMaxTileRecords;
    poison = true;
  }

  // Tile number -> operands.
  auto describe = [&](uint32_t t, uint32_t seg) -> Tile32 {
    Tile32 r;
    r.poison = poison;
    r.koff = 0;
    r.empty = false;
    r.rows_d = 0;
    r.rot = 0;
    r.odd = 0;
    r.tm = r.tn = 0;
    r.head = 0;
    r.tail = 0;
    const uint8_t* a_codes = (PAIR && seg) ? p.a2_codes : p.a_codes;
    const uint8_t* a_scales = (PAIR && seg) ? p.a2_scales : p.a_scales;
    const uint8_t* b_codes = (PAIR && seg) ? p.b2_codes : p.b_codes;
    const uint8_t* b_scales = (PAIR && seg) ? p.b2_scales : p.b_scales;
    uint16_t* d_base = p.d;
    // p.two: a tile column / row of the second product becomes that product's own, with its
    // operand and output in place of the first's
    auto second_product = [&](uint32_t& tm, uint32_t& tn) {
      if constexpr (!PAIR && (MODE == kDense || MODE == kGrouped2d3d || MODE == kGrouped2d2d)) {
        if (p.two == kTwoB && tn >= tiles_n1) {
          tn -= tiles_n1;
          b_codes = p.b2_codes;
          b_scales = p.b2_scales;
          d_base = p.d2;
        }
        if (p.two == kTwoA && tm >= tiles_m1) {
          tm -= tiles_m1;
          a_codes = p.a2_codes;
          a_scales = p.a2_scales;
          d_base = p.d2;
        }
      }
    };
    uint32_t tm, tn;
    if (MODE == kDense || (MODE == kGrouped2d3d && poison)) {
      tile_coords(t, tiles_m, tiles_n, tm, tn);
      tn += tn0;
      second_product(tm, tn);
#if defined(MX_ABL_SAME_PANEL)  // timing ablation: every 8 x 4 round reads the same twelve operand panels
      r.a = a_codes + (int64_t)(tm & 7) * kT32 * K;
      r.b = b_codes + (int64_t)(tn & 3) * kT32 * K;
#elif defined(MX_ABL_SAME_A)  // ... the same eight A panels only
      r.a = a_codes + (int64_t)(tm & 7) * kT32 * K;
      r.b = b_codes + (int64_t)tn * kT32 * K;
#elif defined(MX_ABL_SAME_B)  // ... the same four B panels only
      r.a = a_codes + (int64_t)tm * kT32 * K;
      r.b = b_codes + (int64_t)(tn & 3) * kT32 * K;
#else
      r.a = a_codes + (int64_t)tm * kEA * Kt;
      r.b = b_codes + (int64_t)tn * kEB * Kt;
#endif
      r.sa = a_scales + (int64_t)(tm * kEA / 128) * ks_n * 256;
      r.sb = b_scales + (int64_t)(tn * kEB / 128) * ks_n * 256;
      r.d = d_base + (((int64_t)tm * kEA * p.ldd + (int64_t)tn * kEB) << (OUT32 ? 1 : 0));
      r.rows_a = p.M - (int64_t)tm * kEA;
      r.rows_b = p.N - (int64_t)tn * kEB;
      r.odd = (tm & 1) | (tn & 1) << 1;
      if constexpr (GATE) {
        r.tm = tm;
        r.tn = tn;
      }
      if (MODE == kGrouped2d3d && p.d_offs) {
        const int64_t left = p.d_rows - (int64_t)tm * kT32;
        r.rows_d = (int32_t)(left < 0 ? 0 : (left > kT32 ? kT32 : left));
      }
      r.nblocks = poison ? 1 : K / kKB;
      r.empty = poison;
    } else if (MODE == kGrouped2d3d) {
      const uint32_t* first = reinterpret_cast<const uint32_t*>(smem + kRing32 + kPatchUsed);
      uint32_t g = 0, hi_g = G + 1;  // first[g] <= t < first[g + 1]
      while (hi_g - g > 1) {
        const uint32_t mid = (g + hi_g) >> 1;
        if (first[mid] <= t) g = mid; else hi_g = mid;
      }
      const int64_t lo = g ? p.offs[g - 1] : 0, hi = g < G ? (int64_t)p.offs[g] : p.M;
      const uint32_t tiles_mg = (uint32_t)((hi - lo + kT32 - 1) / kT32);
      tile_coords(t - first[g], tiles_mg, tiles_n, tm, tn);
      tn += tn0;
      second_product(tm, tn);
      const int64_t row0 = lo + (int64_t)tm * kT32;
      const uint32_t gb = g < G ? g : 0;  // the zero rows have no expert: any valid address
      r.a = a_codes + row0 * K;
      r.b = b_codes + ((int64_t)gb * p.N + (int64_t)tn * kT32) * K;
      r.sa = a_scales + (row0 >> 7) * ks_n * 256;
      r.rot = (uint32_t)(row0 >> 5) & 3;
      r.sb = b_scales + ((int64_t)gb * ((p.N + 127) >> 7) + tn * 2) * ks_n * 256;
      r.d = d_base + row0 * p.ldd + (int64_t)tn * kT32;
      r.rows_a = hi - row0;
      r.rows_b = p.N - (int64_t)tn * kT32;
      if (p.d_offs) {  // the group's rows in D, both ends kept inside D whatever the array holds
        int64_t lo_d = g ? p.d_offs[g - 1] : 0, hi_d = g < G ? (int64_t)p.d_offs[g] : p.d_rows;
        lo_d = lo_d < 0 ? 0 : (lo_d > p.d_rows ? p.d_rows : lo_d);
        hi_d = hi_d < lo_d ? lo_d : (hi_d > p.d_rows ? p.d_rows : hi_d);
        const int64_t left = hi_d - lo_d - (int64_t)tm * kT32;
        r.rows_d = (int32_t)(left < 0 ? 0 : (left > kT32 ? kT32 : left));
        r.d = d_base + (lo_d + (int64_t)tm * kT32) * p.ldd + (int64_t)tn * kT32;
      }
      r.nblocks = g < G ? K / kKB : 1;
      r.empty = g >= G;
    } else if (MODE == kSplitK) {
      // slice g of the K blocks: ceil(blocks / slices) each, the host picks the number so that none is empty
      const uint32_t per_g = tiles_m * tiles_n;
      const uint32_t g = t / per_g;
      tile_coords(t - g * per_g, tiles_m, tiles_n, tm, tn);
      const uint32_t slices = G / (uint32_t)p.sets, slice = g % slices;
      if (g >= slices) {
        a_codes = p.a2_codes;
        a_scales = p.a2_scales;
        b_codes = p.b2_codes;
        b_scales = p.b2_scales;
      }
      const uint32_t blocks = K / kKB, per = (blocks + slices - 1) / slices;
      const uint32_t b_lo = slice * per, b_hi = b_lo + per < blocks ? b_lo + per : blocks;
      const uint32_t lo = b_lo * kKB;
      r.a = a_codes + (int64_t)tm * kEA * Kt + lo;
      r.b = b_codes + (int64_t)tn * kEB * Kt + lo;
      r.sa = a_scales + ((int64_t)(tm * kEA / 128) * ks_n + (lo >> 6)) * 256;
      r.sb = b_scales + ((int64_t)(tn * kEB / 128) * ks_n + (lo >> 6)) * 256;
      float* part = reinterpret_cast<float*>(p.d) +
                    ((int64_t)g * p.M + (int64_t)tm * kEA) * p.ldd + (int64_t)tn * kEB;
      r.d = reinterpret_cast<uint16_t*>(part);
      r.rows_a = p.M - (int64_t)tm * kEA;
      r.rows_b = p.N - (int64_t)tn * kEB;
      r.odd = (tm & 1) | (tn & 1) << 1;
      r.koff = lo;
      r.nblocks = b_hi - b_lo;
    } else {
      const uint32_t per_g = tiles_m * tiles_n;
      uint32_t g = t / per_g, in_g = t - g * per_g;
      if (dealt) {  // t counts this workgroup's tiles: the i-th tile it was dealt
        const uint16_t* g_sorted = reinterpret_cast<const uint16_t*>(smem + kRing32 + kPatchUsed) + kMaxDealt;
        const uint32_t q = wgs_per_xcd * t + snake(t, idx, wgs_per_xcd);  // place in the XCD's tile list
        const uint32_t j = q / per_g;
        in_g = q - j * per_g;
        g = g_sorted[8 * j + snake(j, xcd, 8)];
      }
      tile_coords(in_g, tiles_m, tiles_n, tm, tn);
      tn += tn0;
      second_product(tm, tn);
      const int64_t lo = poison ? 0 : (g ? p.offs[g - 1] : 0), hi = poison ? 0 : p.offs[g];
      // the K blocks keep to multiples of 128 (whole cache lines per operand row: a copy that
      // straddles two lines costs the texture path twice); a range that starts or ends inside
      // a block has the 32-deep blocks outside it masked (head, tail)
      const int64_t lo128 = lo & ~(int64_t)127;
      r.a = a_codes + (int64_t)tm * kT32 * K + lo128;
      r.b = b_codes + (int64_t)tn * kT32 * K + lo128;
      r.sa = a_scales + ((int64_t)(tm * 2) * ks_n + (lo128 >> 6)) * 256;
      r.sb = b_scales + ((int64_t)(tn * 2) * ks_n + (lo128 >> 6)) * 256;
      r.d = d_base + ((int64_t)g * p.M + (int64_t)tm * kT32) * p.ldd + (int64_t)tn * kT32;
      r.rows_a = p.M - (int64_t)tm * kT32;
      r.rows_b = p.N - (int64_t)tn * kT32;
      r.koff = (uint32_t)lo128;
      r.nblocks = hi > lo ? (uint32_t)(((hi + 127) >> 7) - (lo >> 7)) : 0;
      r.head = (uint32_t)(lo >> 5) & 3;
      r.tail = (uint32_t)(hi >> 5) & 3;
      if (r.nblocks == 0) {
        r.nblocks = 1;
        r.empty = true;
      }
    }
    return r;
  };

  // Grouped modes: the map needs loads of the group ends and a search, far too slow for the
  // in-order instruction stream of the MFMA waves.  Every thread works out one of this
  // workgroup's tiles up front and leaves a 64-byte record in the spare 2 KB behind the
  // output patches of waves 1-3 (32 records each; the host splits launches so that a
  // workgroup never has more than kMaxRecords tiles).
  auto record_offset = [&](uint32_t i) -> uint32_t {
    if constexpr (MODE == kSplitK) return Lds::kRing + i * 64;  // (its output is not staged: the patches are free)
    return kRing32 + (1 + i / kRecordsPerPatch) * kPatch32 + kPatchUsed + (i % kRecordsPerPatch) * 64;
  };
  if constexpr (MODE != kDense) {
    for (uint32_t i = tid; i < n_my; i += 256) {
      const uint32_t ti = PAIR ? i >> 1 : i;  // PAIR: records 2t and 2t+1 are the two segments of tile t
      const Tile32 t = describe((MODE == kGrouped2d2d && dealt) ? ti : t_lo + ti * wgs_per_xcd, PAIR ? i & 1 : 0);
      uint64_t* q = reinterpret_cast<uint64_t*>(smem + record_offset(i));
      q[0] = (uint64_t)(uintptr_t)t.a;
      q[1] = (uint64_t)(uintptr_t)t.b;
      q[2] = (uint64_t)(uintptr_t)t.sa;
      q[3] = (uint64_t)(uintptr_t)t.sb;
      q[4] = (uint64_t)(uintptr_t)t.d;
      int32_t* w = reinterpret_cast<int32_t*>(q + 5);
      w[0] = (int32_t)(t.rows_a > 0x7FFFFFFF ? 0x7FFFFFFF : t.rows_a);
      w[1] = (int32_t)(t.rows_b > 0x7FFFFFFF ? 0x7FFFFFFF : t.rows_b);
      w[2] = (int32_t)t.nblocks;
      w[3] = (int32_t)t.koff;
      w[4] = t.empty ? 1 : 0;
      w[5] = (int32_t)(t.rot | (t.odd << 4) | (t.tail << 8) | (t.head << 16) | ((uint32_t)t.rows_d << 20));
    }
    __syncthreads();
  }
  // this workgroup's i-th tile (records are read so that the compiler's wait-count model
  // does not see an LDS read, see the fragment reads; every lane reads the same 64 bytes)
  auto get_tile = [&](uint32_t i) -> Tile32 {
    if constexpr (MODE == kDense) {
      return describe(t_lo + (PAIR ? i >> 1 : i) * wgs_per_xcd, PAIR ? i & 1 : 0);
    } else {
      const uint32_t addr = lds_base + record_offset(i);
      v4i r0, r1, r2, r3;
      asm volatile(
          "ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:16\n\tds_read_b128 %2, %4 offset:32\n\t"
          "ds_read_b128 %3, %4 offset:48\n\ts_waitcnt lgkmcnt(0)"
          : "=&v"(r0), "=&v"(r1), "=&v"(r2), "=&v"(r3)
          : "v"(addr)
          : "memory");
      auto u64 = [](int lo, int hi) -> uint64_t {
        return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane(lo) |
               ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane(hi) << 32);
      };
      Tile32 t;
      t.a = (const uint8_t*)(uintptr_t)u64(r0.x, r0.y);
      t.b = (const uint8_t*)(uintptr_t)u64(r0.z, r0.w);
      t.sa = (const uint8_t*)(uintptr_t)u64(r1.x, r1.y);
      t.sb = (const uint8_t*)(uintptr_t)u64(r1.z, r1.w);
      t.d = (uint16_t*)(uintptr_t)u64(r2.x, r2.y);
      t.rows_a = __builtin_amdgcn_readfirstlane(r2.z);
      t.rows_b = __builtin_amdgcn_readfirstlane(r2.w);
      t.nblocks = (uint32_t)__builtin_amdgcn_readfirstlane(r3.x);
      t.koff = (uint32_t)__builtin_amdgcn_readfirstlane(r3.y);
      t.empty = __builtin_amdgcn_readfirstlane(r3.z) != 0;
      const uint32_t rt = (uint32_t)__builtin_amdgcn_readfirstlane(r3.w);
      t.rot = rt & 3;
      t.odd = (rt >> 4) & 3;
      t.tail = (rt >> 8) & 3;
      t.head = (rt >> 16) & 3;
      t.rows_d = (int32_t)(rt >> 20);
      t.poison = poison;
      return t;
    }
  };

  // ---- per-lane constants
  // global -> LDS: a load unit is 8 rows x 128 B; lane l fetches row l/8 and the logical 16-byte
  // chunk that belongs at physical chunk l%8 of that row:
  // c = (l%8) ^ ((row & 2) | ((row & 8) >> 1)), see the fragment reads
  const uint32_t c_even = (lane & 7) ^ ((lane >> 3) & 2);
  const uint32_t v_even = (uint32_t)(lane >> 3) * Kp + c_even * 16;
  // (odd units: v_even ^ 64 -- K is a multiple of 128, so bit 6 belongs to the chunk alone)
  // LDS -> VGPR: lane (li = l & 15, lj = l >> 4) of a 16-row sub-tile reads chunks lj and lj + 4 of
  // row li (K bytes [16 lj, +16) and [64 + 16 lj, +16)); physical chunk = logical ^ sw with
  // sw = (row & 2) | ((row & 8) >> 1), which spreads the 16 lanes of every b128 pass (lanes
  // {0-3, 12-15, 20-23, 24-27} and {4-11, 16-19, 28-31} of a half-wave) over all bank groups;
  // the second chunk is address ^ 64.  Scales: sub-tile m needs row 16m + li, 32-deep block lj,
  // i.e. 64-deep step lj >> 1, lane 32 (lj & 1) + 16 (m & 1) + li of the 128-row group, byte
  // m >> 1: one dword for the even sub-tiles, the one 64 bytes on for the odd ones.
  const uint32_t sw = (li & 2) | ((li & 8) >> 1);
  const uint32_t lane4 = (uint32_t)(lj >> 1) * 256 + (uint32_t)((lj & 1) * 32 + li) * 4;
  const uint32_t fa0 = (wm * 32 * TA + li) * kKB + ((lj ^ sw) << 4);
  // sub-tiles 0..3 and 4.. of B (see wave_col), from the place of A's first
  const uint32_t fb_delta = Lds::kA + (wave_col<TB>(wn, 0) - wm * 32 * TA) * kKB;
  const uint32_t fb_delta4 = TB == 3 ? Lds::kA + (wave_col<TB>(wn, 4) - 64 - wm * 32 * TA) * kKB : fb_delta;
  // scale copy: lanes 0-31 fetch one 128-row group's 512 bytes of a block, lanes 32-63 the next
  // group's; wave 1 (kGrouped2d3d: a third group of A) has its upper lanes read nothing
  const uint32_t v_scale = (MODE == kGrouped2d3d && wave == 1) || (GATE && wave >= 2)
                               ? (lane < 32 ? (uint32_t)lane * 16 : 0x80000000u)
                               : (uint32_t)(lane >> 5) * ks_n * 256 + (lane & 31) * 16;
  // scale groups of a ring block: A0, A1, B0, B1, A2 (512 bytes each, then 512 unused)
  // (GATE: B's group in place of B0, B2's in place of A2, zeros behind either)
  const uint32_t scale_dst = Lds::kCodes + ((MODE == kGrouped2d3d && wave == 1) || (GATE && wave == 3) ? 2048u : (uint32_t)(wave >> 1) * 1024u);
  // 256 rows: a wave has a scale group of its own (kGrouped2d3d: and the next one, see next_scales);
  // 192: three of the eight bytes of two groups; 128: half of the bytes of one
  const uint32_t fsa_s = Lds::kCodes + (TA == 4 ? wm * 512 : 0), fsb_s = Lds::kCodes + 1024 + (TB == 4 && !GATE ? wn * 512 : 0);
  const uint32_t fsa_hi_s = Lds::kCodes + (TA == 4 && wm != 0 ? 2048 : 512), fsb_hi_s = Lds::kCodes + (GATE ? 2048 : 1536);

  // ---- loader stream: fills ring block `ld_slot` with K block `ld_kb` of tile `ld_tile`
  uint32_t ld_tile = 0, ld_kb = 0, ld_nb = 1;
  int ld_slot = 0;
  auto next_slot = [](int slot) -> int {
    if constexpr (Lds::kStages == 2) return slot ^ 1;
    return slot == Lds::kStages - 1 ? 0 : slot + 1;
  };
  __amdgpu_buffer_rsrc_t ra, rb, rs;  // codes of A, codes of B, scales this wave copies
  // kGrouped2d3d: a group may start at any multiple of 32 rows, the scales come in 128-row groups
  // of the whole matrix: a tile that starts `rot` 32-row blocks into a group fetches three groups
  // and turns the bytes of every scale dword by `rot` (next_scales).  The rotation belongs to
  // the tile whose block sits in a ring slot.
  uint32_t ld_rot = 0, slot_rot0 = 0, slot_rot1 = 0;  // (192-row tiles: Tile32::odd)
  // kGrouped2d2d: a K range may start and end at any multiple of 32.  Its first and last
  // 128-deep blocks send the chunks outside the range out of range, so that zeros land in the
  // ring instead of the neighbouring groups' codes and scales.
  uint32_t ld_head = 0, ld_tail = 0;
  uint32_t cur_v_even = v_even, cur_v_odd = v_even ^ 64, cur_v_scale = v_scale;
  auto set_block_offsets = [&]() {
    if constexpr (MODE == kGrouped2d2d) {
      // 32-deep blocks [first, lim) of this 128-deep block are fetched
      const uint32_t first = ld_kb == 0 ? ld_head : 0;
      const uint32_t lim = (ld_tail != 0 && ld_kb + 1 == ld_nb) ? ld_tail : 4;
      auto inside = [&](uint32_t blk) { return blk >= first && blk < lim; };
      cur_v_even = inside(c_even >> 1) ? v_even : 0x80000000u;
      cur_v_odd = inside((c_even ^ 4) >> 1) ? (v_even ^ 64) : 0x80000000u;
      cur_v_scale = inside((uint32_t)(lane & 31) >> 3) ? v_scale : 0x80000000u;
    }
  };
  auto loader_open_tile = [&]() {
    if (ld_tile < n_my) {
      const Tile32 t = get_tile(ld_tile);
      ld_nb = t.nblocks;
      ld_rot = MODE == kGrouped2d3d ? t.rot : t.odd;
      ld_head = t.head;
      ld_tail = t.tail;
      // (kGrouped2d2d: the range stops at the end of the operand rows, not of the K range;
      //  the K range is exact because nblocks is.)  A tile without a K range reads nothing:
      // its one block arrives as zeros, scales included.
      const bool none = MODE != kDense && t.empty;
      ra = make_rsrc(t.a, none ? 0 : t.rows_a * (int64_t)Kp - t.koff);
      if constexpr (GATE) {  // this wave's 64 rows: of B or of B2
        const uint8_t* from = (wave & 1 ? p.b2_codes + (t.b - p.b_codes) : t.b) + (int64_t)(wave >> 1) * 64 * Kp;
        rb = make_rsrc(from, (t.rows_b - (wave >> 1) * 64) * (int64_t)Kp);
      } else
        rb = make_rsrc(t.b, none ? 0 : t.rows_b * (int64_t)Kp - t.koff);
      // wave 0 copies the scales of A's two 128-row groups, wave 2 those of B's (one copy per
      // block each: lanes 0-31 fetch group 0, lanes 32-63 group 1); a group beyond the operand
      // is cut off by the range and arrives as zeros
      // (kGrouped2d3d: rows counted from the start of the first scale group; wave 1 copies a
      // third group of A when the tile's rows reach into it)
      // (192-row tiles: likewise, 64 rows into the group for every other tile)
      const int64_t into_a = TA == 3 ? 64 * (int64_t)(t.odd & 1) : 32 * (int64_t)t.rot;
      const int64_t into_b = TB == 3 ? 64 * (int64_t)(t.odd >> 1) : 0;
      const int64_t rows = wave < 2 ? (t.rows_a > 0 ? t.rows_a + into_a : 0) : t.rows_b > 0 ? t.rows_b + into_b : 0;
      const uint8_t* sbase = wave < 2 ? t.sa : GATE && wave == 3 ? p.b2_scales + (t.sb - p.b_scales) : t.sb;
      if (MODE == kGrouped2d3d && wave == 1)
        rs = make_rsrc(sbase + (int64_t)ks_n * 512, (none || rows <= 256) ? 0 : (int64_t)ld_nb * 512);
      else
        rs = make_rsrc(sbase, none ? 0
                                   : rows > 128 ? (int64_t)ks_n * 256 + (int64_t)ld_nb * 512
                                                : (rows > 0 ? (int64_t)ld_nb * 512 : 0));
    } else {  // past the last tile: every lane reads out of range (zeros, no traffic)
      ld_nb = 1;
      ld_rot = 0;
      ld_head = 0;
      ld_tail = 0;
      ra = make_rsrc(p.a_codes, 0);
      rb = ra;
      rs = ra;
    }
    set_block_offsets();
  };
#ifndef MX_LOAD_AUX  // cache policy bits of the operand copies (0: default)
#define MX_LOAD_AUX 0
#endif
  // The copies of a block (17 of a 256 x 256 tile) are issued one at a time, between MFMAs (see
  // block_steps): units of A and of B alternating as long as there are both, scales last, then advance.
  auto issue_piece = [&](auto i_) {
    constexpr int i = decltype(i_)::value;
#ifdef MX_ABL_DMA_OOB  // timing ablation: every copy is issued with all lanes out of range (zeros land in LDS, nothing is fetched)
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.a_codes, 0), rb = ra, rs = ra;
#endif

    const uint32_t sbase = lds_base + ld_slot * Lds::kBlock;
    if constexpr (i < 2 * (TA + TB)) {
      constexpr int kBoth = 4 * (TA < TB ? TA : TB);
      constexpr bool is_a = i < kBoth ? (i & 1) == 0 : TA > TB;
      constexpr int q = i < kBoth ? i >> 1 : i - kBoth / 2;
      const int unit = wave * 2 * (is_a ? TA : TB) + q;
      const uint32_t v = MODE == kGrouped2d2d ? ((q & 1) ? cur_v_odd : cur_v_even)
                                              : ((q & 1) ? (v_even ^ 64) : v_even);
      const uint32_t so = (uint32_t)((GATE && !is_a ? q : unit) * 8) * Kp + ld_kb * kKB;
      if constexpr (is_a)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void_t*)(uintptr_t)(sbase + unit * 1024), 16, v, so, 0, MX_LOAD_AUX);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rb, (lds_void_t*)(uintptr_t)(sbase + Lds::kA + unit * 1024), 16, v, so, 0, MX_LOAD_AUX);
    } else {
      // scales: a group's two 64-deep steps are 512 contiguous bytes, the two groups land behind
      // one another, which is the order the fragment reads expect.  Waves 0 and 2 copy A's and
      // B's; waves 1 and 3 copy the same bytes to the same place once more (kGrouped2d3d: wave 1
      // the third group of A instead): every wave then runs the same instructions, where a
      // branch around the copy costs the two waves that take it more than the copy itself
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rs, (lds_void_t*)(uintptr_t)(sbase + scale_dst), 16,
          MODE == kGrouped2d2d ? cur_v_scale : v_scale, ld_kb * 512, 0, 0);
    }
  };
  auto issue_advance = [&]() {
    if constexpr (MODE == kGrouped2d3d || TA == 3 || TB == 3) {
      if (ld_slot) slot_rot1 = ld_rot; else slot_rot0 = ld_rot;
    }
    if (++ld_kb == ld_nb) {
      ld_kb = 0;
      ++ld_tile;
      loader_open_tile();
    } else {
      set_block_offsets();
    }
    ld_slot = next_slot(ld_slot);
  };
  auto issue_block = [&]() {
    static_for<0, Plan::kCopies>([&](auto i_) { issue_piece(i_); });
    issue_advance();
  };

  // Fragment reads are issued as inline assembly: the compiler cannot tell which ring block a
  // ds_read touches, so for reads it can see it waits until every global->LDS copy in flight
  // has landed (vmcnt(0)) and the prefetch distance collapses.  The reads are therefore
  // invisible to its wait-count tracking; `pin_set` / `landed` (after an explicit lgkmcnt wait)
  // are what the MFMAs depend on.
#ifdef MX_ABL_TR_READ
  constexpr int kReadsPerPiece = 2;
#else
  constexpr int kReadsPerPiece = 1;
#endif
  auto lds_b128 = [&](uint32_t addr, auto off_) -> v4i {
    constexpr int off = decltype(off_)::value;
    v4i v;
#ifdef MX_ABL_TR_READ  // timing ablation: the 16 bytes come as two transposing 8-byte reads
    typedef int v2i_t __attribute__((ext_vector_type(2)));
    v2i_t lo, hi;
    const uint32_t first = addr + ((lane & 16) >> 1);  // each 32-lane pass still covers all banks
    asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(lo) : "v"(first), "n"(off));
    asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(hi) : "v"(first ^ 8u), "n"(off));
    v = v4i{lo.x, lo.y, hi.x, hi.y};
#else
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(off));
#endif
    return v;
  };
  // ---- fragment sets, scale dwords
  // one b128 read of a fragment set: i = 2t + (0: K bytes [16 lj, +16), 1: [64 + 16 lj, +16)) of
  // the set's sub-tile t, which is sub-tile m of the wave
  auto read_piece = [&](v8i& dst, uint32_t sbase, uint32_t delta, auto m_, auto i_) {
    constexpr int m = decltype(m_)::value;
    constexpr bool hi = decltype(i_)::value & 1;
    const uint32_t base = (fa0 ^ (hi ? 64u : 0u)) + delta;
    const v4i v = lds_b128(sbase + base, std::integral_constant<int, m * 2048>{});
    if constexpr (hi) {
      dst[4] = v.x; dst[5] = v.y; dst[6] = v.z; dst[7] = v.w;
    } else {
      dst[0] = v.x; dst[1] = v.y; dst[2] = v.z; dst[3] = v.w;
    }
  };
  auto read_a = [&](Frags& f, uint32_t sbase, auto h_, auto i_) {
    constexpr int h = decltype(h_)::value, t = decltype(i_)::value >> 1;
    read_piece(f.a[h][t], sbase, 0u, std::integral_constant<int, TA * h + t>{}, i_);
  };
  auto read_b = [&](Frags& f, uint32_t sbase, auto h_, auto i_) {
    constexpr int h = decltype(h_)::value, t = decltype(i_)::value >> 1, n = TB * h + t;
    read_piece(f.b[h][t], sbase, n < 4 ? fb_delta : fb_delta4, std::integral_constant<int, n>{}, i_);
  };
  // the scale dwords of a block, into the "next" registers: piece 0, 1 = A even / odd
  // sub-tiles, 2, 3 = B, then those of the next 128-row group of A (kGrouped2d3d, 192 rows) and of
  // B (192 columns)
  constexpr bool kHiA = MODE == kGrouped2d3d || TA == 3, kHiB = TB == 3 || GATE;
  constexpr int kScalePieces = 4 + (kHiA ? 2 : 0) + (kHiB ? 2 : 0);
  auto read_scale_piece = [&](Frags& f, uint32_t sbase, auto i_) {
    constexpr int i = decltype(i_)::value;
    constexpr int e = i & 1;
    if constexpr (i < 2) {
      const uint32_t ps = sbase + fsa_s + lane4 + e * 64;
      asm volatile("ds_read_b32 %0, %1" : "=v"(f.san[e]) : "v"(ps));
    } else if constexpr (i < 4) {
      const uint32_t ps = sbase + fsb_s + lane4 + e * 64;
      asm volatile("ds_read_b32 %0, %1" : "=v"(f.sbn[e]) : "v"(ps));
    } else if constexpr (kHiA && i < 6) {
      const uint32_t ps = sbase + fsa_hi_s + lane4 + e * 64;
      asm volatile("ds_read_b32 %0, %1" : "=v"(f.sa_hi[e]) : "v"(ps));
    } else {
      const uint32_t ps = sbase + fsb_hi_s + lane4 + e * 64;
      asm volatile("ds_read_b32 %0, %1" : "=v"(f.sb_hi[e]) : "v"(ps));
    }
  };
  auto pin_set = [&](auto& set) {
    for (auto& frag : set) asm volatile("" : "+v"(frag));
  };
  // The next block's scales become the current ones, once their reads have landed.
  // kGrouped2d3d: byte k of an A scale dword becomes the scale of the tile's k-th 32-row block,
  // which is byte (rot + k) of the eight bytes that two neighbouring 128-row groups hold for
  // this lane
  // 192 rows: a tile's six 32-row blocks are bytes 0..5 or, every other tile, 2..7 of the eight of
  // its two groups; three of them, in the order of the wave's sub-tiles, are picked.
  // 128 rows: the upper wave's two bytes are brought down.
  auto next_scales = [&](Frags& f, int slot) {
    asm volatile("" : "+v"(f.san[0]), "+v"(f.san[1]), "+v"(f.sbn[0]), "+v"(f.sbn[1]));
    if constexpr (kHiA) asm volatile("" : "+v"(f.sa_hi[0]), "+v"(f.sa_hi[1]));
    if constexpr (kHiB) asm volatile("" : "+v"(f.sb_hi[0]), "+v"(f.sb_hi[1]));
    const uint32_t rot = slot ? slot_rot1 : slot_rot0;
    static_for<0, 2>([&](auto e_) {
      constexpr int e = decltype(e_)::value;
      if constexpr (MODE == kGrouped2d3d) f.sa[e] = __builtin_amdgcn_alignbyte(f.sa_hi[e], f.san[e], rot);
      else if constexpr (TA == 3) {
        const uint32_t sel = (wm ? 0x00050403u : 0x00020100u) + ((rot & 1) ? 0x00020202u : 0u);
        f.sa[e] = __builtin_amdgcn_perm(f.sa_hi[e], f.san[e], sel);
      } else if constexpr (TA == 2) f.sa[e] = f.san[e] >> (16 * wm);
      else f.sa[e] = f.san[e];
      if constexpr (TB == 3) {
        const uint32_t sel = (wn ? 0x00030504u : 0x00020100u) + ((rot & 2) ? 0x00020202u : 0u);
        f.sb[e] = __builtin_amdgcn_perm(f.sb_hi[e], f.sbn[e], sel);
      } else if constexpr (GATE) {  // sub-tiles 0 .. 3: two of B's four 32-row blocks, 4 .. 7: the same two of B2's
        f.sb[e] = __builtin_amdgcn_perm(f.sb_hi[e], f.sbn[e], wn ? 0x07060302u : 0x05040100u);
      } else if constexpr (TB == 2) f.sb[e] = f.sbn[e] >> (16 * wn);
      else f.sb[e] = f.sbn[e];
    });
  };
  // ---- compute stream
  v4f acc[2 * TA][2 * TB];
  int c_slot = 0;  // ring block holding the K block being computed
  uint64_t prof_vm = 0, prof_bar = 0, prof_body = 0, prof_last = 0, prof_epi = 0;
  uint64_t prof_e_stage = 0, prof_e_wait = 0, prof_e_store = 0;

// Output stores carry the nontemporal policy bit: written once, never re-read by this kernel,
// and without it the output lines displace operand panels in L2 and the copies of the next
// tile's first blocks queue behind the draining stores.
#ifndef MX_STORE_AUX
#define MX_STORE_AUX 2
#endif
  // A K block of a 256x256 tile is 64 MFMAs, one per 16x16 sub-tile, in four quarters of 16 (512 MFMA cycles each)
  // over the fragment sets a[0], a[1] (rows 0-63, 64-127 of the wave) and b[0], b[1], in an
  // order that needs every set for two quarters in a row (slots 0-63 = the block's MFMAs; for
  // the smaller tiles, whose sets hold TA and TB sub-tiles, BlockPlan has the slots):
  //   quarter 0: a[0] x b[0], a[0]'s sub-tiles one after the other.  Read meanwhile, from this
  //              block: the last sub-tile of a[0] (slots 0, 1; used from slot 12) and b[1]
  //              (2-9).  Once every wave has done so (barrier in front of slot kRelease) the
  //              ring block is free and the copies of block b+2 start, one every third slot
  //              (the copy unit takes about 20 cycles per copy for each of the four waves)
  //   quarter 1: a[1] x b[0]
  //   quarter 2: a[1] x b[1].  Block b+1 must have landed (wait, barrier); its b[0] and scales
  //              are read
  //   quarter 3: a[0] x b[1], a[0]'s sub-tiles one after the other.  a[1] takes block b+1's data,
  //              and so does a sub-tile of a[0] as soon as an MFMA of the next sub-tile has been
  //              issued (slots 52/53, 56/57, 60/61)
  // A register is read from LDS between the last MFMA that uses its old contents and its first
  // use; LDS reads return in order, so "the reads issued up to some point have landed" is
  // s_waitcnt lgkmcnt(number of reads issued since).  An MFMA occupies the matrix pipe for 32
  // cycles and the wave's issue for about half of that: what is issued behind it has to fit
  // the other half, so copies and reads are spread over the slots as evenly as the rules above
  // allow.
  auto copy_at = [&](auto slot_) {  // slot of the block
#ifndef MX_ABL_NO_DMA
    constexpr int j = Plan::copy_of(decltype(slot_)::value);
    if constexpr (j >= 0) issue_piece(std::integral_constant<int, j>{});
#endif
  };
  // quarter: the MFMAs of a[ah] x b[bh]; AMAJOR: a's sub-tiles one after the other (else b's);
  // side(slot, false) runs in front of a slot's MFMA, side(slot, true) behind it
  auto quarter = [&](Frags& f, auto first_, auto ah_, auto bh_, auto amajor_, auto&& side) {
    constexpr bool kFirst = decltype(first_)::value;
    constexpr int ah = decltype(ah_)::value, bh = decltype(bh_)::value;
    constexpr bool kAMajor = decltype(amajor_)::value;
    static_for<0, Plan::kQ>([&](auto i_) {
      constexpr int i = decltype(i_)::value;
      constexpr int tm = kAMajor ? i / TB : i % TA, tn = kAMajor ? i % TB : i / TA;
      constexpr int m = TA * ah + tm, n = TB * bh + tn;
      side(i_, std::false_type{});
      mfma16_asm<(n >> 1), (m >> 1), kFirst>(acc[m][n], f.b[bh][tn], f.a[ah][tm], f.sb[n & 1], f.sa[m & 1]);
      side(i_, std::true_type{});
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  auto landed = [&](auto n_, v8i& frag) {  // all LDS reads but the n youngest have landed
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(kReadsPerPiece * decltype(n_)::value > 15 ? 15 : kReadsPerPiece * decltype(n_)::value) : "memory");
    asm volatile("" : "+v"(frag));
  };
  auto block_steps = [&](Frags& f, auto first_) {
    using H0 = std::integral_constant<int, 0>;
    using H1 = std::integral_constant<int, 1>;
    constexpr int kQ = Plan::kQ;
    const uint32_t s_cur = lds_base + c_slot * Lds::kBlock, s_nxt = lds_base + next_slot(c_slot) * Lds::kBlock;
    // in front of slot kRelease: this wave's reads of the block are done, and once every wave's are
    // its place in the ring is free
    auto release = [&]() {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      asm volatile("" : "+v"(f.a[0][TA - 1]));
      uint64_t t0 = 0;
      if constexpr (PROF) t0 = __builtin_readcyclecounter();
      __builtin_amdgcn_s_barrier();
      if constexpr (PROF) {
        const uint64_t t1 = __builtin_readcyclecounter();
        prof_bar += t1 - t0;
        prof_last += t1 - t0;  // keep the barrier out of the body figure
      }
    };
    // quarter 0.  In flight on entry: what quarter 3 read after a[0][0], of a[1] and a[0][1] up to a[0][TA - 2]
    quarter(f, first_, H0{}, H0{}, std::true_type{}, [&](auto i_, auto after_) {
      constexpr int i = decltype(i_)::value;
      if constexpr (!decltype(after_)::value) {
        if constexpr (i == Plan::kRelease) release();
        else if constexpr (i % TB == 0 && i != 0) {
          constexpr int t = i / TB;  // a sub-tile of a[0] begins
          // (the last one was read in this quarter's first slots)
          constexpr int since = t < TA - 1 ? Plan::after_a0(t) + Plan::before0(i) : Plan::before0(i) - 2;
          landed(std::integral_constant<int, since>{}, f.a[0][t]);
        }
      } else {
#ifndef MX_ABL_NO_READ
        static_for<Plan::before0(i), Plan::before0(i + 1)>([&](auto r_) {
          constexpr int r = decltype(r_)::value;
          if constexpr (r < 2) read_a(f, s_cur, H0{}, std::integral_constant<int, 2 * (TA - 1) + r>{});
          else read_b(f, s_cur, H1{}, std::integral_constant<int, r - 2>{});
        });
#endif
        copy_at(i_);
      }
    });
    if constexpr (Plan::kRelease == kQ) release();
    pin_set(f.a[1]);
    pin_set(f.b[1]);
    // quarter 1
    quarter(f, first_, H1{}, H0{}, std::false_type{}, [&](auto i_, auto after_) {
      if constexpr (decltype(after_)::value) copy_at(std::integral_constant<int, kQ + decltype(i_)::value>{});
    });
    uint64_t t0 = 0, t1 = 0;
    if constexpr (PROF) {
      t0 = __builtin_readcyclecounter();
      prof_body += t0 - prof_last;
    }
    // block b+1 (and any output stores): everything but the copies issued so far in this block, and
    // a whole block's where the ring holds three
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(Plan::copies_before(2 * kQ) + (Lds::kStages - 2) * Plan::kCopies) : "memory");
    if constexpr (PROF) {
      t1 = __builtin_readcyclecounter();
      prof_vm += t1 - t0;
    }
    __builtin_amdgcn_s_barrier();
    if constexpr (PROF) {
      prof_last = __builtin_readcyclecounter();
      prof_bar += prof_last - t1;
    }
    // quarter 2: b[0] of block b+1 and its first three scale dwords
    quarter(f, first_, H1{}, H1{}, std::false_type{}, [&](auto i_, auto after_) {
      constexpr int i = decltype(i_)::value;
      if constexpr (decltype(after_)::value) {
        copy_at(std::integral_constant<int, 2 * kQ + i>{});
#ifndef MX_ABL_NO_READ
        static_for<Plan::first2(i), Plan::first2(i + 1)>([&](auto r_) {
          constexpr int r = decltype(r_)::value;
          if constexpr (r < 2 * TB) read_b(f, s_nxt, H0{}, r_);
          else read_scale_piece(f, s_nxt, std::integral_constant<int, r - 2 * TB>{});
        });
#endif
      }
    });
    // quarter 3: the other scale dwords before the first read of a[0]; a[1] and a[0] as
    // BlockPlan::plan3 has them (256 x 256: a[1] 0-3, a[0][0], a[1] 4, 5, a[0][1], a[1] 6, 7, a[0][2], one a slot)
    quarter(f, first_, H0{}, H1{}, std::true_type{}, [&](auto i_, auto after_) {
      constexpr int i = decltype(i_)::value;
      if constexpr (decltype(after_)::value) {
        copy_at(std::integral_constant<int, 3 * kQ + i>{});
#ifndef MX_ABL_NO_READ
        static_for<0, Plan::kReads3>([&](auto k_) {
          constexpr auto plan = Plan::plan3();
          constexpr int k = decltype(k_)::value, r = plan.what[k];
          if constexpr (plan.slot[k] == i) {
            if constexpr (r < 2 * TA) read_a(f, s_nxt, H1{}, std::integral_constant<int, r>{});
            else read_a(f, s_nxt, H0{}, std::integral_constant<int, r - 2 * TA>{});
          }
        });
        static_for<3, kScalePieces>([&](auto e_) {
          if constexpr ((decltype(e_)::value - 3) % TB == i) read_scale_piece(f, s_nxt, e_);
        });
#endif
      }
    });
    c_slot = next_slot(c_slot);
    // the next block's first MFMAs need its b[0], its scales and the first sub-tile of its
    // a[0]: everything but the reads issued since
    constexpr int since0 = kReadsPerPiece * Plan::after_a0(0);
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(since0 > 15 ? 15 : since0) : "memory");
    pin_set(f.b[0]);
    asm volatile("" : "+v"(f.a[0][0]));
    next_scales(f, c_slot);
    issue_advance();
  };

  // Output: a lane holds, per 16x16 sub-tile, row li and columns 4lj + 0..3.  Lanes of
  // neighbouring lane groups trade halves with v_permlane16_swap so that each owns 8 consecutive
  // bf16 of a row; a 32-row x 64-column piece is then turned around in this wave's private LDS
  // patch (the 26 KB the ring leaves free) so that 8 lanes store one full 128-byte line of a row
  // -- stores that scatter 32-byte pieces over many rows back up the write path.
  // Buffer stores: one descriptor per tile bounds the rows, a 32-bit offset per lane, scalar
  // offsets per piece.  Requires N % 8 == 0 and ldd % 8 == 0 (checked on the host).
  // (LDS accesses as assembly, for the reason given at the fragment reads.)
  const uint32_t patch = lds_base + Lds::kRing + wave * Lds::kPatch;
  const uint32_t nan_mask = (MODE != kDense && poison) ? 0x7FC07FC0u : 0u;
  auto epilogue = [&](const Tile32& t) {
    // The epilogue's per-lane addresses are worked out here, from a lane number the compiler
    // cannot see through, every time: kept across the K loop instead they push its register
    // file over the edge, and a spilled register's reload waits for every copy and store in
    // flight (s_waitcnt vmcnt(0)) at exactly the two places where those should keep running.
    uint32_t lane_e = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(lane_e));
    // + (m & 1) * 16 rows + (second sub-tile pair of the piece) * 64
    const uint32_t patch_w = patch + (lane_e & 15) * kPatchPitch + ((lane_e >> 4) & 1) * 32 + (lane_e >> 5) * 16;
    const uint32_t patch_r = patch + (lane_e >> 3) * kPatchPitch + (lane_e & 7) * 16;  // + pass*8 rows
    const int64_t rows_valid = (MODE == kGrouped2d3d && p.d_offs) ? (int64_t)t.rows_d : t.rows_a;
    const uint32_t cols_valid = (uint32_t)(t.rows_b < kEB ? t.rows_b : kEB);
    if constexpr (MODE == kSplitK) {
      // float32 partial sums straight from the accumulators: a lane stores 16 bytes of row li
      // per sub-tile and q; short pieces, but the partial tiles are few and are read back at once
      const uint32_t ld_b = (uint32_t)p.ldd * 4;
      const __amdgpu_buffer_rsrc_t rp = make_rsrc(t.d, (rows_valid < kEA ? rows_valid : kEA) * ld_b);
      const uint32_t row_b = (wm * 32 * TA + li) * ld_b;
      // (a lane holds row 16m + li, columns 16n + 4lj + 0..3 of sub-tile (m, n))
      static_for<0, 4 * TA * TB>([&](auto i_) {
        constexpr int m = decltype(i_)::value / (2 * TB), n = decltype(i_)::value % (2 * TB);
        const uint32_t col = wave_col<TB>(wn, n) + 4 * lj;
        const uint32_t v = col < cols_valid ? row_b + col * 4 : 0x80000000u;
        const u32x4 w = {__float_as_uint(acc_read<0>(acc[m][n])), __float_as_uint(acc_read<1>(acc[m][n])),
                         __float_as_uint(acc_read<2>(acc[m][n])), __float_as_uint(acc_read<3>(acc[m][n]))};
        __builtin_amdgcn_raw_buffer_store_b128(w, rp, v, m * 16 * ld_b, MX_STORE_AUX);
      });
      return;
    }
    if constexpr (GATE) {
      // A lane holds, of row 16 m + li, columns 16 n + 4 lj .. + 3 of both factors.  A 32-column block's maximum is over two
      // n and the four lanes of a row; four dwords of codes are turned around among those lanes, so that each stores 16
      // consecutive bytes; the wave's 128 rows of two blocks are one whole 256-byte group of scales, lane 32 b + r
      // its dword of rows r, r + 32, r + 64, r + 96 of block b.
      const uint32_t gi = lane_e & 15, gj = lane_e >> 4, ldc = (uint32_t)p.ldd;
      const bool rceil = p.scale_mode == MX_SCALE_RCEIL;
      const __amdgpu_buffer_rsrc_t rc = make_rsrc(reinterpret_cast<uint8_t*>(p.d) + (int64_t)t.tm * kEA * p.ldd + t.tn * kEB,
                                                  (rows_valid < kEA ? rows_valid : kEA) * (int64_t)ldc - t.tn * kEB);
      const uint32_t v = (wm * 128 + gi) * ldc + wn * 64 + gj * 16;
      auto rows_max = [](uint32_t x) -> uint32_t {  // over the four lanes of a row
        const u32x2 a = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        const uint32_t y = max(a.x, a.y);
        const u32x2 b = __builtin_amdgcn_permlane32_swap(y, y, false, false);
        return max(b.x, b.y);
      };
      uint32_t scales = 0, inside[4];  // (columns of the fill are zeros, also where the row's sums are NaN)
      static_for<0, 4>([&](auto n_) {
        inside[decltype(n_)::value] = wn * 64 + 16 * decltype(n_)::value + 4 * gj < cols_valid ? ~0u : 0u;
      });
      static_for<0, 8>([&](auto m_) {
        constexpr int m = decltype(m_)::value;
        uint32_t g[4][2], top[2] = {0, 0};
        static_for<0, 4>([&](auto n_) {
          constexpr int n = decltype(n_)::value;
          const v4f &c = acc[m][n], &c2 = acc[m][n + 4];
          const uint32_t a0 = pack_bf16(acc_read<0>(c), acc_read<1>(c)), a1 = pack_bf16(acc_read<2>(c), acc_read<3>(c));
          const uint32_t b0 = pack_bf16(acc_read<0>(c2), acc_read<1>(c2)), b1 = pack_bf16(acc_read<2>(c2), acc_read<3>(c2));
          g[n][0] = swiglu2(a0, b0) & inside[n];
          g[n][1] = swiglu2(a1, b1) & inside[n];
          top[n >> 1] = pk_max_u16(top[n >> 1], pk_max_u16(g[n][0] & 0x7FFF7FFFu, g[n][1] & 0x7FFF7FFFu));
          __builtin_amdgcn_sched_barrier(0);
        });
        uint32_t sb[2];
        float mult[2];
        static_for<0, 2>([&](auto b_) {
          constexpr int b = decltype(b_)::value;
          const uint32_t amax = rows_max(max(top[b] & 0xFFFFu, top[b] >> 16));
          sb[b] = rceil ? scale_byte<MX_SCALE_RCEIL>(amax) : scale_byte<MX_SCALE_FLOOR>(amax);
          mult[b] = rceil ? scale_multiplier<MX_SCALE_RCEIL>(sb[b]) : scale_multiplier<MX_SCALE_FLOOR>(sb[b]);
        });
        uint32_t d[4];
        static_for<0, 4>([&](auto n_) {
          constexpr int n = decltype(n_)::value;
          d[n] = cvt2<true>(g[n][1], mult[n >> 1], cvt2<false>(g[n][0], mult[n >> 1], 0));
          if (sb[n >> 1] == 255) d[n] = nan_block_codes2(g[n][0]) | (nan_block_codes2(g[n][1]) << 16);
        });
        const u32x2 e0 = __builtin_amdgcn_permlane16_swap(d[0], d[1], false, false);
        const u32x2 e1 = __builtin_amdgcn_permlane16_swap(d[2], d[3], false, false);
        const u32x2 f0 = __builtin_amdgcn_permlane32_swap(e0.x, e1.x, false, false);
        const u32x2 f1 = __builtin_amdgcn_permlane32_swap(e0.y, e1.y, false, false);
        __builtin_amdgcn_raw_buffer_store_b128(u32x4{f0.x, f1.x, f0.y, f1.y}, rc, v, m * 16 * ldc, 0);
        if ((gj & 1) == (m & 1)) scales |= (gj >> 1 ? sb[1] : sb[0]) << (8 * (m >> 1));
        __builtin_amdgcn_sched_barrier(0);
      });
      if ((int64_t)t.tm * kEA + wm * 128 < p.M) {
        const int64_t steps = (p.N + 127) / 128 * 2;
        reinterpret_cast<uint32_t*>(p.d2)[(((int64_t)t.tm * 2 + wm) * steps + t.tn * 2 + wn) * 64 + lane_e] = scales;
      }
      return;
    }
    const uint32_t ldd_b = (uint32_t)p.ldd * 2;
    const __amdgpu_buffer_rsrc_t rd = make_rsrc(t.d, rows_valid * ldd_b);
    // lane's place in a stored piece: row (lane >> 3) + 8*pass, columns (lane & 7)*8 .. +7
    const uint32_t colp = wave_col<TB>(wn, 0) + (lane_e & 7) * 8;
    const uint32_t vrow = (wm * 32 * TA + (lane_e >> 3)) * ldd_b + colp * 2;
    // ... of a piece of 32 columns: row (lane >> 2) + 16*pass, columns (lane & 3)*8 .. +7
    const uint32_t patch_r4 = patch + (lane_e >> 2) * kPatchPitch + (lane_e & 3) * 16;
    const uint32_t colp4 = TB == 3 ? wave_col<TB>(wn, 4) + (lane_e & 3) * 8 : 0;
    const uint32_t vrow4 = (wm * 32 * TA + (lane_e >> 2)) * ldd_b + colp4 * 2;
    // Pieces: 32 rows (sub-tile rows m = 2 mp, + 1; 16 where the ring holds three blocks) x 64 columns
    // (sub-tiles n = 4 np .. + 3), 192-wide tiles' second ones x 32.
    // A wave's LDS instructions execute in order, so a piece's reads may follow its writes
    // without a wait, and the next piece's writes may follow those reads: the only waits are
    // for the read data, with the next piece's conversion and writes already under way.
    // a lane holds row 16m + li, columns 16n + 4lj + 0..3 of sub-tile (m, n).  A part of a
    // piece covers 16 rows x 32 columns: sub-tiles (m, n) and (m, n + 1).
    // v_permlane16_swap trades the halves of two neighbouring lane
    // groups: the even groups end up with 8 consecutive columns of sub-tile n, the odd ones with
    // 8 of sub-tile n + 1.
    constexpr int kNP = (TB + 1) / 2, kSubs = Lds::kPatchRows / 16, kPieces = 2 * TA / kSubs * kNP;
    constexpr auto col_parts = [](int pc) { return TB == 3 && pc % 2 ? 1 : 2; };
    constexpr auto parts_of = [col_parts](int pc) { return kSubs * col_parts(pc); };  // parts, and 1 KB stores, of a piece
    auto stage_part = [&](auto p_, auto k_) {
      constexpr int mp = decltype(p_)::value / kNP, np = decltype(p_)::value % kNP, k = decltype(k_)::value;
      constexpr int kc = col_parts(decltype(p_)::value);
      constexpr int m = kSubs * mp + k / kc, n = 4 * np + 2 * (k % kc);
      const v4f& c0 = acc[m][n];
      const v4f& c1 = acc[m][n + 1];
      const float a[8] = {acc_read<0>(c0), acc_read<1>(c0), acc_read<2>(c0), acc_read<3>(c0),
                          acc_read<0>(c1), acc_read<1>(c1), acc_read<2>(c1), acc_read<3>(c1)};
      uint32_t x0 = pack_bf16(a[0], a[1]), y0 = pack_bf16(a[2], a[3]);
      uint32_t x1 = pack_bf16(a[4], a[5]), y1 = pack_bf16(a[6], a[7]);
      if constexpr (MODE != kDense) {  // a broken group contract must not pass unnoticed: NaN
        x0 |= nan_mask;
        y0 |= nan_mask;
        x1 |= nan_mask;
        y1 |= nan_mask;
      }
      const u32x2 sx = __builtin_amdgcn_permlane16_swap(x0, x1, false, false);
      const u32x2 sy = __builtin_amdgcn_permlane16_swap(y0, y1, false, false);
      const v4i w = {(int)sx.x, (int)sy.x, (int)sx.y, (int)sy.y};
      lds_write_b128_hidden<(k / kc) * 16 * kPatchPitch + (k % kc) * 64>(patch_w, w);
      __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (OUT32) {
      // The gradient of a float32 parameter or activation: bf16 values, 4 bytes each.  Written here they cost
      // 4 bytes per element instead of the 8 of a bf16 matrix and its conversion by a launch of its own.  A store covers
      // 4 rows of 64 columns (8 of 32), 16 bytes a lane.
      const uint32_t ld_b = (uint32_t)p.ldd * 4;
      const __amdgpu_buffer_rsrc_t rf = make_rsrc(t.d, rows_valid * ld_b);
      static_for<0, kPieces>([&](auto p_) {
        constexpr int pc = decltype(p_)::value, m = pc / kNP, np = pc % kNP;
        constexpr int kLanes = col_parts(pc) == 2 ? 16 : 8, kRows = 64 / kLanes, kStores = 16 * kSubs / kRows;
        static_for<0, parts_of(pc)>([&](auto k_) { stage_part(p_, k_); });
        const uint32_t row = lane_e / kLanes, col = wave_col<TB>(wn, 4 * np) + (lane_e % kLanes) * 4;
        const uint32_t from = patch + row * kPatchPitch + (lane_e % kLanes) * 8;
        const uint32_t v = col < cols_valid ? (wm * 32 * TA + m * 16 * kSubs + row) * ld_b + col * 4 : 0x80000000u;
        static_for<0, kStores>([&](auto q_) {
          constexpr int q = decltype(q_)::value;
          u32x2 x;
          // (in order behind this wave's writes; waited for on the spot)
          asm volatile("ds_read_b64 %0, %1 offset:%2\n\ts_waitcnt lgkmcnt(0)"
                       : "=&v"(x) : "v"(from), "n"(q * kRows * kPatchPitch) : "memory");
          const u32x4 w = {x.x << 16, x.x & 0xFFFF0000u, x.y << 16, x.y & 0xFFFF0000u};
          __builtin_amdgcn_raw_buffer_store_b128(w, rf, v, q * kRows * ld_b, MX_STORE_AUX);
        });
      });
      return;
    }
    v4i r[2][4];
    static_for<0, parts_of(0)>([&](auto k_) { stage_part(std::integral_constant<int, 0>{}, k_); });
    static_for<0, kPieces>([&](auto p_) {
      constexpr int pc = decltype(p_)::value, m = pc / kNP, np = pc % kNP;
      constexpr int kStores = parts_of(pc), kNext = pc + 1 < kPieces ? parts_of(pc + 1) : 0;
      constexpr int kEach = (kNext + kStores - 1) / kStores;  // parts of the next piece in front of each store
      constexpr bool kWide = col_parts(pc) == 2;
      constexpr int kRows = kWide ? 8 : 16;  // rows of a store
      uint64_t e0 = 0;
      if constexpr (PROF) e0 = __builtin_readcyclecounter();
      static_for<0, kStores>([&](auto q_) {
        constexpr int q = decltype(q_)::value;
        r[pc & 1][q] = lds_read_b128_hidden<q * kRows * kPatchPitch>(kWide ? patch_r : patch_r4);
      });
      const uint32_t v = kWide ? ((colp + np * 64 < cols_valid) ? vrow + np * 128 : 0x80000000u)
                                      : (colp4 < cols_valid ? vrow4 : 0x80000000u);
      // the next piece's conversion runs between this piece's stores, which drain at the
      // write path's pace
      static_for<0, kStores>([&](auto q_) {
        constexpr int q = decltype(q_)::value;
        static_for<q * kEach, (q + 1) * kEach < kNext ? (q + 1) * kEach : (q * kEach < kNext ? kNext : q * kEach)>(
            [&](auto k_) { stage_part(std::integral_constant<int, pc + 1>{}, k_); });
        // the reads are done once at most the younger writes are outstanding
        if constexpr (q == 0) asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(kEach < kNext ? kEach : kNext) : "memory");
        const v4i rq = pin(r[pc & 1][q]);
        const u32x4 w = {(uint32_t)rq.x, (uint32_t)rq.y, (uint32_t)rq.z, (uint32_t)rq.w};
#ifdef MX_ABL_STORE_ROWS  // timing ablation: only sub-tile rows below this many are written
        if constexpr (kSubs * m < 2 * MX_ABL_STORE_ROWS)
#endif
        __builtin_amdgcn_raw_buffer_store_b128(w, rd, v, (m * 16 * kSubs + q * kRows) * ldd_b, MX_STORE_AUX);
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (PROF) prof_e_stage += __builtin_readcyclecounter() - e0;
    });
  };

  uint64_t prof_t0 = 0;
  if constexpr (PROF) prof_t0 = __builtin_readcyclecounter();
  // ---- prologue: fill the ring, fetch the first fragments
  loader_open_tile();
#pragma unroll 1
  for (int i = 0; i < Lds::kStages; ++i) issue_block();
  // block 0; the others are in flight when the first step starts
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((Lds::kStages - 1) * Plan::kCopies) : "memory");
  __builtin_amdgcn_s_barrier();
  Frags f;
  {
    using Z = std::integral_constant<int, 0>;
    using O = std::integral_constant<int, 1>;
    static_for<0, 2 * TA>([&](auto i_) { read_a(f, lds_base, Z{}, i_); });
    static_for<0, 2 * TA>([&](auto i_) { read_a(f, lds_base, O{}, i_); });
    static_for<0, 2 * TB>([&](auto i_) { read_b(f, lds_base, Z{}, i_); });
    static_for<0, kScalePieces>([&](auto i_) { read_scale_piece(f, lds_base, i_); });
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    pin_set(f.a[0]);
    pin_set(f.a[1]);
    pin_set(f.b[0]);
    next_scales(f, 0);
  }
  if constexpr (PROF) prof_last = __builtin_readcyclecounter();

  // ---- tiles; at the top of every tile f0 holds the fragments of its first half block (the
  // last step of a tile has already read them from the next tile's first block, which the
  // loader fetched like any other block).
  for (uint32_t tile = 0; tile < n_my; tile += PAIR ? 2 : 1) {
    const Tile32 t = get_tile(tile);
    {
      // PAIR: the loader walks both segments of the tile one after the other (same K for both);
      // for the compute stream they are one run of blocks
      const uint32_t nblocks = PAIR ? 2 * t.nblocks : t.nblocks;
      block_steps(f, std::true_type{});
      // two blocks per trip: a taken branch stalls the lone wave of a SIMD for longer than the
      // 32 cycles its last MFMA covers, and the trip's end has two of them
      uint32_t i = 1;
      for (; i + 2 <= nblocks; i += 2) {
        block_steps(f, std::false_type{});
        block_steps(f, std::false_type{});
      }
      if (i < nblocks) block_steps(f, std::false_type{});
      // the next tile's first fragments, read in the last quarter, become ordinary values
      // before anything else runs
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      pin_set(f.a[0]);
      pin_set(f.a[1]);
      if constexpr (PROF) {
        const uint64_t e0 = __builtin_readcyclecounter();
        prof_body += e0 - prof_last;
        epilogue(t);
        prof_last = __builtin_readcyclecounter();
        prof_epi += prof_last - e0;
      } else {
#ifndef MX_ABL_NO_EPILOGUE
        epilogue(t);
#else
        (void)t;  // timing ablation: the MFMAs are volatile assembly and stay
#endif
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // drain the over-issued prefetches before retiring
  if constexpr (PROF) {
    if (lane == 0) {
      uint64_t* o = p.prof + (blockIdx.x * 4 + wave) * 8;
      o[0] = prof_vm;
      o[1] = prof_bar;
      o[2] = prof_body;
      o[3] = prof_epi;
      o[4] = prof_e_stage;
      o[5] = prof_e_wait;
      o[6] = prof_e_store;
      o[7] = __builtin_readcyclecounter() - prof_t0;
    }
  }
}

// Test hook, process-wide: > 0 = number of persistent workgroups (also lowers how many tiles one
// grouped launch covers, which is what the tests use it for); 0 = one per CU.
static std::atomic<int> debug_grid{0};
#ifdef MX_TIMING_BUILD
static uint64_t* debug_prof = nullptr;  // device buffer for the per-wave cycle counts, or nullptr
#else
static constexpr uint64_t* debug_prof = nullptr;
#endif

// One persistent workgroup per CU of the current device, a multiple of the 8 XCDs (0: the device
// cannot be queried).
static int64_t persistent_grid() {
  const int num_cus = current_device_cus();
  if (num_cus == 0) return 0;
  int64_t grid = (num_cus / 8) * 8;
  if (grid < 8) grid = 8;
  if (debug_grid > 0) grid = (debug_grid + 7) / 8 * 8;
  return grid;
}

template <int MODE, bool PROF, bool PAIR = false, int TA = 4, int TB = 4, bool OUT32 = false, bool GATE = false>
static bool configure32() {
  static std::atomic<bool> configured[kMaxDevices];
  return raise_lds_limit(reinterpret_cast<const void*>(gemm_nt32_kernel<MODE, PROF, PAIR, TA, TB, OUT32, GATE>),
                         Lds32<TA, TB>::kBytes, configured);
}
bool prepare_dense();
template <int MODE, bool PROF, bool PAIR = false, int TA = 4, int TB = 4, bool OUT32 = false, bool GATE = false>
static int launch32(const Gemm32Args& p, int64_t nb, hipStream_t st) {
  auto kern = gemm_nt32_kernel<MODE, PROF, PAIR, TA, TB, OUT32, GATE>;
  constexpr int lds = Lds32<TA, TB>::kBytes;  // ring + one output patch per wave: most of the CU's 160 KB
  constexpr bool kDenseForm = !PROF && (MODE == kDense || MODE == kSplitK);
  if (!(kDenseForm ? prepare_dense() : configure32<MODE, PROF, PAIR, TA, TB, OUT32>())) return MX_ERR_LAUNCH;
  int64_t grid = persistent_grid();
  if (grid == 0) return MX_ERR_LAUNCH;
  const int64_t need = (nb + 7) / 8 * 8;  // nb: the tile count, or an upper bound of it
  if (need < grid && debug_grid <= 0) grid = need;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), lds, st, p);
  return hipGetLastError() == hipSuccess ? MX_OK : MX_ERR_LAUNCH;
}

// Test hook: edges of the dense kernels' tiles, 64 ta x 64 tb, and slices (0: by shape).
static std::atomic<int> debug_tile{0}, debug_slices{0};
void set_debug_tile(int ta, int tb, int slices) {
  debug_tile = ta * 16 + tb;
  debug_slices = slices;
}

// ---- which tile, and whether to split along K ---------------------------------------------------
// The dense tiles, and what a 128-deep block of one takes a CU with all CUs busy, in microseconds.
// Smaller ones cost a little more per flop (operand bytes per flop x 1.17 and 1.5) and leave fewer
// CUs idle in a launch's last round: 4096 x 2048, K 6144 runs 128 tiles of 256 x 256 in 58 us and
// 256 of 128 x 256 in 41; 3001 x 4096, K 4096 192 in 49 and 256 of 192 x 256 in 40; with many
// rounds 256 x 256 stays ahead (16384 x 14336, K 4096: 671 us, 697, 756, 778, 837 in this order).
struct DenseTile {
  int ta, tb;
  double block_us;
};
static constexpr DenseTile kDenseTiles[] = {{4, 4, 1.32}, {3, 4, 1.00}, {4, 3, 1.04}, {2, 4, 0.75}, {4, 2, 0.74}};

static int64_t tile_count(const DenseTile& t, int64_t M, int64_t N) {
  return ((M + 64 * t.ta - 1) / (64 * t.ta)) * ((N + 64 * t.tb - 1) / (64 * t.tb));
}

// Microseconds that `tiles` tiles of `blocks` blocks each take on `grid` CUs.  Fitted to 240 shapes of
// 16..16384 rows, 1024..151936 columns and K 256..16384 in every way to run them (residual 5 to 10 %;
// choosing by it loses 2 % against the best of them): a round costs 3.6 us to fill and up to
// 1.5 us to drain, and CUs that idle let the others clock higher.
static double tiles_us(const DenseTile& t, int64_t tiles, int64_t blocks, int64_t grid) {
  const double area = t.ta * t.tb / 16.0, rest = (double)(tiles % grid) / grid;
  double us = (double)(tiles / grid) * (blocks * t.block_us + 3.6 + 1.5 * area);
  if (tiles % grid) us += blocks * t.block_us * (0.68 + 0.32 * rest) + 3.6 + 1.5 * area * rest;
  return us;
}

// The tile for `products` products of one launch, their tiles side by side (each with K blocks of
// its own, or of two operand sets: `blocks` counts both).
static const DenseTile* best_tile(int64_t M, int64_t N, int64_t blocks, int products, int64_t grid) {
  const DenseTile* best = nullptr;
  double best_us = 0;
  for (const DenseTile& t : kDenseTiles) {
    if (debug_tile && debug_tile != t.ta * 16 + t.tb) continue;
    // (a smaller tile has to promise 6 %: over many rounds the power limit leaves less of its gain than
    // idle CUs cost, 4096 x 14336, K 16384 2 % slower on 192 x 256 where 3 % less was predicted)
    const double us = (t.ta * t.tb == 16 ? 1.0 : 1.06) * tiles_us(t, products * tile_count(t, M, N), blocks, grid);
    if (!best || us < best_us) {
      best = &t;
      best_us = us;
    }
  }
  return best;
}

// The tiles of the kernel of few tiles, and the microseconds that `tiles` of `blocks` blocks each take on it, fitted to the
// 225 shapes of 72..2048 rows, 512..10240 columns and K 256..10240 for which it may be chosen (residual 4 %).
struct RingTile {
  int ta, tb;
  double start_us, block_us, part_us, share_us, round_us;
};
static constexpr RingTile kRingTiles[] = {{1, 1, 1.74, 0.289, 0.242, 0.038, 2.88}, {2, 1, 1.26, 0.436, 0.350, 0.087, 3.73}};
static double ring_us(const RingTile& t, int64_t tiles, int64_t blocks, int64_t grid) {
  const double rest = (double)(tiles % grid) / grid;
  double us = t.start_us + (double)(tiles / grid) * (blocks * t.block_us + t.round_us);
  if (tiles % grid) us += blocks * (t.part_us + t.share_us * rest) + t.round_us;
  return us;
}
// The one of them that promises 3 % over `us`, which then becomes its time.  (Over those shapes the choice takes 0.81 of
// the time without it, the best one of either 0.81; none of them got slower by more than 3 %.)
static const RingTile* better_ring(int64_t M, int64_t N, int64_t blocks, int products, int64_t grid, double& us) {
  const RingTile* best = nullptr;
  for (const RingTile& t : kRingTiles) {
    if (debug_tile && debug_tile != t.ta * 16 + t.tb) continue;
    const int64_t tiles = products * ((M + 64 * t.ta - 1) / (64 * t.ta)) * ((N + 64 * t.tb - 1) / (64 * t.tb));
    const double mine = ring_us(t, tiles, blocks, grid);
    if (mine < (best ? us : 0.97 * us) || debug_tile) {
      best = &t;
      us = mine;
    }
  }
  return best;
}

// What a dense product runs on: the persistent kernel with tiles of 64 ta x 64 tb in `slices` slices
// of K, or (ta == 0) the kernel of one 128 x 128 tile per workgroup.
//   * That one is ahead for short contractions only: it starts faster (512 x 4096: K 256 6.1 us, 7.4
//     on the persistent kernel; K 1024 10.2 and 10.2; K 4096 28.5 and 22.7).
//   * S slices add float32 partial sums, written and read back (3.2 TB/s) by a launch of their own,
//     and are taken for a predicted gain of 8 %: 256 x 4096, K 8192 40 us unsplit, 23 in four
//     slices; 512 x 4096, K 14336 85 and 39; 2048 x 2048, K 147456 976 and 427 (rows 128 bytes further apart than
//     they are long; dense rows 1300 and 537).  The partial sums stay under 64 MiB,
//     one 256 x 256 tile per CU; more only where 256 x 256 tiles leave a good part of their rounds empty: half to 5/7 of
//     the CUs (1280 x 6656, K 131072: 130 tiles, 1050 us unsplit, 940 in five slices; 2304 x 4096, K 147456: 144,
//     1511 and 1405), or one to one and a half times (4352 x 4352, K 147456: 289, 3045 and 2777).  In
//     between the promise is not kept: 592 x 16416, K 147456: 195 tiles, 1470 unsplit and 1577 in five
//     slices; 4864 x 2560: 190 tiles, K 98304 1215 and 1244 in four, K 147456 1743 and 1641.
//     Contractions of up to 4096 stay one chain of sums.  Up to 2048 slices gain nothing (256 x 1024, K 2048 13.9 us
//     and 13.9 in four; 256 x 2048, K 1024 9.6 and 13.1 in two; 2048 x 2048, K 2048 15.3 and 26.9); at 4096 they would
//     (256 x 1024 22.9 and 16.1 in four, 256 x 4096 23.2 and 17.9), which is given up so that at these
//     widths a row's result of more than 64 rows does not depend on how many there are: all tiles add in one order.
GemmPlan plan_dense(int64_t M, int64_t N, int64_t K, bool may_split) {
  const int64_t grid = persistent_grid(), blocks = K / kKB;
  if (grid == 0 || K % kKB) return {0, 0, 1};
  const DenseTile* t = best_tile(M, N, blocks, 1, grid);
  if (!t) {
    double us = 0;
    const RingTile* r = better_ring(M, N, blocks, 1, grid, us);
    return r ? GemmPlan{r->ta, r->tb, 1} : GemmPlan{0, 0, 1};
  }
  GemmPlan best{t->ta, t->tb, 1};
  double best_us = tiles_us(*t, tile_count(*t, M, N), blocks, grid) + 2.0;
  if (!debug_tile) {
    const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128), rounds = (tiles + grid - 1) / grid;
    const double us = 4.3 * rounds + (0.28 + 0.47 * rounds) * blocks;
    if (us < best_us) {
      best = {0, 0, 1};
      best_us = us;
    }
  }
  const double plain_us = best_us;
  if (may_split && (blocks > 32 || debug_slices)) {
    for (const DenseTile& u : kDenseTiles) {
      if (u.ta * u.tb == 12 || (debug_tile && debug_tile != u.ta * 16 + u.tb)) continue;
      const int64_t tiles = tile_count(u, M, N);
      for (int s = 2; s <= 8; ++s) {
        const int64_t per = (blocks + s - 1) / s;
        if (per < 4 || (s - 1) * per >= blocks || (debug_slices && s != debug_slices)) continue;
        const double bytes = 4.0 * s * M * N;
        const bool large = bytes > (double)(64 << 20);
        if (large && (u.ta * u.tb < 16 || 2 * tiles <= grid || (7 * tiles > 5 * grid && tiles <= grid) || 2 * tiles >= 3 * grid))
          continue;
        const double us = tiles_us(u, tiles * s, per, grid) + 2.0 + 4.2 + bytes / 3.2e6;
        if (us < best_us && us <= 0.92 * plain_us || debug_slices) {
          best = {u.ta, u.tb, s};
          best_us = us;
        }
      }
    }
  }
  // Few tiles, not split: 64-wide ones (up to 64 rows have a kernel of their own).  A split is not compared with them.  Of
  // 151 shapes that are split (72..1024 rows, 512..4096 columns) the better 64-wide tile in one chain takes, over the split's
  // time, 0.72 to 0.89 with 34 blocks (1024 x 1024 14.8 and 20.6 us), 0.81 to 1.07 with 48, 0.89 to 1.30 with 64, 0.97 to 1.49
  // with 80 and 1.10 to 1.57 with 112 (256 x 512 33.5 and 22.3).  Sums of two products, which plan_pair splits (83 shapes): 0.91 to
  // 1.33 with 2 x 32 blocks, 1.05 to 1.52 with 2 x 48, 1.37 to 2.18 with 2 x 112.
  if (best.slices == 1 && !debug_tile && M > 64)
    if (const RingTile* r = better_ring(M, N, blocks, 1, grid, best_us)) best = {r->ta, r->tb, 1};
  return best;
}

// What the sum of two products over K each runs on: one chain over both (slices == 1), or `slices` slices of
// which half belong to either, under the conditions above.  One chain of 2 K / 128 blocks per tile bounds few
// rows: 256 x 4096, K 2 x 14336 takes 189 us so (16 tiles on 256 CUs), 53 in eight slices; 512 rows 189 and 74 in four;
// 1024 rows 191 and 121 in two; 512 x 2048, K 2 x 6144 57 and 27 in six; 4096 rows 80 and 94 in two: not split.
GemmPlan plan_pair(int64_t M, int64_t N, int64_t K) {
  const int64_t grid = persistent_grid(), blocks = K / kKB;
  GemmPlan best{0, 0, 1};
  if (grid == 0 || K % kKB || (2 * blocks <= 32 && !debug_slices)) return best;
  const DenseTile* t = best_tile(M, N, 2 * blocks, 1, grid);
  if (!t) return best;
  const double plain_us = tiles_us(*t, tile_count(*t, M, N), 2 * blocks, grid) + 2.0;
  double best_us = plain_us;
  for (const DenseTile& u : kDenseTiles) {
    if (u.ta * u.tb == 12 || (debug_tile && debug_tile != u.ta * 16 + u.tb)) continue;
    for (int s = 1; s <= 4; ++s) {
      const int64_t per = (blocks + s - 1) / s;
      const double bytes = 8.0 * s * M * N;
      if (per < 4 || (s - 1) * per >= blocks || bytes > (double)(64 << 20) || (debug_slices && 2 * s != debug_slices)) continue;
      const double us = tiles_us(u, tile_count(u, M, N) * 2 * s, per, grid) + 2.0 + 4.2 + bytes / 3.2e6;
      if ((us < best_us && us <= 0.92 * plain_us) || debug_slices) {
        best = {u.ta, u.tb, 2 * s};
        best_us = us;
      }
    }
  }
  return best;
}

// Whether two products of one launch (products == 2), or one over the K blocks of two operand sets (`blocks` counts both),
// run on the kernel of few tiles: ring() then.
GemmPlan plan_ring(int64_t M, int64_t N, int64_t blocks, int products) {
  const int64_t grid = persistent_grid();
  if (grid == 0) return {0, 0, 1};
  const DenseTile* t = best_tile(M, N, blocks, products, grid);
  double us = t ? tiles_us(*t, products * tile_count(*t, M, N), blocks, grid) + 2.0 : 0;
  if (t && debug_tile) return {0, 0, 1};
  const RingTile* r = better_ring(M, N, blocks, products, grid, us);
  return r ? GemmPlan{r->ta, r->tb, 1} : GemmPlan{0, 0, 1};
}

// Launches the persistent dense kernel on `p` with tiles of 64 ta x 64 tb.
template <int MODE, bool PAIR, bool OUT32, int TA, int TB>
static int launch_tile(Gemm32Args p, hipStream_t st) {
  int64_t tm = (p.M + 64 * TA - 1) / (64 * TA), tn = (p.N + 64 * TB - 1) / (64 * TB);
  if (p.two == kTwoA) tm *= 2;
  if (p.two == kTwoB) tn *= 2;
  if (MODE == kSplitK) p.tn_cnt = (int32_t)tn;
  return launch32<MODE, false, PAIR, TA, TB, OUT32>(p, tm * tn * (MODE == kSplitK ? p.G : 1), st);
}
template <int MODE, bool PAIR = false, bool OUT32 = false>
static int launch_dense32(const Gemm32Args& p, int ta, int tb, hipStream_t st) {
  switch (ta * 16 + tb) {
    case 0x44: return launch_tile<MODE, PAIR, OUT32, 4, 4>(p, st);
    case 0x24: return launch_tile<MODE, PAIR, OUT32, 2, 4>(p, st);
    case 0x42: return launch_tile<MODE, PAIR, OUT32, 4, 2>(p, st);
    default: break;
  }
  if constexpr (MODE != kSplitK) {
    if (ta == 3 && tb == 4) return launch_tile<MODE, PAIR, OUT32, 3, 4>(p, st);
    if (ta == 4 && tb == 3) return launch_tile<MODE, PAIR, OUT32, 4, 3>(p, st);
  }
  return MX_ERR_UNSUPPORTED;
}
// ... with the tile that suits its shape
template <bool PAIR = false, bool OUT32 = false>
static int launch_best32(const Gemm32Args& p, hipStream_t st) {
  const int64_t grid = persistent_grid();
  if (grid == 0) return MX_ERR_LAUNCH;
  const DenseTile* t = best_tile(p.M, p.N, (PAIR ? 2 : 1) * p.K / kKB, p.two ? 2 : 1, grid);
  return t ? launch_dense32<kDense, PAIR, OUT32>(p, t->ta, t->tb, st) : MX_ERR_UNSUPPORTED;
}

// Raises the LDS limit of every persistent kernel that a dense product may run on (prepare_dense).
template <int TA, int TB>
static bool prepare_tile() {
  return configure32<kDense, false, false, TA, TB>() && configure32<kDense, false, true, TA, TB>() &&
         configure32<kDense, false, false, TA, TB, true>();
}
bool prepare_dense32() {
  return prepare_tile<4, 4>() && prepare_tile<3, 4>() && prepare_tile<4, 3>() && prepare_tile<2, 4>() &&
         prepare_tile<4, 2>() && configure32<kDense, false, false, 4, 4, false, true>() && configure32<kSplitK, false, false, 4, 4>() &&
         configure32<kSplitK, false, false, 2, 4>() && configure32<kSplitK, false, false, 4, 2>();
}

void set_debug_grid(int g) { debug_grid = g; }
#ifdef MX_TIMING_BUILD
void set_debug_prof(uint64_t* buf) { debug_prof = buf; }
#endif

int launch_gemm_nt32(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                     const uint8_t* b_scales, void* d, int64_t M, int64_t N, int64_t K,
                     int64_t ldk, int64_t ldd, bool f32, hipStream_t st) {
  Gemm32Args p{a_codes, a_scales, b_codes, b_scales, (uint16_t*)d, M, N, K, ldd, nullptr, 0, 0, 0, debug_prof};
  p.ldk = ldk;
#ifdef MX_TIMING_BUILD
  if (debug_prof) return launch32<kDense, true>(p, ((M + kT32 - 1) / kT32) * ((N + kT32 - 1) / kT32), st);
#endif
  if (f32) return launch_best32<false, true>(p, st);
  return launch_best32(p, st);
}

// ---- split along K for shapes whose 256x256 tiles do not fill the CUs ----------------------
// Sum of the S float32 partial matrices [S][M][N], in slice order, rounded once to bf16 (F32: and written as
// float32).
template <bool F32>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ part, int S,
                                                            int64_t M, int64_t N,
                                                            uint16_t* __restrict__ d, int64_t ldd) {
  const int64_t per_row = N / 8, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= M * per_row) return;
  const int64_t r = i / per_row, c = (i - r * per_row) * 8;
  const float* src = part + r * N + c;
  float acc[8];
  {
    const v4f lo = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(src));
    const v4f hi = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(src) + 1);
    acc[0] = lo.x; acc[1] = lo.y; acc[2] = lo.z; acc[3] = lo.w;
    acc[4] = hi.x; acc[5] = hi.y; acc[6] = hi.z; acc[7] = hi.w;
  }
  for (int s = 1; s < S; ++s) {
    const float* q = src + (int64_t)s * M * N;
    const v4f lo = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(q));
    const v4f hi = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(q) + 1);
    acc[0] += lo.x; acc[1] += lo.y; acc[2] += lo.z; acc[3] += lo.w;
    acc[4] += hi.x; acc[5] += hi.y; acc[6] += hi.z; acc[7] += hi.w;
  }
  if constexpr (F32) {
    v4f* out = reinterpret_cast<v4f*>(reinterpret_cast<float*>(d) + r * ldd + c);
    out[0] = v4f{round_bf16(acc[0]), round_bf16(acc[1]), round_bf16(acc[2]), round_bf16(acc[3])};
    out[1] = v4f{round_bf16(acc[4]), round_bf16(acc[5]), round_bf16(acc[6]), round_bf16(acc[7])};
    return;
  }
  const u32x4 w = {pack_bf16(acc[0], acc[1]), pack_bf16(acc[2], acc[3]), pack_bf16(acc[4], acc[5]),
                   pack_bf16(acc[6], acc[7])};
  *reinterpret_cast<u32x4*>(d + r * ldd + c) = w;
}

int launch_splitk_reduce(const float* part, int slices, int64_t M, int64_t N, void* d, int64_t ldd, bool f32,
                         hipStream_t st) {
  const int64_t threads = M * (N / 8);
  hipLaunchKernelGGL(f32 ? splitk_reduce_kernel<true> : splitk_reduce_kernel<false>, dim3((unsigned)((threads + 255) / 256)),
                     dim3(256), 0, st, part, slices, M, N, (uint16_t*)d, ldd);
  return hipGetLastError() == hipSuccess ? MX_OK : MX_ERR_LAUNCH;
}

// D = sum over slices, through `workspace` (S * M * N floats).
int launch_gemm_nt32_splitk(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                            const uint8_t* b_scales, void* d, int64_t M, int64_t N, int64_t K,
                            int64_t ldk, int64_t ldd, const GemmPlan& plan, void* workspace, bool f32,
                            hipStream_t st) {
  Gemm32Args p{a_codes, a_scales, b_codes, b_scales, (uint16_t*)workspace, M, N, K, N, nullptr,
               plan.slices, 0, 0, nullptr};
  p.ldk = ldk;
  const int rc = launch_dense32<kSplitK>(p, plan.ta, plan.tb, st);
  if (rc != MX_OK) return rc;
  return launch_splitk_reduce((const float*)workspace, plan.slices, M, N, d, ldd, f32, st);
}

// Grouped forms with every group end a multiple of 32 and all scales in MFMA order
// (a_scales over the whole [T, K/32] matrix, b_scales one block per expert).  A workgroup keeps
// a record per tile in LDS, at most kMaxRecords of them: larger problems are cut into several
// launches over ranges of tile columns.
constexpr int64_t kMaxRecords = kMaxTileRecords;

template <int MODE, bool PAIR = false>
static int launch_grouped32(Gemm32Args p, int64_t tiles_per_column, int64_t tiles_n, hipStream_t st) {
  const int64_t grid = persistent_grid();
  if (grid == 0) return MX_ERR_LAUNCH;
  // tiles of one launch <= grid * kMaxRecords - slack for the rounding of the per-XCD runs
  // (PAIR: two records per tile)
  int64_t cols = (grid * (kMaxRecords / (PAIR ? 2 : 1)) - 8 * (grid / 8)) / tiles_per_column;
  if (cols < 1) return MX_ERR_UNSUPPORTED;
  if (cols > tiles_n) cols = tiles_n;
  for (int64_t tn0 = 0; tn0 < tiles_n; tn0 += cols) {
    p.tn0 = (int32_t)tn0;
    p.tn_cnt = (int32_t)(tiles_n - tn0 < cols ? tiles_n - tn0 : cols);
    const int64_t nb = tiles_per_column * p.tn_cnt;
    int rc;
    if constexpr (PAIR)
      rc = launch32<MODE, false, true>(p, nb, st);
    else {
#ifdef MX_TIMING_BUILD
      rc = p.prof ? launch32<MODE, true>(p, nb, st) : launch32<MODE, false>(p, nb, st);
#else
      rc = launch32<MODE, false>(p, nb, st);
#endif
    }
    if (rc != MX_OK) return rc;
  }
  return MX_OK;
}

int launch_grouped32_2d3d(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                          const uint8_t* b_scales, const int32_t* offs, void* d, int64_t T,
                          int64_t N, int64_t K, int64_t G, int64_t ldd, hipStream_t st) {
  Gemm32Args p{a_codes, a_scales, b_codes, b_scales, (uint16_t*)d, T, N, K, ldd, offs, G, 0, 0, debug_prof};
  // an upper bound of the tile rows: every group may add one partly filled tile
  return launch_grouped32<kGrouped2d3d>(p, (T + kT32 - 1) / kT32 + G + 1, (N + kT32 - 1) / kT32, st);
}

// D = A B^T and D2 = A B2^T in one launch (same shapes), dense and grouped 2D x 3D.
int launch_gemm_nt32_two_b(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                           const uint8_t* b_scales, const uint8_t* b2_codes, const uint8_t* b2_scales,
                           void* d, void* d2, int64_t M, int64_t N, int64_t K, int64_t ldk, int64_t ldd,
                           hipStream_t st) {
  Gemm32Args p{a_codes, a_scales, b_codes, b_scales, (uint16_t*)d, M, N, K, ldd, nullptr, 0, 0, 0, nullptr};
  p.b2_codes = b2_codes;
  p.b2_scales = b2_scales;
  p.two = kTwoB;
  p.d2 = (uint16_t*)d2;
  p.ldk = ldk;
  return launch_best32(p, st);
}
int launch_grouped32_2d3d_two_b(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                                const uint8_t* b_scales, const uint8_t* b2_codes, const uint8_t* b2_scales,
                                const int32_t* offs, void* d, void* d2, int64_t T, int64_t N, int64_t K,
                                int64_t G, int64_t ldd, hipStream_t st) {
  Gemm32Args p{a_codes, a_scales, b_codes, b_scales, (uint16_t*)d, T, N, K, ldd, offs, G, 0, 0, nullptr};
  p.b2_codes = b2_codes;
  p.b2_scales = b2_scales;
  p.two = kTwoB;
  p.d2 = (uint16_t*)d2;
  return launch_grouped32<kGrouped2d3d>(p, (T + kT32 - 1) / kT32 + G + 1, 2 * ((N + kT32 - 1) / kT32), st);
}
// D = A B^T and D2 = A2 B^T in one launch (same shapes), dense and grouped 2D x 2D.
int launch_gemm_nt32_two_a(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* a2_codes,
                           const uint8_t* a2_scales, const uint8_t* b_codes, const uint8_t* b_scales,
                           void* d, void* d2, int64_t M, int64_t N, int64_t K, int64_t ldk, int64_t ldd,
                           hipStream_t st) {
  Gemm32Args p{a_codes, a_scales, b_codes, b_scales, (uint16_t*)d, M, N, K, ldd, nullptr, 0, 0, 0, nullptr};
  p.a2_codes = a2_codes;
  p.a2_scales = a2_scales;
  p.two = kTwoA;
  p.d2 = (uint16_t*)d2;
  p.ldk = ldk;
  return launch_best32(p, st);
}
int launch_grouped32_2d2d_two_a(const uint8_t* at_codes, const uint8_t* at_scales, const uint8_t* at2_codes,
                                const uint8_t* at2_scales, const uint8_t* bt_codes, const uint8_t* bt_scales,
                                const int32_t* offs, void* d, void* d2, int64_t T, int64_t N, int64_t K,
                                int64_t G, hipStream_t st) {
  Gemm32Args p{at_codes, at_scales, bt_codes, bt_scales, (uint16_t*)d, N, K, T, K, offs, G, 0, 0, nullptr};
  p.a2_codes = at2_codes;
  p.a2_scales = at2_scales;
  p.two = kTwoA;
  p.d2 = (uint16_t*)d2;
  return launch_grouped32<kGrouped2d2d>(p, (G + 7) / 8 * 8 * 2 * ((N + kT32 - 1) / kT32), (K + kT32 - 1) / kT32, st);
}

// D = A B^T + A2 B2^T (dense) and its grouped 2D x 3D form: both operand sets of the same shapes.
int launch_gemm_nt32_pair(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                          const uint8_t* b_scales, const uint8_t* a2_codes, const uint8_t* a2_scales,
                          const uint8_t* b2_codes, const uint8_t* b2_scales, void* d, int64_t M,
                          int64_t N, int64_t K, int64_t ldk, int64_t ldd, hipStream_t st) {
  Gemm32Args p{a_codes, a_scales, b_codes, b_scales, (uint16_t*)d, M, N, K, ldd, nullptr, 0, 0, 0, nullptr,
               a2_codes, a2_scales, b2_codes, b2_scales};
  p.ldk = ldk;
  return launch_best32<true>(p, st);
}

// Whether the gated product of [M, K] with two weights of N rows leaves its product as codes: where that is predicted to be
// done before the two products and the cast of their gate.  The gate costs 6 us a round, also a last one of few tiles,
// which then does not pay: 288 tiles of 12 blocks (2270 x 4096, K 1536) 45 us in two launches and 50 gated, 352 of 16 (2048 x 5632,
// K 2048) 58 and 63, 518 of 15 (3533 x 4736, K 1920) 79 and 86.  Full rounds win (3001 x 8192, K 1024 75 and 65 us; 4096 x 6144,
// K 2048 105 and 96; 1500 x 4992, K 2048 38 and 35), tiles that leave half of the CUs idle lose to the smaller ones of the
// two launches (512 x 8192, K 3072 34 and 42).  Fitted to 228 shapes of 129..4600 rows, 1024..14336 columns and K 512..5400, on
// operands from the cache and from memory: of the 107 that it chooses none is slower, and the choice takes 0.1 % more than
// the better of both each time.  (4 us a round chose 134 of them, 19 slower by 3 to 13 %.)
bool plan_gated(int64_t M, int64_t N, int64_t K) {
  const int64_t grid = persistent_grid(), blocks = K / kKB;
  if (grid == 0) return false;
  const DenseTile* t = best_tile(M, N, blocks, 2, grid);
  if (!t) return false;
  double us = tiles_us(*t, 2 * tile_count(*t, M, N), blocks, grid) + 2.0;
  better_ring(M, N, blocks, 2, grid, us);
  const int64_t tiles = ((M + 255) / 256) * ((N + 127) / 128);
  const double gated = tiles_us(kDenseTiles[0], tiles, blocks, grid) + 1.0 + 6.0 * ((tiles + grid - 1) / grid);
  return gated < us + 2.0 + M * N / 1e6;
}
int launch_gemm_nt32_gated(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes, const uint8_t* b_scales,
                           const uint8_t* b2_codes, const uint8_t* b2_scales, uint8_t* codes, uint8_t* scales, int64_t M,
                           int64_t N, int64_t K, int64_t ldk, int64_t ld_codes, int scale_mode, hipStream_t st) {
  Gemm32Args p{a_codes, a_scales, b_codes, b_scales, (uint16_t*)codes, M, N, K, ld_codes, nullptr, 0, 0, 0, nullptr};
  p.b2_codes = b2_codes;
  p.b2_scales = b2_scales;
  p.d2 = (uint16_t*)scales;
  p.ldk = ldk;
  p.scale_mode = scale_mode;
  return launch32<kDense, false, false, 4, 4, false, true>(p, ((M + 255) / 256) * ((N + 127) / 128), st);
}

// ... in the slices of `plan`, through `workspace` (slices * M * N floats).
int launch_gemm_nt32_pair_splitk(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                                 const uint8_t* b_scales, const uint8_t* a2_codes, const uint8_t* a2_scales,
                                 const uint8_t* b2_codes, const uint8_t* b2_scales, void* d, int64_t M, int64_t N,
                                 int64_t K, int64_t ldk, int64_t ldd, const GemmPlan& plan, void* workspace,
                                 hipStream_t st) {
  Gemm32Args p{a_codes, a_scales, b_codes, b_scales, (uint16_t*)workspace, M, N, K, N, nullptr, plan.slices, 0, 0, nullptr,
               a2_codes, a2_scales, b2_codes, b2_scales};
  p.ldk = ldk;
  p.sets = 2;
  const int rc = launch_dense32<kSplitK>(p, plan.ta, plan.tb, st);
  if (rc != MX_OK) return rc;
  return launch_splitk_reduce((const float*)workspace, plan.slices, M, N, d, ldd, false, st);
}

int launch_grouped32_2d3d_pair(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                               const uint8_t* b_scales, const uint8_t* a2_codes,
                               const uint8_t* a2_scales, const uint8_t* b2_codes,
                               const uint8_t* b2_scales, const int32_t* offs, void* d, int64_t T,
                               int64_t N, int64_t K, int64_t G, int64_t ldd, hipStream_t st) {
  Gemm32Args p{a_codes, a_scales, b_codes, b_scales, (uint16_t*)d, T, N, K, ldd, offs, G, 0, 0, nullptr,
               a2_codes, a2_scales, b2_codes, b2_scales};
  return launch_grouped32<kGrouped2d3d, true>(p, (T + kT32 - 1) / kT32 + G + 1, (N + kT32 - 1) / kT32, st);
}

// Grouped 2D x 3D (one product, or with a2_codes the sum of two) whose output leaves the groups'
// padding out: see Gemm32Args::d_offs.
int launch_grouped32_2d3d_rows_out(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                                   const uint8_t* b_scales, const uint8_t* a2_codes,
                                   const uint8_t* a2_scales, const uint8_t* b2_codes,
                                   const uint8_t* b2_scales, const int32_t* offs, const int32_t* d_offs,
                                   void* d, int64_t T, int64_t d_rows, int64_t N, int64_t K, int64_t G,
                                   int64_t ldd, hipStream_t st) {
  Gemm32Args p{a_codes, a_scales, b_codes, b_scales, (uint16_t*)d, T, N, K, ldd, offs, G, 0, 0, nullptr,
               a2_codes, a2_scales, b2_codes, b2_scales};
  p.d_offs = d_offs;
  p.d_rows = d_rows;
  const int64_t tile_rows = (T + kT32 - 1) / kT32 + G + 1, tiles_n = (N + kT32 - 1) / kT32;
  if (a2_codes) return launch_grouped32<kGrouped2d3d, true>(p, tile_rows, tiles_n, st);
  return launch_grouped32<kGrouped2d3d>(p, tile_rows, tiles_n, st);
}

// D[g][N, K] = A^T[N, lo:hi] B^T[K, lo:hi]^T; operand rows are T long.
int launch_grouped32_2d2d(const uint8_t* at_codes, const uint8_t* at_scales,
                          const uint8_t* bt_codes, const uint8_t* bt_scales, const int32_t* offs,
                          void* d, int64_t T, int64_t N, int64_t K, int64_t G, hipStream_t st) {
  Gemm32Args p{at_codes, at_scales, bt_codes, bt_scales, (uint16_t*)d, N, K, T, K, offs, G, 0, 0, debug_prof};
  // tiles per column counted with G rounded up to the 8 XCDs: the kernel deals whole groups to
  // XCDs, and the busiest XCD's share must fit its workgroups' records
  return launch_grouped32<kGrouped2d2d>(p, (G + 7) / 8 * 8 * ((N + kT32 - 1) / kT32), (K + kT32 - 1) / kT32, st);
}

}  // namespace mx
