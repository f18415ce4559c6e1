// fp16 "NT" GEMM core on the gfx950 matrix cores with direct global -> LDS loads:
// C[m][n] = sum_k A[m][k] B[n][k], fp32 accumulation in v_mfma_f32_32x32x16_f16 tiles, the
// accumulators handed to an epilogue functor.
//
// Operand tiles travel HBM/L2 -> LDS through global_load_lds_dwordx4: the data never passes
// through VGPRs, so the load path costs one issue slot per 16 bytes and no registers. Each
// such instruction writes 64 consecutive 16-byte LDS slots (M0 base + 16 * lane); the XOR
// swizzle of the LDS rows (swz()) is therefore applied on the global side: the lane that owns
// LDS slot (row, physical chunk) fetches logical chunk physical ^ swz(row) of that row.
// Rows past the operands' end are fetched from the last valid row (they feed only outputs that are
// never stored), so a tile at the edge costs nothing more; columns past k_len are fetched from a
// 16-byte zero block (hidden sizes are multiples of 8, so a 16-byte chunk is either wholly inside
// or wholly outside).
//
// The LDS holds a ring of SA stages of A and SB of B, each of 64 columns; the loads of stage
// kt + SA - 1 of A and kt + SB - 1 of B are issued while stage kt is multiplied. One barrier per
// stage: after it every wavefront has finished reading stage kt - 1 (so its buffers can be
// refilled) and every wavefront's loads of stage kt have landed.
//
// An A-fragment transform FX may rescale each 8-element A fragment between the LDS read and the
// MFMA (used by the LM head's gradient GEMM to turn stored e^{z - m} into probabilities). The
// epilogue's prepare() runs before the main loop (to issue its own loads early), start() gives
// the accumulators their initial values (it may issue loads) and started() runs after the
// prologue's loads; apply() receives the accumulators and the LDS ring, which it may reuse
// after a barrier. ZeroStart is the plain start (zero accumulators).
#pragma once

#include <type_traits>
#include <utility>

#include "common.h"
#include "gemm_nt.h"

namespace cm {
namespace gemm {

// Source of the chunks that lie outside an operand.
static __device__ const uint4 kZeroChunk[1] = {{0u, 0u, 0u, 0u}};

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// One global_load_lds_dwordx4: 64 lanes x 16 bytes into 64 consecutive 16-byte LDS slots from
// lds_slot0 (wave-uniform, passed in M0). Issued through inline assembly: the compiler models the
// builtin like a FLAT access that may complete out of order with LDS reads, and then turns every
// later fragment wait into lgkmcnt(0), which ties the LDS reads of each substep to the freshly
// issued ds_reads. Completion of these loads is waited for explicitly (wait_vmcnt before the
// stage barrier); a counter the compiler does not know about can only make its own waits
// longer, never shorter.
// M0 is set inside the statement; no other code in these kernels keeps a value in M0.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(const void* g, uint4* lds_slot0) {
  const uint32_t m0v = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr_t)lds_slot0));
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :
               : "s"(m0v), "v"(g)
               : "memory", "m0");
}
#pragma clang diagnostic pop

// s_waitcnt vmcnt(n) with the other counters left alone (gfx9 encoding: vmcnt in bits 3:0 and
// 15:14, expcnt 6:4, lgkmcnt 11:8).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// LDS operand tiles of ROWS rows x BK fp16 columns = BK / 8 chunks of 16 bytes per row, in one of
// two layouts, chosen per operand by its source layout (Src::kChunkMajor):
//  - row-major (CM = false): slot row * kRC + (chunk ^ swz(row)). The XOR swizzle is chosen for
//    the 64 banks of 4 bytes of the gfx950 LDS: a ds_read_b128 is served 16 lanes (256 bytes)
//    at a time, and the 16 lanes of a fragment read are 16 consecutive rows at one logical
//    chunk, so those rows must land in 16 distinct 16-byte bank groups. With 8-chunk rows the
//    row parity already picks the half of the 256-byte bank span and (row >> 1) & 7 the chunk;
//    with 4-chunk rows row & 3 picks the quarter and (row >> 2) & 3 the chunk. A wavefront's
//    direct load then fetches 8 rows x 128 bytes, the right shape for row-contiguous sources.
//  - chunk-major (CM = true): slot chunk * ROWS + row. A fragment read's 16 rows are 16
//    consecutive slots (conflict-free with no swizzle), and a wavefront's direct load fetches 64
//    consecutive rows at one chunk: two 512-byte spans of a Tiled32 source.
template <int BK, bool CM, int ROWS>
struct LdsTile {
  static constexpr int kRC = BK / 8;
  static_assert(kRC == 8 || kRC == 4, "stages of 64 or 32 columns");
  static __device__ __forceinline__ int swz(int row) {
    return kRC == 8 ? ((row >> 1) & 7) : ((row >> 2) & 3);
  }
  static __device__ __forceinline__ int slot(int row, int ch) {
    return CM ? ch * ROWS + row : row * kRC + (ch ^ swz(row));
  }
  static __device__ __forceinline__ half8 frag(const uint4* lds, int row, int ch) {
    return __builtin_bit_cast(half8, lds[slot(row, ch)]);
  }
};

// The row-major layout on its own (its slots do not depend on the tile's row count).
template <int BK>
using LdsRows = LdsTile<BK, false, 0>;

// Direct loads of one ROWS x BK operand tile by NW wavefronts. Instruction i of a lane fills
// LDS slot (i * NW + wave) * 64 + lane of the tile: row-major, row row0 + i * kRowStep and (with
// NW >= 2) the same swizzled column for every i, since kRowStep is a multiple of the swizzle's
// period; chunk-major, row row0 and column col0 + 8 i * kColStep. A lane keeps one byte offset
// per instruction from the stage's origin, a wave-uniform pointer; rows past the operand's end
// are already replaced in it (clamp_row), so a row edge takes no test in the loop (testing and
// selecting per load cost 16 us of 93 where one tile row of five was partial: 1276 x 1536 x 17920).
template <int ROWS, int NW, int BK, bool CM = false>
struct DmaTile {
  using L = LdsTile<BK, CM, ROWS>;
  static constexpr int kChunks = ROWS * L::kRC;
  static constexpr int kPer = kChunks / (NW * kWave);  // instructions per lane
  static constexpr int kRowStep = CM ? 0 : NW * kWave / L::kRC;  // tile rows between them
  static constexpr int kColStep = CM ? NW * kWave / ROWS : 0;    // chunks between them
  static_assert(kPer * NW * kWave == kChunks, "tile chunks must split over the wavefronts");
  static_assert(CM || NW >= 2, "one swizzled column per lane needs a row step of 16 or more");
  static_assert(!CM || kColStep * ROWS == NW * kWave, "an instruction covers whole chunk columns");
  // byte offset of the lane's chunk of instruction i from the stage origin (chunk-major:
  // instruction 0's, the others a constant step apart)
  uint32_t off[CM ? 1 : kPer];
  int col0;  // tile column of the lane's chunk of instruction 0

  // r0: the tile's first row (a valid one)
  template <class Src>
  __device__ __forceinline__ void init(const Src& src, int r0, int wave, int lane) {
    const int c = wave * kWave + lane;
    const int row0 = CM ? c % ROWS : c / L::kRC;
    col0 = CM ? (c / ROWS) * 8 : ((c % L::kRC) ^ L::swz(row0)) * 8;
#pragma unroll
    for (int i = 0; i < (CM ? 1 : kPer); ++i)
      off[i] = src.tile_offset(src.clamp_row(r0, row0 + i * kRowStep), col0);
  }
  template <class Src>
  __device__ __forceinline__ uint32_t offset(int i) const {
    if constexpr (CM) return off[0] + i * kColStep * Src::kChunkBytes;
    else return off[i];
  }

  // Instruction i of the stage whose origin is (r0, k0), a stage wholly inside k_len.
  template <class Src>
  __device__ __forceinline__ void issue_inside(const Src& src, int r0, int k0, uint4* tile,
                                               int wave, int i) const {
    const char* base = reinterpret_cast<const char*>(src.at(r0, k0));
    dma16(base + offset<Src>(i), tile + (i * NW + wave) * kWave);
  }

  // Instruction i of the stage whose origin is (r0, k0); `inside` = the stage lies wholly inside
  // k_len (wave-uniform).
  template <class Src>
  __device__ __forceinline__ void issue(const Src& src, int r0, int k0, uint4* tile, int wave,
                                        int i, bool inside) const {
    const char* base = reinterpret_cast<const char*>(src.at(r0, k0));
    const bool ok = inside || src.col_ok(k0 + col0 + i * kColStep * 8);
    const void* g = ok ? static_cast<const void*>(base + offset<Src>(i))
                       : static_cast<const void*>(kZeroChunk);
    dma16(g, tile + (i * NW + wave) * kWave);
  }
};

// Direct loads of a row-major LDS tile from a SegRows operand: as DmaTile, but a lane keeps its
// (clamped) rows, because the row stride changes with the stage's segment: one multiply-add per
// instruction.
template <int ROWS, int NW, int BK>
struct DmaTileSeg {
  using L = LdsTile<BK, false, ROWS>;
  static constexpr int kPer = ROWS * L::kRC / (NW * kWave);
  static constexpr int kRowStep = NW * kWave / L::kRC;
  static_assert(kPer * NW * kWave == ROWS * L::kRC, "tile chunks must split over the wavefronts");
  static_assert(NW >= 2, "one swizzled column per lane needs a row step of 16 or more");
  int row[kPer];
  int col0;

  template <class Src>
  __device__ __forceinline__ void init(const Src& src, int r0, int wave, int lane) {
    const int c = wave * kWave + lane, row0 = c / L::kRC;
    col0 = ((c % L::kRC) ^ L::swz(row0)) * 8;
#pragma unroll
    for (int i = 0; i < kPer; ++i) row[i] = min(row0 + i * kRowStep, src.rows - 1 - r0);
  }
  template <class Src>
  __device__ __forceinline__ void issue_inside(const Src& src, int r0, int k0, uint4* tile,
                                               int wave, int i) const {
    int64_t ld;
    const _Float16* base = src.at(r0, k0, ld);
    const uint32_t off = (row[i] * static_cast<uint32_t>(ld) + col0) * 2;
    dma16(reinterpret_cast<const char*>(base) + off, tile + (i * NW + wave) * kWave);
  }
  template <class Src>
  __device__ __forceinline__ void issue(const Src& src, int r0, int k0, uint4* tile, int wave,
                                        int i, bool) const {
    issue_inside(src, r0, k0, tile, wave, i);  // segments are whole stages
  }
};

// Direct loads of a k-major operand (KMajor): the LDS tile is BK rows (k) of BN fp16 (n), row by
// row, with the 32-byte segments of a row XOR-swizzled by kswz(k): 2 (k & 3) where rows are whole
// multiples of 256 bytes (the 64 banks), else 2 ((k >> 1) & 1) (neighbouring rows of an odd number
// of 128-byte halves already start half the banks apart). A transposing fragment read
// (frag_kmajor) has its 16-lane groups read rows k .. k + 3 (k a multiple of 4) at one 32-byte
// segment and the next, so with this swizzle the 8 (row, segment) pieces a 32-lane half serves at
// once cover the 64 banks exactly once. Instruction i of a lane fills slot c = (i NW + wave) 64 + lane of the tile: row
// c / (BN / 8), physical slot c % (BN / 8). As in DmaTile, a lane keeps one byte offset per
// instruction; chunks past the operand's last n are read from its last whole chunk.
template <int BN, int NW, int BK>
struct DmaTileK {
  static constexpr int kSlotsRow = BN / 8;
  static constexpr int kChunks = BK * kSlotsRow;
  static constexpr int kPer = kChunks / (NW * kWave);
  static_assert(kPer * NW * kWave == kChunks, "tile chunks must split over the wavefronts");
  static_assert(BN % 64 == 0, "rows of whole groups of four 32-byte segments");
  static __device__ __forceinline__ int kswz(int k) {
    return BN % 128 == 0 ? (k & 3) * 2 : ((k >> 1) & 1) * 2;
  }
  uint32_t off[kPer];  // byte offset of the lane's chunk of instruction i from the stage origin
  int krow[kPer];

  template <class Src>
  __device__ __forceinline__ void init(const Src& src, int n0, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int c = (i * NW + wave) * kWave + lane;
      const int k = c / kSlotsRow, ps = c % kSlotsRow;
      const int ls = (((ps >> 1) ^ kswz(k)) << 1) | (ps & 1);  // logical slot of the row
      krow[i] = k;
      const int n = min(ls * 8, (src.rows - n0 - 1) & ~7);
      off[i] = static_cast<uint32_t>((static_cast<int64_t>(k) * src.ld + n) * 2);
    }
  }
  template <class Src>
  __device__ __forceinline__ void issue_inside(const Src& src, int n0, int k0, uint4* tile,
                                               int wave, int i) const {
    const char* base = reinterpret_cast<const char*>(src.at(n0, k0));
    dma16(base + off[i], tile + (i * NW + wave) * kWave);
  }
  template <class Src>
  __device__ __forceinline__ void issue(const Src& src, int n0, int k0, uint4* tile, int wave,
                                        int i, bool inside) const {
    const char* base = reinterpret_cast<const char*>(src.at(n0, k0));
    const bool ok = inside || k0 + krow[i] < src.k_len;
    const void* g = ok ? static_cast<const void*>(base + off[i])
                       : static_cast<const void*>(kZeroChunk);
    dma16(g, tile + (i * NW + wave) * kWave);
  }
};

typedef short short4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4v lds_short4_t;

// The B fragment of v_mfma_f32_32x32x16_f16 (lane l: n = l % 32 of the 32-column tile at n_base,
// k = ks * 16 + (l / 32) * 8 .. + 7) from a k-major LDS tile of BN columns, as two
// ds_read_b64_tr_b16. That instruction (lane layout checked by a probe kernel) gives lane i of each
// 16-lane group element i % 4 of the 8 bytes that lane 4 j + i / 4 of the group addressed, for
// j = 0 .. 3: so lane a of group g addresses row k0 + a / 4, columns n_base + 16 (g % 2) +
// 4 (a % 4) .. + 3, and lane i receives rows k0 .. k0 + 3 of column n_base + 16 (g % 2) + i.
template <int BN>
__device__ __forceinline__ half8 frag_kmajor(const uint4* tile, int n_base, int ks, int lane) {
  const int g = lane / 16, a = lane % 16;
  const int n = n_base + (g % 2) * 16 + 4 * (a % 4);
  const int k = ks * 16 + (g / 2) * 8 + a / 4;
  const int seg = (n / 16) ^ DmaTileK<BN, 1, 16>::kswz(k);  // kswz(k + 4) == kswz(k)
  const char* row = reinterpret_cast<const char*>(tile) + k * (BN * 2) + seg * 32 + (n % 16) * 2;
  const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)(row));
  const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)(row + 4 * BN * 2));
  const short4v v[2] = {lo, hi};
  return __builtin_bit_cast(half8, v);
}

// Workgroup barrier that orders LDS only: the loads into LDS are waited for explicitly
// (vmcnt), so the barrier must not wait for every outstanding global load.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The same without a wait for the wavefront's own LDS reads, for a loop whose buffers are refilled no
// earlier than two barriers after their last read (by then the arithmetic that uses the values has
// waited for them). The compiler moves no memory access across it; the fences emit nothing.
__device__ __forceinline__ void lds_barrier_reads_pending() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "singlethread");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "singlethread");
  __builtin_amdgcn_sched_barrier(0);
}

// Accumulators starting at zero, for epilogues with nothing to add to the product.
struct ZeroStart {
  template <int TM, int TN>
  static __device__ __forceinline__ void start(floatx16 (&acc)[TM][TN], int, int, int) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  }
  template <int TM, int TN>
  static __device__ __forceinline__ void started(floatx16 (&)[TM][TN]) {}
};

// Compile-time loop: f(std::integral_constant<int, 0>) .. f(std::integral_constant<int, N - 1>).
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// Identity A-fragment transform (the default FX of gemm_lds). An FX may stage data of its own with
// the A operand: kDma direct loads per wavefront and stage (issue(k0, slot), the last of A's loads
// of the stage at column k0 into ring slot `slot`), fetch(slot) reads it back into registers at
// the start of the stage, and apply(frag, i) transforms the A fragment of the wavefront's tile
// row i.
struct PlainA {
  static constexpr int kDma = 0;
  __device__ __forceinline__ void issue(int, int) const {}
  __device__ __forceinline__ void fetch(int) {}
  __device__ __forceinline__ half8 apply(half8 f, int) const { return f; }
};

// Bounds handling of the operand loads' columns (EDGE): kEdgeEither picks per workgroup (a second
// copy of the main loop without bounds selection, taken when every stage lies inside both
// operands' k_len), kEdgeAlways always selects, kEdgeNever never does (the caller guarantees whole
// stages: one loop, for kernels where two copies would not fit the registers).
enum EdgeMode { kEdgeEither = 0, kEdgeAlways = 1, kEdgeNever = 2 };

// Main loop, per stage kt: wait until stage kt has landed and this wavefront's fragment reads of
// stage kt - 1 have returned, one barrier, then four groups of TM x TN MFMAs: the last 16-column
// substep of stage kt - 1 (its fragments are already in registers, so these MFMAs cover the
// latency of the first fragment reads of stage kt), then substeps 0 .. 2 of stage kt. The groups
// are walked in slots of one MFMA: the first slots of a group also read one fragment of the next
// substep each, and the stage's direct loads are spread evenly over the slots of all four groups
// (of their first halves when both rings hold two stages), B's before A's when A's ring is the
// deeper one. sched_barrier pins the order.
//
// What bounds it: the direct loads' issue. A CU takes one 1 KiB load instruction per ~16 cycles
// (64 bytes per cycle, 57 measured), so several in a row from every wavefront at once hold the
// wavefronts with the matrix cores idle; four in a row per group (an earlier form of this loop)
// cost a quarter of the time: 8192 x 7680 x 8192 in 950 us with them, 715 us with the loads left
// out, 922 us with the fragment reads left out. One load every four MFMAs needs a longer way
// from issue to use than two stages give (the last load of a stage is then issued just before
// the wait), hence the third stage of A; B, issued first, has half a stage and more. And a loop
// without branches: the stages that load nothing, or only B, are separate copies. Together
// 846 us, and 211 -> 176 us at 2048 x 1536 x 32768 in 4 slices with B k-major.
template <int BM, int BN, int WM, int WN, int SA, int SB, class SrcA, class SrcB, class Epi,
          class FX = PlainA, int EDGE = kEdgeEither>
__device__ __forceinline__ void gemm_lds(const SrcA& A, const SrcB& B, int k_begin, int k_end,
                                         int tm, int tn, Epi& epi, uint4* lds, FX fx = FX()) {
  constexpr int BK = 64;
  constexpr int NW = WM * WN;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / 32, TN = WTN / 32;
  using LA = LdsTile<BK, SrcA::kChunkMajor, BM>;
  using LB = LdsTile<BK, SrcB::kChunkMajor, BN>;
  constexpr int KS = BK / 16;  // MFMA substeps per stage
  static_assert(TM * 32 == WTM && TN * 32 == WTN, "wave tiles are multiples of 32");
  static_assert(SB >= 2 && (SA == SB || SA == SB + 1), "A's ring is B's or one stage deeper");
  static_assert(NW * kWave >= 128, "tiles are loaded by at least two wavefronts");
  constexpr int kTileA = BM * LA::kRC, kTileB = BN * LB::kRC;  // uint4 per stage
  using TA = std::conditional_t<SrcA::kSegmented, DmaTileSeg<BM, NW, BK>,
                                DmaTile<BM, NW, BK, SrcA::kChunkMajor>>;
  static_assert(!SrcA::kKMajor, "a k-major operand is B");
  using TB = std::conditional_t<SrcB::kKMajor, DmaTileK<BN, NW, BK>,
                                DmaTile<BN, NW, BK, SrcB::kChunkMajor>>;
  constexpr int kDmaA = TA::kPer + FX::kDma;  // direct loads per lane per stage
  constexpr int kDmaB = TB::kPer;
  constexpr int kDma = kDmaA + kDmaB;
  constexpr int DA = SA - 1, DB = SB - 1;  // stages from issue to use
  // loads of later stages that may still be in flight when stage kt is needed: those issued after
  // B's of stage kt
  constexpr int kLate = (DB - 1) * kDma + (DA > DB ? kDmaA : 0);
  constexpr int NM = TM * TN, NR = TM + TN;  // MFMAs and fragments per substep
  constexpr int kSlots = NM > NR ? NM : NR;
  const int m0 = tm * BM, n0 = tn * BN;
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wm = wave / WN, wn = wave % WN;
  uint4* const lds_b = lds + SA * kTileA;
  TA la;
  TB lb;
  la.init(A, m0, wave, lane);
  lb.init(B, n0, wave, lane);
  epi.template prepare<TM, TN>(m0 + wm * WTM, n0 + wn * WTN, lane);

  // The epilogue's start() sets the accumulators (zero, or loads issued here so that they are
  // in flight with the first stage's loads); started() runs once the first stage has landed.
  floatx16 acc[TM][TN];
  epi.template start<TM, TN>(acc, m0 + wm * WTM, n0 + wn * WTN, lane);

  const int n_kt = (k_end - k_begin + BK - 1) / BK;
  auto inside_a = [&](int kt) { return A.k_inside(k_begin + kt * BK); };
  auto inside_b = [&](int kt) { return B.k_inside(k_begin + kt * BK); };
  // Every stage lies inside both operands' columns (the common case: the bounds tests are
  // monotonic in the stage, so the last stage decides); the main loop then issues its loads with
  // no bounds selection.
  const bool all_inside = n_kt > 0 && inside_a(n_kt - 1) && inside_b(n_kt - 1);
  // load instruction i of an operand's stage kt into ring slot `slot`
  auto load_a = [&](int kt, int slot, int i, auto edge) {
    const int k0 = k_begin + kt * BK;
    if (i >= TA::kPer) fx.issue(k0, slot);
    else if constexpr (decltype(edge)::value)
      la.issue(A, m0, k0, lds + slot * kTileA, wave, i, inside_a(kt));
    else la.issue_inside(A, m0, k0, lds + slot * kTileA, wave, i);
  };
  auto load_b = [&](int kt, int slot, int i, auto edge) {
    const int k0 = k_begin + kt * BK;
    if constexpr (decltype(edge)::value)
      lb.issue(B, n0, k0, lds_b + slot * kTileB, wave, i, inside_b(kt));
    else lb.issue_inside(B, n0, k0, lds_b + slot * kTileB, wave, i);
  };
  // ring slots of the current stage (counted up: a remainder by three per use costs more); the
  // stage loaded SA - 1 ahead goes into the slot before it
  int slot_a = 0, slot_b = 0;
  const int arow = wm * WTM + lane % 32, brow = wn * WTN + lane % 32;
  half8 af[2][TM], bf[2][TN];
  // fragment r of substep ks, alternately of A and of B while both have one left: is_a(r) / its
  // tile row or column
  constexpr int kBoth = TM < TN ? TM : TN;
  auto is_a = [](int r) { return r < 2 * kBoth ? r % 2 == 0 : TM > TN; };
  auto index_of = [](int r) { return r < 2 * kBoth ? r / 2 : r - kBoth; };
  auto read = [&](int ks, int buf, auto rc) {
    constexpr int r = decltype(rc)::value;
    const int ch = ks * 2 + lane / 32, x = index_of(r);
    if (is_a(r)) {
      af[buf][x] = LA::frag(lds + slot_a * kTileA, arow + x * 32, ch);
    } else {
      const uint4* Bs = lds_b + slot_b * kTileB;
      if constexpr (SrcB::kKMajor) bf[buf][x] = frag_kmajor<BN>(Bs, wn * WTN + x * 32, ks, lane);
      else bf[buf][x] = LB::frag(Bs, brow + x * 32, ch);
    }
  };
  auto mfma = [&](int b, int g) {
    const int i = g / TN, j = g % TN;
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[b][i], bf[b][j], acc[i][j], 0, 0, 0);
  };

  // Prologue: the loads of the first stages, in the order in which the loop would issue them.
  static_for<DA>([&](auto sc) {
    constexpr int s = decltype(sc)::value;
    if (s < DB && s < n_kt) {
#pragma unroll
      for (int i = 0; i < kDmaB; ++i) load_b(s, s, i, std::true_type{});
    }
    if (s < n_kt) {
#pragma unroll
      for (int i = 0; i < kDmaA; ++i) load_a(s, s, i, std::true_type{});
    }
  });

  // Waits for the prologue's loads (the first stage and whatever start() issued).
  epi.template started<TM, TN>(acc);

  // Direct load q of stage kt's slots: B's of stage kt + DB, then A's of stage kt + DA. LOADS: 2
  // both, 1 B's alone, 0 none.
  auto load = [&](int kt, int q, auto loads, auto edge) {
    if (q < kDmaB) {
      if constexpr (decltype(loads)::value >= 1)
        load_b(kt + DB, slot_b == 0 ? SB - 1 : slot_b - 1, q, edge);
    } else {
      if constexpr (decltype(loads)::value == 2)
        load_a(kt + DA, slot_a == 0 ? SA - 1 : slot_a - 1, q - kDmaB, edge);
    }
  };
  constexpr int kSpread = KS * NM / (DA > 1 ? 1 : 2);  // MFMA slots the loads are spread over
  // Group g of stage kt: reads the fragments of substep g (an FX is applied a few slots after its
  // fragment's read), multiplies those of the substep before.
  auto group = [&](int kt, auto gc, auto multiply, auto loads, auto edge) {
    constexpr int g = decltype(gc)::value, buf = g & 1;
    if constexpr (g == 0) fx.fetch(slot_a);
    static_for<kSlots>([&](auto mc) {
      constexpr int m = decltype(mc)::value;
      if constexpr (m < NR) read(g, buf, mc);
      if constexpr (m < NM && decltype(multiply)::value) mfma(buf ^ 1, m);
      if constexpr (FX::kDma > 0) {
        constexpr int kLag = kSlots - NR < 5 ? kSlots - NR : 5;
        constexpr int r = m - kLag;
        if constexpr (r >= 0 && r < NR)
          if (is_a(r)) af[buf][index_of(r)] = fx.apply(af[buf][index_of(r)], index_of(r));
      }
      static_for<kDma>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if constexpr ((2 * q + 1) * kSpread / (2 * kDma) == g * NM + m && m < NM)
          load(kt, q, loads, edge);
      });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  auto stage = [&](int kt, auto first, auto loads, auto edge) {
    if (kLate > 0 && kt + DA - 1 < n_kt) {  // none of them was left out
      wait_vmcnt<kLate>();
    } else {
      wait_vmcnt<0>();
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): own fragment reads have landed
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
    static_for<KS>([&](auto gc) {
      constexpr bool kMul = decltype(gc)::value > 0 || !decltype(first)::value;
      group(kt, gc, std::bool_constant<kMul>{}, loads, edge);
    });
    slot_a = slot_a == SA - 1 ? 0 : slot_a + 1;
    slot_b = slot_b == SB - 1 ? 0 : slot_b + 1;
  };
  static_assert(KS % 2 == 0, "substep buffers alternate within a stage");
  using Zero = std::integral_constant<int, 0>;
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  auto run = [&](auto edge) {
    if (n_kt <= 0) return;
    if (DA < n_kt) stage(0, std::true_type{}, Two{}, edge);
    else if (DA > DB && DB < n_kt) stage(0, std::true_type{}, One{}, edge);
    else stage(0, std::true_type{}, Zero{}, edge);
    int kt = 1;
    for (; kt + DA < n_kt; ++kt) stage(kt, std::false_type{}, Two{}, edge);
    if constexpr (DA > DB)
      for (; kt + DB < n_kt; ++kt) stage(kt, std::false_type{}, One{}, edge);
    for (; kt < n_kt; ++kt) stage(kt, std::false_type{}, Zero{}, edge);
  };
  if constexpr (EDGE == kEdgeEither) {
    if (all_inside) {
      run(std::false_type{});
    } else {
      run(std::true_type{});
    }
  } else {
    (void)all_inside;
    run(std::bool_constant<EDGE == kEdgeAlways>{});
  }
  if (n_kt > 0) {
#pragma unroll
    for (int g = 0; g < NM; ++g) mfma(1, g);
  }
  epi.template apply<TM, TN>(acc, m0 + wm * WTM, n0 + wn * WTN, lane, lds);
}

// The same product for small wavefront tiles (64 x 64 and below), whose substep is too few MFMAs to
// cover an LDS read: the fragments of a whole stage are in registers, and while stage kt - 1 is
// multiplied substep by substep, the registers of each finished substep are refilled from stage kt.
// A fragment then has three substeps of MFMAs to arrive in. One ring of S stages of both operands,
// loaded S - 2 stages ahead: the slot that stage kt's loads fill was last read two barriers ago, so
// the barrier waits for no fragment read. With SLICED the n_kt stages are summed in `slices` parts of
// their own, stages [s n_kt / slices, (s + 1) n_kt / slices), added in order: the sums of a contraction
// split over workgroups. Slices have at least D + 3 stages.
template <int BM, int BN, int WM, int WN, int S, bool SLICED, class SrcA, class SrcB, class Epi>
__device__ __forceinline__ void gemm_lds_small(const SrcA& A, const SrcB& B, int k_begin, int k_end,
                                               int tm, int tn, Epi& epi, uint4* lds,
                                               int slices = 1) {
  constexpr int BK = 64, NW = WM * WN, KS = BK / 16, D = S - 2;
  constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / 32, TN = WTN / 32;
  static_assert(TM * 32 == WTM && TN * 32 == WTN, "wave tiles are multiples of 32");
  static_assert(D >= 1, "a ring of at least three stages");
  using LA = LdsTile<BK, false, BM>;
  using LB = LdsTile<BK, false, BN>;
  constexpr int kTileA = BM * LA::kRC, kStage = (BM + BN) * LA::kRC;
  using TA = std::conditional_t<SrcA::kSegmented, DmaTileSeg<BM, NW, BK>, DmaTile<BM, NW, BK>>;
  using TB = std::conditional_t<SrcB::kKMajor, DmaTileK<BN, NW, BK>, DmaTile<BN, NW, BK>>;
  constexpr int kDma = TA::kPer + TB::kPer, NM = TM * TN, NR = TM + TN;
  const int m0 = tm * BM, n0 = tn * BN;
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wm = wave / WN, wn = wave % WN;
  TA la;
  TB lb;
  la.init(A, m0, wave, lane);
  lb.init(B, n0, wave, lane);
  epi.template prepare<TM, TN>(m0 + wm * WTM, n0 + wn * WTN, lane);
  floatx16 acc[TM][TN];
  epi.template start<TM, TN>(acc, m0 + wm * WTM, n0 + wn * WTN, lane);
  const int n_kt = (k_end - k_begin + BK - 1) / BK;
  auto load = [&](int kt, int q) {
    uint4* st = lds + (kt % S) * kStage;
    const int k0 = k_begin + kt * BK;
    if (q < TA::kPer) la.issue_inside(A, m0, k0, st, wave, q);
    else lb.issue_inside(B, n0, k0, st + kTileA, wave, q - TA::kPer);
  };
  const int arow = wm * WTM + lane % 32, brow = wn * WTN + lane % 32;
  half8 af[KS][TM], bf[KS][TN];
  auto read = [&](const uint4* st, int ks, int r) {
    const int ch = ks * 2 + lane / 32;
    if (r < TM) {
      af[ks][r] = LA::frag(st, arow + r * 32, ch);
    } else if constexpr (SrcB::kKMajor) {
      bf[ks][r - TM] = frag_kmajor<BN>(st + kTileA, wn * WTN + (r - TM) * 32, ks, lane);
    } else {
      bf[ks][r - TM] = LB::frag(st + kTileA, brow + (r - TM) * 32, ch);
    }
  };
  // fresh: the sum starts anew with substep 0
  auto mfma = [&](int ks, int g, auto fresh) {
    const int i = g / TN, j = g % TN;
    const floatx16 c = decltype(fresh)::value && ks == 0 ? floatx16{} : acc[i][j];
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[ks][i], bf[ks][j], c, 0, 0, 0);
  };
  static_for<D>([&](auto sc) {
    constexpr int s = decltype(sc)::value;
    if (s < n_kt) {
#pragma unroll
      for (int q = 0; q < kDma; ++q) load(s, q);
    }
  });
  epi.template started<TM, TN>(acc);
  auto stage = [&](int kt, auto first, auto loads, auto fresh) {
    // the loads of stages kt + 1 .. kt + D - 1 may still be in flight when all were issued
    if (D > 1 && kt + D - 1 < n_kt) wait_vmcnt<(D - 1) * kDma>();
    else wait_vmcnt<0>();
    lds_barrier_reads_pending();
    const uint4* st = lds + (kt % S) * kStage;
    constexpr int kStep = NM > NR ? NM : NR;  // slots per substep
    // substep s's slots multiply it and read substep s - 1 of the new stage
    static_for<(KS + 1) * kStep>([&](auto sc) {
      constexpr int slot = decltype(sc)::value, ks = slot / kStep, m = slot % kStep;
      if constexpr (ks < KS && m < NM && !decltype(first)::value) mfma(ks, m, fresh);
      if constexpr (ks > 0 && m < NR) read(st, ks - 1, m);
      if constexpr (decltype(loads)::value) {
        static_for<kDma>([&](auto qc) {
          constexpr int q = decltype(qc)::value;
          if constexpr ((2 * q + 1) * KS * kStep / (2 * kDma) == slot) load(kt + D, q);
        });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  floatx16 sum[SLICED ? TM : 1][SLICED ? TN : 1];  // of the finished slices
  if constexpr (SLICED) ZeroStart::start<TM, TN>(sum, 0, 0, 0);
  if (n_kt > 0) {
    constexpr auto kYes = std::true_type{};
    constexpr auto kNo = std::false_type{};
    if (D < n_kt) stage(0, kYes, kYes, kNo);
    else stage(0, kYes, kNo, kNo);
    int slice = 1, slice_at = SLICED && slices > 1 ? n_kt / slices : n_kt;
    int kt = 1;
    for (; kt + D < n_kt; ++kt) {
      stage(kt, kNo, kYes, kNo);
      if constexpr (SLICED) {
        if (kt != slice_at) continue;
        // the slice's last stage, kt - 1, is multiplied; the next stage's slots start a new one
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) sum[i][j][r] += acc[i][j][r];
        ++slice;
        slice_at = slice < slices ? slice * n_kt / slices : n_kt;
        ++kt;
        stage(kt, kNo, kYes, kYes);
      }
    }
    for (; kt < n_kt; ++kt) stage(kt, kNo, kNo, kNo);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int g = 0; g < NM; ++g) mfma(ks, g, kNo);
  }
  if constexpr (SLICED) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] += sum[i][j][r];
  }
  epi.template apply<TM, TN>(acc, m0 + wm * WTM, n0 + wn * WTN, lane, lds);
}

}  // namespace gemm
}  // namespace cm
