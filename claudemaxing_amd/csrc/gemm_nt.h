// Operand layouts of the fp16 "NT" GEMMs on the gfx950 matrix cores (C[m][n] = sum_k A[m][k]
// B[n][k], both operands K-contiguous), the MFMA register types, and the workgroup -> tile map.
//   RowMajor  element (r, k) at p[r * ld + k];
//   Tiled32   32-row x 64-column blocks of 8-column chunks (below);
//   KMajor    the operand stored transposed, [K][N] with N contiguous (below).
// The main loop that consumes them is in gemm_lds.h. Of a tile that reaches past the operand's last
// row, the rows outside are read from its last valid row: they feed only outputs that are never
// stored. Columns past k_len must come as zeros (k_inside says whether a stage has any).
#pragma once

#include "common.h"

namespace cm {
namespace gemm {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kBK = 64;              // K elements per stage
constexpr int kRowChunks = kBK / 8;  // 16-byte chunks per tile row

struct RowMajor {
  static constexpr bool kChunkMajor = false;  // LDS tile layout (gemm_lds.h)
  static constexpr bool kKMajor = false;
  static constexpr bool kSegmented = false;
  const _Float16* p;
  int64_t ld;
  int rows;   // valid rows
  int k_len;  // valid columns
  __device__ __forceinline__ const _Float16* at(int r, int k) const {
    return p + static_cast<int64_t>(r) * ld + k;
  }
  __device__ __forceinline__ bool k_inside(int k0) const { return k0 + kBK <= k_len; }
  __device__ __forceinline__ bool col_ok(int k) const { return k < k_len; }
  // the row of a tile at r0 that stands in for its row r (valid rows for themselves)
  __device__ __forceinline__ int clamp_row(int r0, int r) const { return min(r, rows - 1 - r0); }
  // bytes from element (r0, k0) to (r0 + r, k0 + k) of a tile (k < 64)
  __device__ __forceinline__ uint32_t tile_offset(int r, int k) const {
    return static_cast<uint32_t>((static_cast<int64_t>(r) * ld + k) * 2);
  }
};

// 4 KiB blocks of 32 rows x 64 columns, 8-column chunks inside: element (r, k) at
// p[(((k / 64) * row_blocks + r / 32) * 8 + (k % 64) / 8) * 256 + (r % 32) * 8 + k % 8], with
// row_blocks = ceil(rows / 32). One 16-byte chunk is 8 consecutive columns of a row, and the
// chunks of 32 consecutive rows at one 8-column position are one 512-byte span, so a producer
// whose lanes hold consecutive rows (the LM head's logits epilogue: one token per lane) writes
// whole spans straight from registers, while a GEMM stage's 8-row x 64-column slices stay inside
// one block. The columns up to the end of the last 64-column panel must hold finite
// values, and the rows up to the end of the last tile must exist (their values are not used).
struct Tiled32 {
  static constexpr bool kChunkMajor = true;
  static constexpr int kChunkBytes = 512;  // between a row's neighbouring 8-column chunks
  static constexpr bool kKMajor = false;
  static constexpr bool kSegmented = false;
  const _Float16* p;
  int rows;        // valid rows
  int k_len;       // columns
  int row_blocks;  // ceil(rows / 32)
  static __host__ __device__ __forceinline__ int64_t index(int64_t r, int64_t k, int row_blocks) {
    return (((k / 64) * row_blocks + r / 32) * 8 + (k % 64) / 8) * 256 + (r % 32) * 8 + k % 8;
  }
  __device__ __forceinline__ const _Float16* at(int r, int k) const {
    return p + index(r, k, row_blocks);
  }
  __device__ __forceinline__ bool k_inside(int k0) const { return k0 < k_len; }
  __device__ __forceinline__ bool col_ok(int k) const { return (k / kBK) * kBK < k_len; }
  __device__ __forceinline__ int clamp_row(int, int r) const { return r; }
  // bytes from element (r0, k0) to (r0 + r, k0 + k) of a tile (r0 a multiple of 32, k0 of 64,
  // k < 64 a multiple of 8)
  __device__ __forceinline__ uint32_t tile_offset(int r, int k) const {
    return static_cast<uint32_t>(((r / 32) * 8 + k / 8) * kChunkBytes + (r % 32) * 16);
  }
};

// Up to three row-major arrays side by side along k, each with its own base and row stride: segment s
// holds columns first[s] .. first[s + 1] - 1 (whole 64-column stages). The gradients of several
// outputs of one input, contracted together.
struct SegRows {
  static constexpr bool kChunkMajor = false;
  static constexpr bool kKMajor = false;
  static constexpr bool kSegmented = true;
  const _Float16* p[3];
  int64_t ld[3];
  int first[3];  // an unused segment's is past k_len
  int rows;
  int k_len;
  // the address of (r, k) and the row stride there; k uniform over the wavefront
  __device__ __forceinline__ const _Float16* at(int r, int k, int64_t& stride) const {
    const bool s1 = k >= first[1], s2 = k >= first[2];
    stride = s2 ? ld[2] : s1 ? ld[1] : ld[0];
    const _Float16* base = s2 ? p[2] : s1 ? p[1] : p[0];
    return base + static_cast<int64_t>(r) * stride + (k - (s2 ? first[2] : s1 ? first[1] : 0));
  }
  __device__ __forceinline__ bool k_inside(int) const { return true; }
};

// An NT operand stored transposed, [K][N] with N contiguous: element (row n, column k) of the
// operand at p[k * ld + n]. The LM head reads its weight W [V][H] this way as the gradient GEMM's
// B operand (rows = hidden units, K = vocabulary), so that no transposed copy of W is needed.
// Its LDS tiles are k-major and its MFMA fragments are assembled by transposing LDS reads
// (gemm_lds.h, DmaTileK and frag_kmajor).
struct KMajor {
  static constexpr bool kChunkMajor = false;
  static constexpr bool kKMajor = true;
  static constexpr bool kSegmented = false;
  const _Float16* p;
  int64_t ld;  // elements between consecutive k
  int rows;    // valid n
  int k_len;   // valid k
  __device__ __forceinline__ const _Float16* at(int n, int k) const {
    return p + static_cast<int64_t>(k) * ld + n;
  }
  __device__ __forceinline__ bool k_inside(int k0) const { return k0 + kBK <= k_len; }
};

// Workgroup -> (tile_m, tile_n), tile_n fastest, for block `bid` of `count` blocks. With remap
// (count % 8 == 0), logical tile ids are laid out so that consecutive ones run on the same XCD
// (hardware dispatches workgroup ids round-robin over the 8 XCDs), so workgroups that share operand
// tiles share an L2.
__device__ __forceinline__ void tile_of(int bid, int count, int tiles_n, int remap, int& tm,
                                        int& tn) {
  if (remap) bid = (bid % 8) * (count / 8) + bid / 8;
  tm = bid / tiles_n;
  tn = bid % tiles_n;
}

// Split-K form of tile_of: `count` = tiles * slices blocks; each XCD gets a contiguous range of
// (slice, tile) ids, i.e. one K-slice and a block of tile rows.
__device__ __forceinline__ void tile_of_sliced(int bid, int count, int tiles, int tiles_n,
                                               int remap, int& tm, int& tn, int& slice) {
  if (remap) bid = (bid % 8) * (count / 8) + bid / 8;
  slice = bid / tiles;
  const int t = bid % tiles;
  tm = t / tiles_n;
  tn = t % tiles_n;
}

// The same over a 2-D grid (blockIdx.y = K-slice): the flattened (slice, tile) ids are laid out
// so that each XCD gets a contiguous range, i.e. one K-slice and a block of tile rows, whose
// operand tiles its L2 then shares. remap requires gridDim.x * gridDim.y % 8 == 0.
__device__ __forceinline__ void tile_of_block_2d(int tiles_n, int remap, int& tm, int& tn,
                                                 int& slice) {
  const int total = gridDim.x * gridDim.y;
  int bid = blockIdx.x + blockIdx.y * gridDim.x;
  if (remap) bid = (bid % 8) * (total / 8) + bid / 8;
  slice = bid / gridDim.x;
  const int t = bid % gridDim.x;
  tm = t / tiles_n;
  tn = t % tiles_n;
}

}  // namespace gemm
}  // namespace cm
