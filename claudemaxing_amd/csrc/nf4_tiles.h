// Host rule shared by the NF4-fused GEMM (nf4_gemm.hip) and the fp16 linear layers' input gradient
// (gemm_f16.hip): the tiles of the first and the slices in which both sum a contraction.
#pragma once

#include <cstdint>

namespace cm {

constexpr int kNf4CUs = 256;

struct Nf4Tiles {
  int bm, bn, split;  // tile of the weight's extent x tokens; slices of the contraction
  int64_t tiles;      // workgroups = tiles * split
};

// m tokens against an extent (a multiple of 128; ext256: of 256 throughout) of weight rows or columns,
// contracted over n_stages stages of 64. The contraction is split when the tiles alone leave CUs idle
// and the call has one output to sum into (can_split).
inline Nf4Tiles nf4_tiles(int64_t m, int extent, bool ext256, bool can_split, int n_stages) {
  Nf4Tiles p{};
  const int64_t tb = (m + 127) / 128;
  p.bn = 128;
  p.bm = ext256 ? 256 : 128;
  p.tiles = extent / p.bm * tb;
  if (p.bm == 256 && p.tiles < kNf4CUs / 2) {
    p.bm = 128;
    p.tiles = extent / p.bm * tb;
  }
  // 256-token tiles expand each weight element half as often; taken when they, split over the
  // contraction where that is allowed, still give most CUs a workgroup
  const int64_t tiles2 = extent / 128 * ((m + 255) / 256);
  int64_t sp2 = 1;
  if (can_split && tiles2 < kNf4CUs * 3 / 4) {
    sp2 = kNf4CUs / (tiles2 > 0 ? tiles2 : 1);
    if (sp2 > 8) sp2 = 8;
    if (sp2 > n_stages / 8) sp2 = n_stages / 8;
    if (sp2 < 1) sp2 = 1;
  }
  if (m >= 384 && tiles2 * sp2 >= kNf4CUs * 3 / 4) {
    p.bm = 128;
    p.bn = 256;
    p.tiles = tiles2;
  }
  p.split = 1;
  if (p.tiles < 3 * kNf4CUs / 4 && can_split) {
    int64_t sp = kNf4CUs / (p.tiles > 0 ? p.tiles : 1);
    if (sp > 8) sp = 8;
    if (sp > n_stages / 8) sp = n_stages / 8;
    if (sp > 1) p.split = static_cast<int>(sp);
  }
  return p;
}

}  // namespace cm
