// How the products of bf16 pieces (caifx_gemm_pieces.hip) are cut into workgroups: host arithmetic alone, so that it can be checked
// without a GPU.
#pragma once
#include "caifx.h"

#include <cstddef>
#include <cstdint>

namespace caifx {

constexpr int kPK = 64;                   // reduction extent of a step
constexpr int kPN = 64;                   // columns of a tile

// Rows of a tile and workgroups that share its reduction.  What a call costs in us, fitted to 20 weights from 512 x 512 to 8192 x
// 4096 and 33 to 600 rows (2132 plans, 4.5 % rms): a step of a workgroup alone on its compute unit and what every further one
// there adds to it, for up to four, three or two of them by the tile's size, in rounds that overlap; the launch that adds the
// parts and their bytes.  The plan it picks is within 4.5 % of the fastest in the mean (fixed: 32 rows up to M = 32, 64 up to 64, 128
// beyond, as many parts as fill the chip: M = 200, N = 3456, K = 3712 70 us against 52; M = 100, N = K = 512 19 against 9.5).
// The parts' sums stay within the library's own buffer for callers without a workspace.
struct PiecesPlan {
  int bm, parts, part_steps;
  size_t bytes;
};
inline PiecesPlan plan_pieces(int64_t M, int64_t C, int64_t R, bool int4, size_t room)
{
  struct Tile {
    int bm, slots;
    double alone, more;
  };
  static constexpr Tile tiles4[3] = {{32, 4, 1.03, 0.30}, {64, 3, 1.57, 0.23}, {128, 2, 2.60, 0.155}};
  static constexpr Tile tiles8[3] = {{32, 4, 1.20, 0.38}, {64, 3, 1.71, 0.36}, {128, 2, 2.63, 0.29}};
  constexpr int kMostParts = 12;
  constexpr int64_t kMostRowTiles = 65535;        // gridDim.y
  const int64_t steps = R / kPK;
  PiecesPlan best{};
  double least = 0.0;
  for (int t = 0; t < 3; ++t) {
    const Tile &tile = (int4 ? tiles4 : tiles8)[t];
    if (t > 0 && M <= tile.bm / 2) break;
    if ((M + tile.bm - 1) / tile.bm > kMostRowTiles) continue;
    for (int k = 1; k <= kMostParts; ++k) {
      const int64_t per = (steps + k - 1) / k, parts = (steps + per - 1) / per;
      if (k > 1 && (per < 2 || parts < k)) continue;
      const size_t bytes = parts > 1 ? static_cast<size_t>(parts) * static_cast<size_t>(M) * static_cast<size_t>(C) * sizeof(float) : 0;
      if (bytes > CAIFX_STATIC_SCRATCH_BYTES || bytes > room) continue;
      const int64_t groups = (M + tile.bm - 1) / tile.bm * ((C + kPN - 1) / kPN) * parts, round = 256 * tile.slots;
      const int64_t full = groups / round, rest = (groups - full * round + 255) / 256;
      const auto cost_of = [&](int64_t resident) { return static_cast<double>(per) * (tile.alone + tile.more * static_cast<double>(resident - 1)) - 5.0; };
      double cost = static_cast<double>(full) * cost_of(tile.slots) + (rest > 0 ? cost_of(rest) : 0.0);
      if (parts > 1) cost += 1.2 + 0.78e-6 * static_cast<double>(bytes);
      if (best.bm == 0 || cost < least) {
        best = PiecesPlan{tile.bm, static_cast<int>(parts), static_cast<int>(per), bytes};
        least = cost;
      }
    }
  }
  return best;
}

}  // namespace caifx
