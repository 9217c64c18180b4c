// How fp32-compute calls over int8 and int4 codes are cut into workgroups, and which of the two kernels takes them: the products of bf16
// pieces (caifx_gemm_pieces.hip) or the fp32 instruction's split tile (caifx_gemm_f32.hip).  Host arithmetic alone, so that it can be
// checked without a GPU.
#pragma once
#include "caifx.h"

#include <cstddef>
#include <cstdint>

namespace caifx {

constexpr int kPK = 64;                   // reduction extent of a step
constexpr int kPN = 64;                   // columns of a tile

// What a call of the pieces costs in us, fitted to 3005 calls and 27 thousand plans (forward and gradient, 64 to 14336 columns, reductions of
// 64 to 4096, 16 to 4096 rows, a quarter of them of random sizes; 6 % rms): a step of a workgroup alone on its compute unit, and what
// every further one there adds to it, for up to four, three or two of them by the tile's size; beyond that a step of a full chip and
// the stores of its tiles, in proportion, or in rounds of which the last overlaps a little where only two share a unit; the launch
// that adds the parts, and their sums.
struct PiecesTile {
  int bm, slots;
  double alone, more, full;
};
constexpr PiecesTile kTiles4[3] = {{32, 4, 1.035, 0.32, 2.07}, {64, 3, 1.63, 0.32, 2.60}, {128, 2, 2.78, 0.29, 2.97}};
constexpr PiecesTile kTiles8[3] = {{32, 4, 1.33, 0.42, 2.68}, {64, 3, 1.82, 0.46, 3.09}, {128, 2, 2.90, 0.46, 3.34}};

inline double pieces_us(const PiecesTile &tile, int64_t groups, int per)
{
  const int64_t residents = (groups + 255) >> 8;
  const double steps = static_cast<double>(per), full = steps * tile.full + 0.042 * tile.bm;
  const auto some = [&](int64_t n) { return steps * (tile.alone + tile.more * static_cast<double>(n - 1)); };
  if (residents <= tile.slots) return 4.9 + some(residents);
  if (tile.slots == 2) return 4.9 + full * static_cast<double>(residents >> 1) + ((residents & 1) != 0 ? 0.85 * some(1) : 0.0);
  return 4.9 + full * static_cast<double>(residents) * (tile.slots == 3 ? 1.0 / 3.0 : 0.25);
}
inline double pieces_sums_us(int parts, size_t bytes) { return parts > 1 ? 1.0 + 0.086 * parts + 0.59e-6 * static_cast<double>(bytes) : 0.0; }

// Rows of a tile and workgroups that share its reduction: the plan of the least cost.  It is within 0.6 % of the fastest in the mean, 19 %
// at the worst (fixed: 32 rows up to M = 32, 64 up to 64, 128 beyond, as many parts as fill the chip: M = 200, N = 3456, K = 3712 70 us
// against 52; M = 100, N = K = 512 19 against 9.5).  The parts' sums stay within the library's own buffer for callers without a workspace.
struct PiecesPlan {
  int bm, parts, part_steps;
  size_t bytes;
  double us;
  bool limited;          // with more room another plan would be faster
};
// (made for every call, and for every question how much workspace one takes: no division but those of the steps)
inline PiecesPlan plan_pieces(int64_t M, int64_t C, int64_t R, bool int4, size_t room)
{
  constexpr int kMostParts = 12;
  constexpr int64_t kMostRowTiles = 65535;        // gridDim.y
  const int steps = static_cast<int>(R / kPK);
  const size_t part_bytes = static_cast<size_t>(M) * static_cast<size_t>(C) * sizeof(float);
  PiecesPlan best{};
  double least = 0.0;
  for (int k = 1; k <= kMostParts; ++k) {
    const int per = (steps + k - 1) / k, parts = (steps + per - 1) / per;
    if (k > 1 && per < 2) break;
    if (parts < k) continue;
    const size_t bytes = parts > 1 ? static_cast<size_t>(parts) * part_bytes : 0;
    if (bytes > CAIFX_STATIC_SCRATCH_BYTES) break;
    const double sums = pieces_sums_us(parts, bytes);
    for (int t = 0; t < 3; ++t) {
      const PiecesTile &tile = (int4 ? kTiles4 : kTiles8)[t];
      if (t > 0 && M <= tile.bm / 2) break;
      const int64_t row_tiles = (M + tile.bm - 1) >> (5 + t);
      if (row_tiles > kMostRowTiles) continue;
      const double us = sums + pieces_us(tile, row_tiles * ((C + kPN - 1) / kPN) * parts, per);
      if (least == 0.0 || us < least) least = us;
      if (bytes <= room && (best.bm == 0 || us < best.us)) best = PiecesPlan{tile.bm, parts, per, bytes, us, false};
    }
  }
  best.limited = least < best.us;
  return best;
}

// The fp32 instruction's tile of 32 x 32 whose waves share 128-deep steps, for up to kSplitTileRows rows and reductions that are a multiple
// of 128.  There are C / 32 such tiles per 32 rows: a chain of R / 128 dependent steps on half of the chip at 32 rows and C = 4096.
// With a workspace from the caller up to 4 workgroups share a tile's reduction (at least 8 steps each, about one workgroup per
// compute unit in total) and a second launch adds their partial tiles in a fixed order.
constexpr int kSplitTileRows = 128;   // M = 64: 256 workgroups instead of 64
struct SplitTilePlan {
  int parts, part_steps;
  size_t bytes;
};
inline SplitTilePlan plan_split_tile(int64_t M, int64_t C, int64_t R)
{
  SplitTilePlan p{1, 0, 0};
  if (M > kSplitTileRows || R % 128 != 0) return p;
  const int64_t tiles = ((C + 31) / 32) * ((M + 31) / 32);
  if (tiles > 128) return p;
  const int64_t steps = R / 128;
  int64_t k = 256 / tiles;
  if (k > 4) k = 4;
  if (k > steps / 8) k = steps / 8;
  if (k < 2) return p;
  const int64_t per = (steps + k - 1) / k;
  k = (steps + per - 1) / per;
  if (k < 2) return p;
  p.parts = static_cast<int>(k);
  p.part_steps = static_cast<int>(per);
  p.bytes = static_cast<size_t>(k) * static_cast<size_t>(M) * static_cast<size_t>(C) * sizeof(float);
  return p;
}
// us of a call, fitted to 760 of them (4.5 % rms)
inline double split_tile_us(int64_t M, int64_t C, int64_t R, bool int4, size_t room)
{
  const SplitTilePlan p = plan_split_tile(M, C, R);
  const bool shared = p.parts > 1 && p.bytes <= room;
  const int64_t parts = shared ? p.parts : 1;
  const double steps = static_cast<double>(shared ? p.part_steps : R / 128);
  const double more = static_cast<double>((((C + 31) / 32) * ((M + 31) / 32) * parts + 255) / 256 - 1);
  const double us = 3.6 + steps * (int4 ? 1.19 + 0.76 * more : 1.28 + 0.81 * more) + 0.4 * more;
  return shared ? us + 1.6 + 1.6e-6 * static_cast<double>(p.bytes) : us;
}

// Whether the split tile takes a call that the pieces could take too, by `plan` in that room: where it is estimated to be faster, for short reductions (M = 100, R = 256, int8
// 6.8 us against 9.1) and, whatever their length, where the room keeps the pieces from sharing a reduction as they would (without a
// workspace M = 64, C = 1024, R = 4096 44.5 us against 92.5, R = 2048 24.4 against 48.7; M = 33, int4, 43 against 76).  Elsewhere the
// two are within 20 % of each other, and the pieces have the smaller error.
inline bool split_tile_first(int64_t M, int64_t C, int64_t R, bool int4, size_t room, const PiecesPlan &plan)
{
  if (M > kSplitTileRows || R % 128 != 0) return false;
  if (R > 640 && !plan.limited) return false;
  return split_tile_us(M, C, R, int4, room) < plan.us;
}

}  // namespace caifx
