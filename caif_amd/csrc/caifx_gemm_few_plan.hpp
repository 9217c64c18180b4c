// Which calls caifx_gemm_few.hip takes, and how it cuts them (host only).
#pragma once

#include <cstdint>

namespace caifx {

enum { FK_INT4 = 0, FK_INT8 = 1, FK_INT8_ONE = 2 };      // int8 with a scale vector; with one scale or none

constexpr int kFewCols = 64, kFewWaves = 8;      // of a workgroup

struct FewPlan {
  int row_tiles, col_tiles, tile_rows;      // of tile_rows rows (a multiple of 16) x kFewCols columns
  int parts, part_units;                    // workgroups that share a tile's reduction, units of each; 0: another kernel's call
};

// Whole rounds: with more tiles than compute units a second round costs as much as the first (int8 per channel, N = 11008, K = 4096:
// M = 100, 172 tiles, 39.4 us here and 45.3 tiled; M = 128, 344 of 64 rows, 56.0 and 46.0).  Among the row tiles that fit, the height
// whose estimate is the least: low ones repeat the dequantisation, which beats few parts of a long reduction (M = 256, N = K = 2048,
// int8: 32 rows 13.3 us, 64 16.2, 112 18.3) but not many parts (M = 33, N = 5952, K = 3072, int4: 48 rows 12.6 us, 32 14.2).
//
// int4 runs the tiled kernel faster, four steps of codes to a line: here where a workgroup's share is short (units x 16-row blocks up
// to 64; N = K = 2048, M = 256 16.6 tiled, 12.4 here; above it N = K = 4096, M = 200 25.4 and 27.7, N = 14336, K = 4096, M = 80
// 29.8 and 31.2) and up to 64 rows, which leave half of a 128-row tile idle (N = 14336, K = 4096: M = 64 29.5 and 27.9, M = 33
// 29.0 and 21.1).  int8 with a scale vector and more than 256 rows: up to twice that share (N = K = 2048, M = 512 23.1 and 18.3; above it
// N = 2048, K = 4096, M = 320 21.8 and 23.8).  With one scale the tiled kernel takes twice as long.
//
// At the end of that share with tiles of 32 rows (int4 K = 4096, int8 from K = 3648 on) the two are within 5 % on repeated passes, and a first
// one pays 2 to 3 us for the instructions, 11 KB of them (us, tiled / here, repeated | other code run in between: int4 N = K = 4096, M = 100 19.6 /
// 18.8 | 19.5 / 21.8; N = 2752, K = 4096, M = 97 17.6 / 19.7 | 17.6 / 21.1; int8 N = 1024, K = 3968, M = 444 20.3 / 21.3 | 21.5 / 22.8).
// Not where the tiled kernel's 128 x 128 tiles, 33 to 36 of them, come in seven parts, which it takes longer for (int4 N = 2240,
// K = 4096, M = 192 24.5 / 20.3 | 24.3 / 21.6; int8 N = 704, K = 4096, M = 698 25.8 / 21.5 | 27.2 / 22.4).
//
// Reductions below 512 stay with the kernel that adds up in the order of the grouped ones; they would leave waves without a unit (as int4
// below 1024 does: N = 4416, M = 330, K = 512 10.4 / 10.0).
inline FewPlan plan_few(int64_t M, int64_t N, int64_t K, int kind)
{
  FewPlan g{};
  const int unit = kind == FK_INT4 ? 128 : 64;
  if (M < 17 || K < 512 || K % unit != 0 || N % 8 != 0 || N * K >= (int64_t{1} << 32) || M * K >= (int64_t{1} << 31)) return g;
  const int64_t col_tiles = (N + kFewCols - 1) / kFewCols, units = K / unit;
  int64_t best = 0;
  for (int blocks = 2; blocks <= 7; ++blocks) {
    const int64_t row_tiles = (M + 16 * blocks - 1) / (16 * blocks), tiles = row_tiles * col_tiles;
    if (tiles > 256) continue;
    const int64_t tile_rows = ((M + row_tiles - 1) / row_tiles + 15) / 16 * 16, nb = tile_rows / 16;
    int64_t parts = 256 / tiles;
    if (parts > units / kFewWaves) parts = units / kFewWaves;
    if (parts > 8) parts = 8;
    if (parts < 1) parts = 1;
    const int64_t per = (units + parts - 1) / parts;
    // beginning and end of a workgroup, and its share of the reduction, in units of about 0.15 us
    const int64_t cost = 8 * (4 + 2 * nb) + per * (1 + nb);
    if (best != 0 && cost >= best) continue;
    best = cost;
    g.row_tiles = static_cast<int>(row_tiles);
    g.col_tiles = static_cast<int>(col_tiles);
    g.tile_rows = static_cast<int>(tile_rows);
    g.parts = static_cast<int>((units + per - 1) / per);
    g.part_units = static_cast<int>(per);
  }
  if (best == 0) return g;
  const int64_t share = static_cast<int64_t>(g.part_units) * (g.tile_rows / 16);
  const int64_t most = kind == FK_INT4 ? 64 : 128, tiled = (M + 127) / 128 * ((N + 127) / 128);
  const bool always = kind == FK_INT8_ONE || M <= (kind == FK_INT4 ? 64 : 256);
  const bool at_the_end = g.tile_rows == 32 && share > (kind == FK_INT4 ? 62 : 112) && 256 / tiled != 7;
  if (!always && (share > most || at_the_end)) g = FewPlan{};
  return g;
}

}  // namespace caifx
