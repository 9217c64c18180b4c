// How high the row tiles of caifx_gemm_tall.hpp may be (host only).
#pragma once

#include <cmath>
#include <cstdint>

namespace caifx {

constexpr int kTallRows = 256, kTallCols = 256;      // of a tile at most

struct TallPlan {
  int height;      // a multiple of 32
  double us;       // estimate of the launch without its ends
};

// A launch lasts as many tiles one after the other as its fullest compute unit gets, so few tiles are made low and many high, and one
// tile more than there are compute units costs a round.  Of equal heights the highest: a segment longer than expected is no tile more.

// One weight: nb blocks of 16 rows take 3 + 0.33 nb us and 0.47 + 0.06 nb per step (the dequantisation, two meetings and the way of the
// requests; then the products, 16 rows 0.055).  Rows that fill the tiles to the last count half a tile more (1792 rows, 8832 x
// 2304, 245 full tiles 76 us, 72 with a copy of the weight).
inline TallPlan plan_tall_one(int64_t M, int64_t C, int64_t R)
{
  const double rows = static_cast<double>(M), steps = static_cast<double>(R) / 64, cols = static_cast<double>((C + kTallCols - 1) / kTallCols);
  TallPlan best{kTallRows, 0.0};
  for (int h = 64; h <= kTallRows; h += 32) {
    const double n = M > 8 * h ? rows / h + 0.5 : std::ceil(rows / h) + (M % h == 0 ? 0.5 : 0.0);
    const double whole = rows / std::floor(n + 0.1);
    double nb = 2.0 * std::ceil((whole < h ? whole : h) / 32.0);
    nb = nb < 4.0 ? 4.0 : nb;
    const double rounds = cols * n / 256.0;
    const double us = (rounds < 1.0 ? 1.0 : rounds < 4.0 ? std::ceil(rounds - 0.02) : rounds + 0.5) * (3.0 + 0.33 * nb + steps * (0.47 + 0.06 * nb));
    if (h == 64 || us <= best.us) best = TallPlan{h, us};
  }
  return best;
}

// Expert segments: 4 + 0.45 nb us and 0.51 + 0.04 nb per step (of calls replayed with the segments known: within 6 to 7 %).
//
// Their lengths are on the device, so the number of tiles is not known here.  The cost is an expectation, two thirds over uniformly drawn
// ids (lengths spread by the square root of their mean), one third over experts drawn 0.25 to 1.75 times as often as the mean.  The rows
// are all there are, so the number is spread by what the segments' last tiles lack alone.
//
// Over 1543 launches (2 to 64 experts, 17 to 2500 rows each, 256 to 2176 columns and reductions, a third of them drawn unevenly, both
// directions) the height chosen is 0.7 % off the best of 64, 96 .. 256 in the mean, and the launch 1.21 times as fast as on the kernels
// this one took the calls from; eight are slower, by 3 to 10 %, most of them reductions of 256 (of 2766 others eleven, by 2 to 16 %).  With the number of tiles taken at its
// mean: 2.2 %, 1.20, and 32 slower, down to 0.65, where a second round was not foreseen (5472 rows, 16 experts, C = 896, R = 1280
// 41.5 us, here 27.2, those kernels 26.7).
inline TallPlan plan_tall(int64_t M, int experts, int64_t C, int64_t R)
{
  if (experts == 1) return plan_tall_one(M, C, R);
  static const double kDrawn[8] = {-1.53, -0.89, -0.49, -0.16, 0.16, 0.49, 0.89, 1.53};      // eighths of a normal spread
  static const double kUneven[8] = {0.34, 0.53, 0.72, 0.91, 1.09, 1.28, 1.47, 1.66};         // eighths of 0.25 .. 1.75
  const double rows = static_cast<double>(M), E = experts, mean = rows / E, steps = static_cast<double>(R) / 64;
  const double cols = static_cast<double>((C + kTallCols - 1) / kTallCols);
  const double spread = std::sqrt((mean > 1.0 ? mean : 1.0) * (1.0 - 1.0 / E));
  const auto tile_us = [&](double nb) { return 4.0 + 0.45 * nb + steps * (0.51 + 0.04 * nb); };
  TallPlan best{kTallRows, 0.0};
  for (int h = 64; h <= kTallRows; h += 32) {
    double us = 0.0;
    for (int uneven = 0; uneven < 2; ++uneven) {
      // of a segment: tiles, blocks of 16 rows in all of them and in the highest, the part of a tile that the last one lacks
      double count = 0.0, blocks = 0.0, highest = 4.0, lack = 0.0, lack2 = 0.0;
      for (int i = 0; i < 8; ++i) {
        const double length = uneven ? mean * kUneven[i] : mean + kDrawn[i] * spread;
        if (length <= 0.0) continue;
        const double n = std::ceil(length / h), rest = n - length / h;
        double nb = 2.0 * std::ceil(std::ceil(length / n) / 32.0);
        nb = nb < 4.0 ? 4.0 : nb;
        count += n;
        blocks += n * nb;
        if (nb > highest) highest = nb;
        lack += rest / 8;
        lack2 += rest * rest / 8;
      }
      double variance = lack2 - lack * lack;
      if ((uneven ? 1.32 * mean : 3.06 * spread) > 3.0 * h) {      // eight lengths of so many tiles say nothing about the last one
        lack = 0.5;
        variance = 1.0 / 12;
      }
      const double usual = count > 0.0 ? tile_us(blocks / count) : 0.0, tiles = rows / h + E * lack, most = rows / h + E * (1.0 - 1.0 / h);
      const double sigma = variance > 0.0 ? std::sqrt(E * variance) : 0.0;
      double launch = (tiles * cols / 256.0 + 0.5) * usual;      // many rounds even out
      if (tiles * cols <= 4 * 256.0) {
        launch = tile_us(highest);
        for (int k = 1; k <= 4; ++k) {      // and a tile for each round that is begun, by how likely it is
          const double fit = std::floor(256.0 * k / cols);
          if (fit + 1.0 > most) break;
          launch += usual * 0.5 * std::erfc((fit + 0.5 - tiles) / (sigma * 1.41421356 + 1e-6));
        }
      }
      us += (uneven ? 1.0 / 3 : 2.0 / 3) * launch;
    }
    if (h == 64 || us <= best.us) best = TallPlan{h, us};
  }
  return best;
}

}  // namespace caifx
