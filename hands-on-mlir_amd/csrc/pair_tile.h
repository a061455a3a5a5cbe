// Which tiles the GEMMs of the layer-norm pair run on.
#pragma once

#include <stdint.h>

namespace hom {

// What beta C reads: nothing, rows that many tiles share, as much as D writes.
enum class PairSource { kNone, kRow, kMatrix };

// The square tile, 64, 128 or 256 on a side, whose rounds cost least; `second`: the
// GEMM of the normalised rows, otherwise the one with row statistics.  In units of a
// slab of a round of 128 x 128 tiles: rounds x (slab x slabs of K + round), for 256
// whole rounds, for the smaller ones, of which a CU holds several, half way between
// whole rounds and their number.  Fitted to all three tiles at 170 sizes (330 with a
// full matrix), M = 200 .. 16384, N = 64 .. 4300, K = 24 .. 4200, each GEMM with each
// source: 0.01 to 0.6 % over the fastest tile in the mean, 20 % at worst but for one
// (24 %: 10000 x 1304 x 256, second, full matrix, 29.2 / 26.2 / 32.4).  64 / 128 / 256, us:
// second, bias row 6872 x 2312 x 80 25.7 / 33.5 / 40.7; first, bias row 4936 x 1728 x 24
// 13.7 / 18.2 / 19.0; 128 / 256: first, no source 5535 x 2408 x 2960 121 / 86, bias row
// 13371 x 1072 x 1392 73 / 91, full matrix 8192 x 3072 x 1024 84 / 93.
inline int pairTileEdge(int64_t M, int64_t N, int64_t K, bool second, PairSource source, int cus) {
  struct Cost {
    double slab64, round64, round128, slab256, round256, early256;
  };
  static const Cost costs[2][3] = {{{0.45, 2.97, 11.1, 1.56, 41.9, 4.5},
                                    {0.52, 4.21, 20.4, 1.56, 68.4, 9.2},
                                    {0.48, 3.46, 11.5, 1.97, 57.4, 9.6}},
                                   {{0.46, 6.34, 23.7, 2.39, 59.3, 0.92},
                                    {0.34, 1.95, 8.87, 1.63, 33.9, 3.3},
                                    {0.38, 1.67, 6.61, 2.12, 37.6, 18.1}}};
  const Cost &c = costs[second ? 1 : 0][int(source)];
  auto tiles = [&](int64_t edge) {
    return ((M + edge - 1) / edge) * ((N + edge - 1) / edge);
  };
  auto whole = [&](int64_t t) { return double((t + cus - 1) / cus); };
  auto between = [&](int64_t t) { return 0.5 * (whole(t) + double(t) / cus); };
  const double slabs = double((K + 63) / 64);
  const double c64 = between(tiles(64)) * (c.slab64 * slabs + c.round64);
  const double c128 = between(tiles(128)) * (slabs + c.round128);
  const double c256 = whole(tiles(256)) * (c.slab256 * slabs + c.round256) - c.early256;
  return c256 < c64 && c256 < c128 ? 256 : c128 < c64 ? 128 : 64;
}

} // namespace hom
