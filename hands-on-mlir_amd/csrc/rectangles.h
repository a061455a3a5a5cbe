// Which tiles an XCD works on.
#pragma once

#include <algorithm>
#include <stdint.h>

namespace hom {

// What an XCD works on: chunkM x chunkN tiles, 2^xmLog XCDs along M.  Its L2 fetches
// the operands of the rectangle once, at about 0.7 TB/s per XCD from the last-level
// cache, which from some 500 rows on is what bounds the kernels without a slab loop (512 x 1024 x
// 4096 moved 42 MB so in 7.2 us); among the splits that leave the fullest CU the
// fewest tiles, the one that fetches least.
struct Rectangles {
  int xmLog, chunkM, chunkN;
  int64_t perCu;    // tiles of the fullest CU
  double fillBytes; // all XCDs
};
// Tiles of 16 mb x 16 nb.
inline Rectangles chooseRectangles(int64_t tilesM, int64_t tilesN, int mb, int nb, int64_t K,
                                   int cus) {
  const int64_t perXcd = std::max(1, cus / 8);
  Rectangles best{};
  for (int x = 0; x <= 3; x++) {
    const int64_t cm = (tilesM + (1 << x) - 1) >> x, cn = (tilesN + (8 >> x) - 1) / (8 >> x);
    const int64_t perCu = (cm * cn + perXcd - 1) / perXcd;
    const double fill = 8.0 * double(cm * mb + cn * nb) * 16 * double(K) * 2;
    if (x == 0 || perCu < best.perCu || (perCu == best.perCu && fill < best.fillBytes))
      best = {x, int(cm), int(cn), perCu, fill};
  }
  return best;
}

} // namespace hom
