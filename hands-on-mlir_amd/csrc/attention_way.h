// Which of its kernels the attention takes.
#pragma once

#include <stdint.h>

namespace hom {

// All with the same arithmetic per 32 query rows (us, batch : seq : heads, lengths uniform
// in [seq / 4, seq] unless said otherwise):
//  - kPrefetch: 64 rows per workgroup with the keys split over two wavefronts per
//    32 rows, K and V of the first 128 keys requested before anything else is
//    known.  Head size 64.  The fastest while that is all of them and every workgroup has a CU of
//    its own (8:128:12 4.2, against 5.0 - 5.3; 26:105:8, where it has not, 6.4 against 4.8 by
//    kDma, 11:119:16 6.45 against 4.9).
//  - kWide: 128 rows, chunks of 128 keys through registers; head size 64 for so
//    many short sequences that the workgroups of a CU cover each other
//    (64:70:12 7.7 against 7.9, but 32:128:16 8.3 against 7.95), and 256, whose chunks by
//    DMA would leave too few registers (8:384:16 42 against 47).
//  - kDma: 128 rows, chunks of 64 keys straight into LDS while the one before is
//    worked on (head size 64, 32:512:16 41.8 -> 40.6, 1:64:12 4.0 -> 3.6; 128,
//    32:512:16 66.9 -> 60.9).  Head size 192: 8 wavefronts, two per 32 rows, which
//    then fit two to a SIMD (32:512:12 117 -> 97).
//  - kDmaSplit: the same with 64 rows and two wavefronts per 32 rows.
enum class AttentionWay { kPrefetch, kWide, kDma, kDmaSplit };

// Head sizes 64 and 128 beyond 128 tokens: split keys (kDmaSplit) or whole rows (kDma).
// Split keys give twice the workgroups of half the work, which spread better over the CUs and
// leave less idle where a sequence ends inside a tile; but all K and V are read twice as often.
// Both timed in turn at 200 shapes of each head size (130 to 770 tokens, 0.4 to 2.2 tiles of 128 rows a
// CU), eight draws of lengths and full ones.  Whole rows over split keys, by tiles a CU:
//  - to 0.6: 1.08 to 1.29.  Up to 192 tokens also to 1.1 workgroups of 64 rows a CU, 1.08 to 1.15.
//  - to 1: of 128 0.87 to 1.08 (full lengths 0.84 to 0.96); of 64 0.94 to 1.0 up to 256 tokens, 0.99 to 1.13 beyond
//    (full 0.87 to 1.03).
//  - to 1.4, where a second tile would be all that some CUs do: 1.0 to 1.2 (full 0.74 to 1.24), but 0.83 to 0.87 from
//    193 to 256 tokens, two full tiles.
//  - to 1.8: 1.0 to 1.15 where the last tile is at most half full (full lengths 0.77 to 0.96), 0.8 to 1.03 where
//    it is more (0.71 to 1.01).
//  - above: 0.76 to 0.95.
// In fragment order split keys gain less (kPipe), and a request is timed, of six layers of BERT-base and -large, six
// draws of lengths and full ones: to 1 tile 0.987 to 1.022 (5 x 150 of large 1.015, 6 x 180 1.022, 5 x 450 of base 0.988; full
// 0.97 to 1.02); from 193 to 256 tokens to 1.4 0.98 to 0.994; to 1.8 0.987 to 1.022 with the last tile at most half full,
// else 0.975 to 1.001; and with up to 160 tokens 0.998 to 1.016 to 2 tiles a CU.
inline bool attentionSplitsKeys(int64_t pairs, int64_t seq, int64_t headDim, bool packed, int cus) {
  const int64_t tiles = pairs * ((seq + 127) / 128), tiles64 = pairs * ((seq + 63) / 64);
  const bool halfTile = (seq - 1) % 128 < 64; // the last one
  if (10 * tiles <= 6 * cus || (seq <= 192 && 10 * tiles64 <= 11 * cus))
    return true;
  if (tiles <= cus)
    return packed || (headDim == 64 && seq > 256);
  if (seq > 192 && seq <= 256)
    return false;
  if (10 * tiles <= 14 * cus)
    return true;
  return halfTile && 10 * tiles < (packed && seq <= 160 ? 20 : 18) * cus;
}

inline AttentionWay attentionWay(int64_t pairs, int64_t seq, int64_t headDim, bool packed, int cus) {
  const int64_t tiles = pairs * ((seq + 127) / 128);
  const bool few = tiles <= cus / 2;
  if (headDim == 64 && seq <= 128)
    return seq <= 64           ? AttentionWay::kDma
           : few               ? AttentionWay::kPrefetch
           : tiles <= 2 * cus ? AttentionWay::kDma
                               : AttentionWay::kWide;
  if (headDim == 128 && seq <= 128)
    return seq > 64 && tiles < cus / 2 ? AttentionWay::kDmaSplit : AttentionWay::kDma;
  if (headDim <= 128)
    return attentionSplitsKeys(pairs, seq, headDim, packed, cus) ? AttentionWay::kDmaSplit : AttentionWay::kDma;
  // (4:185:16 of 256 11.9 against 14.5, 8:200:8 of 192 10.1 against 11.8)
  return few ? AttentionWay::kDmaSplit : headDim == 192 ? AttentionWay::kDma : AttentionWay::kWide;
}

// Order of the workgroups of split keys at head sizes from 128 on: the query tiles of a pair
// (batch entry, head) back to back, or (true) all first tiles, then all second ones, .., so that
// those of nothing but padding come last.  That pays
//  - up to one and a half workgroups a CU, where the last ones find a CU free: of 128, pairs a multiple of 8, eight
//    draws of lengths uniform in [seq / 4, seq], 0.86 to 1.05 of the time with 257 to 320 workgroups (mean of
//    11 shapes 0.94), 0.91 to 1.07 to 384 (13, 0.98), beyond means of 1.01 to 1.05 (118; 8:620:8 17.6 -> 20.5 us);
//  - where the pairs are no multiple of 8: back to back a pair's tiles go to the XCDs in turn, and those past the
//    end of its sequence to the same few of them (22 shapes 0.70 to 1.015; 1:700:12 10.0 -> 9.1 us, of 256 20.0 ->
//    19.5, of 192 14.7 -> 14.3).
constexpr bool attentionTilesOutside(int pairs, int tiles) { return pairs % 8 != 0 || pairs * tiles <= 384; }

// Whether the chunked kernels issue the next chunk's scores between this chunk's exponentials (see
// kPipe in attention.hip for those that never do).  A first and last chunk have nothing to overlap, so it depends on
// the length.  Time with it over without, six draws of lengths uniform in [seq / 4, seq]:
//  - 64, split keys: to 192 tokens 0.99 to 1.05 (9:129:16 5.3 -> 5.6 us), 193 to 256 0.97 to 0.99, beyond 0.95 to
//    1.03 (mean 0.99; 2:520:12 7.0 -> 6.65).
//  - 128, whole rows: 1.0 to 1.01 to 64 tokens, beyond 0.90 to 1.01 (1:720:16 13.6 -> 12.25).  Split keys, which
//    are for more tokens than that anyway, 0.92 to 1.016 (1:720:16 10.5 -> 9.7).
//  - 256, split keys: 1.03 to 1.05 to 65 tokens, 0.986 to 1.017 to 192, beyond 0.97 to 1.0 (3:620:8 23.8 -> 23.1).
constexpr bool attentionOverlapsScores(int64_t headDim, int64_t seq) {
  return headDim == 128 ? seq > 64 : seq > 192;
}

} // namespace hom
