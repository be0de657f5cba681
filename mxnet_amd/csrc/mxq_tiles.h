// Tile choice shared by the FC and the implicit-GEMM convolution launchers.
#ifndef MXQ_TILES_H_
#define MXQ_TILES_H_

#include <cstddef>

namespace mxq {

// What a caller may pin instead of leaving it to the choosers below: a tile configuration
// number of the launcher (0 = choose by shape), the number of work-groups that share one
// output tile along K (0 = choose, 1 = no split) and, for the short-K streaming kernel,
// its work-groups per CU (0 = choose).  The operator entry points pass the default; the
// test-only entry points pass what the test asks for.
struct GemmForce {
  int cfg = 0;
  int splits = 0;
  int stream_groups = 0;
};

// Caller-provided scratch for the split-K route (may be null: then nothing is split).
struct Workspace {
  void* ptr = nullptr;
  size_t bytes = 0;
};

enum class Tile {
  kL8,      // 256 x 256, 64-byte stages, 4-stage ring, pinned pipeline
  kW128x2,  // 256 x 128, 64-byte stages, 2-stage ring
  kW128K2,  // 256 x 128, 128-byte stages, 2-stage ring
  kM128x2,  // 128 x 128, 64-byte stages, 2-stage ring
  kM128K2,  // 128 x 128, 128-byte stages, 2-stage ring
  kS64x2,   // 64 x 64, 64-byte stages, 2-stage ring
  kS64K2,   // 64 x 64, 128-byte stages, 2-stage ring
  kS64K4,   // 64 x 64, 256-byte stages, 2-stage ring
  kR128K2,  // 128 x 64, 128-byte stages, 2-stage ring
  kQ128K2,  // 64 x 128, 128-byte stages, 2-stage ring
  kW192K2,  // 256 x 192, 128-byte stages, 2-stage ring
  kW64x2,   // 256 x 64, 64-byte stages, 2-stage ring
  kS64S4,   // 64 x 64 on eight waves, 256-byte stages, 4-stage ring
  kN32S3,   // 128 x 32 on eight waves, 256-byte stages, 3-stage ring
  kN32K2,   // 128 x 32, 128-byte stages, 2-stage ring
  kM128S3   // 128 x 128 on eight waves, 128-byte stages, 3-stage ring
};

// M x N outputs, reduction length K, `cus` compute units.  Distilled from sweeps over
// BERT-, ResNet-50- and square shapes (each rule names the measurement behind it):
//  * the 256 x 256 tile wins from about 0.56 tiles per CU on (4096 x 2304 x 768: 144 tiles,
//    15.9 us against 20.4 us for 128 x 128), if the output is wider than 128 columns and K
//    is long enough to amortise its prologue and epilogue;
//  * outputs of at most 64 columns take the 64 x 64 tile (nothing wider is useful);
//  * otherwise the 2-stage rings win: they need little LDS, several work-groups share a
//    CU, and one group's epilogue overlaps another's K loop.  A K step costs a barrier and
//    a round of DMA latency whatever its size, so from K = 512 on the stages are 128 bytes
//    deep (half as many steps: 10-20 % on every mid-size shape measured); below that the
//    deeper stage would mostly be padding or leave too few steps to overlap.  Small tiles with
//    little company on their CU take them from K = 256 on, and deeper ones (below);
//  * the 256 x 256 tile holds a CU alone, the 128 x 128 tile comes two to a CU and the 256 x 128
//    tile on 64-byte stages and the 64 x 128 tile three: which of them is ahead is a matter of
//    how many rounds the grid takes.  Once 128 x 128 tiles no longer fill the chip, 64 x 64 ones.
// `gather` says that the left operand is gathered pixel by pixel (convolution): the 64-row
// tile then issues half as many gathers per wave and measures a few per cent ahead of the
// 128-row one.
inline Tile choose_tile(long M, long N, long K, long cus, bool gather = false,
                        int* splits = nullptr) {
  if (splits != nullptr) *splits = 1;
  auto tiles = [&](long bm, long bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  // an output whose width is a multiple of 192 and that gives 256 x 192 tiles to (nearly)
  // every CU exactly once: 4096 x 768 -> 3072 is 256 such tiles against 192 of 256 x 256 on
  // 256 CUs (15.9 against 17.0 us), -> 2304 is 192 against 144 (15.4 against 16.1 us)
  if (!gather && K >= 512 && N % 192 == 0 && tiles(256, 192) <= cus &&
      4 * tiles(256, 192) >= 3 * cus && tiles(256, 192) > tiles(256, 256))
    return Tile::kW192K2;
  // A round of 256 x 256 tiles is as long as 1.6 of 128 x 128 tiles, two to a CU.  A few tiles into its
  // second round it is behind (us, 256 x 256 and 128 x 128: 4352 x 1024 -> 4352, 289 tiles, 38.2 / 32.2, 17000 x
  // 4096 -> 1024, 268, 110.8 / 91.4, 95000 x 1024 -> 256, 372, 57.6 / 50.6, but 5120 x 1024 -> 5120, 400, 39.4 /
  // 42.7), and so it is where ragged edges leave 128 x 128 tiles a single one (20000 x 1024 -> 300, 158 and
  // 471 tiles, 21.5 / 17.0; the convolutions 12544 x 512 -> 640 15.3 / 11.5, 19220 x 720 -> 300 18.2 / 14.0).
  // Gathered operands come closer: from 1.35 rounds of the smaller tiles in one of these on the larger are
  // ahead (38400 x 2592 -> 640, 1.46, 90.0 / 104.8, 36800 x 2592 -> 640, 1.41, 83.2 / 85.0, 41600 x 2592 -> 512, 1.27,
  // 81.6 / 83.7, 68992 x 864 -> 256, 1.05, 38.2 / 33.0).
  const long t256 = tiles(256, 256), t128 = tiles(128, 128);
  const long rounds256 = (t256 + cus - 1) / cus, rounds128 = (t128 + 2 * cus - 1) / (2 * cus);
  const bool larger = gather && rounds256 > 1 ? 10 * t128 >= 27 * cus * rounds256
                                              : 5 * rounds128 >= 8 * rounds256;
  if (K > 256 && N > 128 && 16 * t256 >= 9 * cus && larger) return Tile::kL8;
  // Up to one 64 x 64 tile a CU: eight waves share each of its stages, and three stages are under way.
  // With a wave a SIMD the tile's loads, reads of LDS and products were issued one behind the other
  // whatever the ring (us, four waves on two stages and eight on four: the convolutions 14400 x 25088 -> 32
  // 67.6 / 50.6, 850 x 5328 -> 922 20.7 / 16.3, 9216 x 3168 -> 51 12.3 / 10.8, 1125 x 1600 -> 330 9.3 / 9.0, 3971 x 784 -> 193
  // 9.3 / 9.4; plain operands 1024 x 4096 -> 1024 14.0 / 11.4, 100 x 7776 -> 6096 24.2 / 18.3, 78 x 1680 -> 7489 10.1 /
  // 9.7, 252 x 1376 -> 1562 7.4 / 7.6).  From the second tile a CU on two of the small work-groups are level
  // or ahead (7680 x 3200 -> 72, 386 tiles, 16.1 / 21.5).
  // Split-K: where such tiles leave CUs idle and the reduction is long, as many work-groups share one as
  // there are CUs for, each with 1536 of it and more (convolutions, unsplit on four waves, on eight, and split: 1152 x
  // 15680 -> 336 42.0 / 30.3 / 22.2 on two, 1681 x 13328 -> 98, 54 tiles, 36.4 / 26.7 / 16.6 on four, 121 x 34800 ->
  // 153, 6 tiles, 87.8 / 57.8 / 17.0 on 12; on 6, 8 and 16 19.5 / 17.7 / 18.3).  The price is a counter-clearing
  // launch and the partial sums' round trip through memory, about 3 us, and as much of the host's time, which is
  // what a caller of small layers waits for: below 8192 it gains no more than that, with any tile (2500 x 4704 ->
  // 114, 80 tiles, 15.1 / 13.3, 5396 x 8144 -> 58, 85, 19.2 / 17.2, 765 x 3728 -> 512, 96, 11.6 / 12.1; 128 x 128
  // tiles below).
  // Gathered operands of at most 32 columns take 128 x 32 tiles, half as many of which are padding, with
  // one of these a CU (20172 x 11760 -> 11, 158, 41.6 on four waves, 30.4 so, 28512 x 2000 -> 27 12.8 / 11.0) or
  // split over a long reduction (64 x 64 tiles split and these: 14400 x 25088 -> 32 50.6 / 36.4, 7744 x 14112 -> 11
  // 21.9 / 18.6, 15876 x 12400 -> 8 27.3 / 23.3; 14336 x 4000 -> 18 12.5 / 13.6).
  const long t64 = tiles(64, 64), t32 = tiles(128, 32);
  auto sharing = [&](long t, long slice) {
    if (splits == nullptr || t == 0) return 1L;  // (an output without elements has no tile)
    const long sp = cus / t < K / slice ? cus / t : K / slice;
    return sp > 12 ? 12L : sp < 1 ? 1L : sp;
  };
  auto shared = [&](long sp) {
    if (splits != nullptr) *splits = static_cast<int>(sp);
  };
  if (gather && N <= 32 && t32 <= cus &&
      (2 * t32 > cus ? K >= 1536 : K >= 8192 && splits != nullptr)) {
    shared(sharing(t32, 2048));
    return Tile::kN32S3;
  }
  // Tiles of 64 x 64 on 256-byte stages keep 64 KB under way on a CU, two of them at a time: up to two a
  // CU every step waits for memory, and bytes under way are what counts (the operands from HBM, us, 64-
  // and 128-byte stages and these: 1024 x 448 -> 1024 6.0 / 5.2 / 4.8, 2048 x 512 -> 1024 6.9 / 6.4 / 5.9,
  // 16384 x 1024 -> 64 12.1 / 11.0 / 9.9, 32768 x 512 -> 64 10.6 / 10.0 / 9.2, 12351 x 3872 -> 64 49.4 / - /
  // 25.1; 128 x 64 and these: 2048 x 512 -> 1024 7.1 / 5.9, 2048 x 2048 -> 1024 13.1 / 11.0).
  // From the third tile a CU on they wait for LDS (3000 x 512 -> 1024, 752 tiles, 7.8 / 6.8 / 8.7, 65536 x
  // 2048 -> 64, 1024 tiles, 56.7 / 53.0 / 51.3).
  const bool two_a_cu = t64 <= 2 * cus;
  // From half a 64 x 64 tile a CU to two of them and a long reduction: 128 x 128 tiles, which take in half
  // as much an output, split over the chip where that leaves few CUs idle (64 x 64 tiles, on eight waves up to one a
  // CU, and these: 1176 x 45472 -> 653, 209 and 60 on four, 87.1 / 64.6, 720 x 15680 -> 799, 156 and 42 on six,
  // 33.2 / 28.4, 475 x 29008 -> 1145, 144 and 36 on seven, 53.6 / 37.4, but 1568 x 12000 -> 493, 200 and 52 on four,
  // 27.4 / 28.8; with a second of the former on a CU, on four waves, 9408 x 11600 -> 71, 294 and 74 on three, 39.8 /
  // 30.9, 925 x 11712 -> 1712, 405 and 112 on two, 39.9 / 34.7).  90 drawn FC layers and 50 convolutions of that are
  // 1.2 times as fast on three and more from 8192 on, 1.04 below, some of them behind (2512 x 6624 -> 387 20.2 / 22.0,
  // 784 x 6272 -> 1387 19.5 / 20.7), and on two 1.05 up to 10000, 1.09 from there, some level or behind (1150 x 12544 ->
  // 1656 39.7 / 41.3).
  if (N > 64 && 2 * t64 > cus && two_a_cu) {
    const long sp = sharing(t128, 1536);
    if (sp >= 2 && 5 * sp * t128 >= 4 * cus &&
        K >= (t64 <= cus ? 14336 : 8192)) {
      shared(sp);
      return Tile::kM128S3;
    }
  }
  if (t64 <= cus && K >= (gather ? 1024 : 1536)) {
    if (K >= 8192) shared(sharing(t64, 1536));
    return Tile::kS64S4;
  }
  // Gathered operands (a convolution) of at most 64 columns: an address is made per 16 bytes of
  // pixels and stage, so 128-byte stages and tiles of 128 pixels pay from a reduction of 512 on
  // (140544 x 1584 -> 57 56.6 -> 38.4 us, 50176 x 2304 -> 32 24.9 -> 21.8, 50176 x 576 -> 48 14.6 ->
  // 13.6, 57600 x 10400 -> 64 123.5 -> 70.5), with less than a tile per CU the tiles of 64 (25088 x 576
  // -> 64 8.0 -> 6.8, 25088 x 720 -> 40 9.1 -> 8.0), on 256-byte stages from four of them on (6272 x 2304
  // -> 48 13.4 -> 10.5, 12544 x 2304 -> 64 13.8 -> 10.9, 25600 x 1152 -> 64 9.8 -> 9.7, 27648 x 20384 -> 64
  // 108.9 -> 72.7).  Short ones take 256 pixels once there are two such tiles per CU and more (529803 x
  // 144 -> 41 40.2 -> 31.2, 192000 x 432 -> 48 24.0 -> 18.7; 131072 x 432 -> 46, two exactly, is level).
  // At most 32 columns: 128 x 32 tiles, half of 64 columns would be padding (83824 x 2800 -> 19 33.1 -> 29.2,
  // 169756 x 3920 -> 10 63.3 -> 52.2, 68600 x 784 -> 23 14.2 -> 12.2, 60543 x 576 -> 28 9.2 -> 8.1, 178475 x 432 -> 12
  // 17.0 -> 15.2, 26244 x 784 -> 25 9.7 -> 9.1, but 163607 x 288 -> 16 11.0 -> 11.7).
  if (gather && N <= 32 && K >= 432 && 4 * t32 >= 3 * cus) return Tile::kN32K2;
  if (gather && N <= 64 && K >= 512) {
    // (tiles of 256 pixels, many of them, up to 800: 338724 x 576 -> 57 36.3 / 30.2, 159048 x 784 -> 45 24.4 /
    // 21.0, 467046 x 784 -> 34 60.8 / 47.5; 205379 x 864 -> 42 27.9 / 31.9, though of eight drawn of 800 ... 1008 none
    // is behind)
    if (K < 800 && tiles(256, 64) > 2 * cus) return Tile::kW64x2;
    if (tiles(128, 64) >= cus) return Tile::kR128K2;
    return K < 1024 ? Tile::kS64K2 : Tile::kS64K4;
  }
  if (gather && N <= 64)
    return tiles(256, 64) > 2 * cus ? Tile::kW64x2 : Tile::kS64x2;
  // Plain operands: 128-byte stages where there are more than two tiles a CU (65536 x 512 -> 64 17.9 ->
  // 16.3, 200704 x 1024 -> 64 75.5 -> 71.8, 65536 x 256 -> 64 10.4 -> 9.7)
  if (N <= 64) {
    if (K < 256) return Tile::kS64x2;
    if (K < 512 || !two_a_cu) return Tile::kS64K2;
    return Tile::kS64K4;
  }
  // Up to one 128 x 128 tile a CU, more than two of 64 x 64: eight waves on it, two stages under way (us, 64 x
  // 128, 128 x 64 or 128 x 128 tiles on four, whichever is first, and these: 741 x 6352 -> 4954, 234 tiles, 49.5 /
  // 40.1, 321 x 7248 -> 5932, 141, 47.0 / 40.7, 7853 x 2832 -> 441, 248, 23.8 / 21.3, 2048 x 2048 -> 2048, 256, 14.8 /
  // 14.5, 4096 x 3072 -> 768, 192, 18.2 / 17.7, 4096 x 768 -> 768 7.7 / 8.3; the convolutions 5203 x 22400 -> 701, 246,
  // 111.7 / 106.6, 15884 x 3136 -> 204, 250, 22.5 / 22.2, 9522 x 2016 -> 380, 225, 17.9 / 17.2, but 12544 x 2304 -> 256, 196
  // tiles without a ragged edge, 14.8 / 14.9, 12544 x 2880 -> 256 18.4 / 18.6; others of such widths would be ahead, 10192 x
  // 3744 -> 384 26.9 / 23.3).
  if (!two_a_cu && t128 <= cus && K >= 1536 && !(gather && N % 128 == 0 && K < 4096))
    return Tile::kM128S3;
  if (t128 >= cus) {
    if (K < 256) return 4 * tiles(256, 128) >= 3 * cus ? Tile::kW128x2 : Tile::kM128x2;
    // Gathered operands whose last 128 columns are half empty, on 128 x 64 tiles where these are one
    // round as well (16940 x 11760 -> 136, 266 and 399 tiles, 96.4 / 67.9, 18496 x 23520 -> 190, 290 and 435, 163.7 /
    // 135.0, 12138 x 2352 -> 269, 285 and 475, 24.2 / 20.6, 18963 x 288 -> 134, 298 and 447, 9.9 / 8.6, but 14045 x 1872 -> 294, 330
    // and 550, 22.2 / 24.3)
    if (gather && tiles(128, 64) < 2 * cus) return Tile::kR128K2;
    // One round of 128 x 128 tiles, two to a CU (us, 256 x 128 on 128-byte stages, which hold a CU alone,
    // and these, into int32: 16384 x 2048 -> 512 33.5 / 30.8, 9464 x 1920 -> 715 31.2 / 26.2, 2048 x 768 -> 4096 15.6 /
    // 14.5; on 64-byte stages 8192 x 256 -> 1024 12.1 / 11.1).  18 drawn layers are 1.09 times as fast into
    // int32 (0.97 to 1.19).  Into int8 they are 1.05 times as fast while the former are 0.75 to 0.9 a CU (55 layers,
    // 0.93 to 1.35; 8176 x 3376 -> 728 44.1 / 32.7) and 0.99 where those come out at nearly one (23, 0.91 to 1.13;
    // 832 x 2704 -> 7890 29.1 / 33.4, 16384 x 1968 -> 512 23.9 / 25.5, but 8656 x 5392 -> 883 67.3 / 59.7).
    // With a residual sum 8192 x 1024 -> 1024 16.1 / 16.7, 3136 x 512 -> 2048 12.0 / 11.0.
    // Very long reductions of gathered operands are ahead on the former (the convolutions 16000 x 6000 ->
    // 413 62.1 / 69.3, 7840 x 7600 -> 787 64.2 / 69.1, but 12544 x 4608 -> 512 38.7 / 37.8).
    if (t128 <= 2 * cus)
      return gather && K >= 5120 && 4 * tiles(256, 128) >= 3 * cus ? Tile::kW128K2 : Tile::kM128K2;
    // More of them: short reductions and gathered operands on 256 x 128 tiles, three to a CU, unless these
    // are wide and long or very long (128-byte stages, 256 x 128, 128 x 128: the convolutions 200704 x 576 ->
    // 128 45.5 / 33.8 / 41.0, 102400 x 864 -> 128 27.2 / 22.5 / 25.8, 72128 x 1296 -> 128 33.0 / 26.4 / 30.2, 102400 x
    // 2304 -> 128 52.4 / 46.8 / 50.0, 94080 x 4608 -> 100 83.7 / 74.8 / 71.7, 41600 x 2592 -> 512 82.3 / 91.2 / 83.7;
    // 131072 x 320 -> 128 25.5 / 20.5 / 24.6)
    if (K < 512 || (gather && K < (N > 128 ? 1024 : 4096))) return Tile::kW128x2;
    // else what comes out even of 64 x 128, three to a CU, and 128 x 128 (33000 x 512 -> 200, 516 of the
    // latter, 14.4 / 18.3, 90000 x 2048 -> 128, 704, 69.1 / 72.3, 131072 x 1024 -> 128, 1024, 60.6 / 58.1)
    return !gather && t128 <= 3 * cus ? Tile::kQ128K2 : Tile::kM128K2;
  }
  if (K < 256) return Tile::kS64x2;
  if (two_a_cu) {
    if (gather) {
      // A stage that is partly padding is an address for each 16 bytes of it all the same: 256-byte
      // stages from 768 on or where they are whole (3600 x 720 -> 128 7.0 -> 6.4, 3136 x 512 -> 512 7.3 ->
      // 6.8, but 3136 x 576 -> 512 7.0 -> 7.5), 128-byte ones where no more than a fifth of them is not
      // (3136 x 384 -> 192 6.1 -> 5.6, 6272 x 432 -> 256 7.0 -> 6.8, but 12544 x 288 -> 128 6.2 -> 6.3)
      if (K < 768 && K % 256 != 0)
        return K >= 512 || 5 * ((K + 127) / 128 * 128 - K) <= K ? Tile::kS64K2 : Tile::kS64x2;
      if (K < 512) return Tile::kS64K2;
    }
    return Tile::kS64K4;
  }
  // More tiles than that: half-size ones.  12544 x 2304 -> 256 takes 14.1 us on 392 tiles of 64 x 128
  // against 17.6 us on 784 tiles of 64 x 64, 12544 x 432 -> 256 8.0 against 8.8 (of a width between,
  // 7840 x 432 -> 316, 8.9 against 8.4).
  if (gather) {
    if (K < (N % 128 == 0 ? 384 : 512)) return Tile::kS64x2;
    return N % 128 == 0 ? Tile::kQ128K2 : Tile::kR128K2;
  }
  // Plain operands of a short reduction stay on the small ones up to three of them a CU (us, 64 x 64, 128 x
  // 64, 64 x 128: 4096 x 768 -> 768 from memory 9.3 / 10.0 / 9.4, again 7.6 / 8.1 / 8.2, 3000 x 512 -> 1024 6.8 / 7.2 / -
  // and 6.6 / 7.2 / 7.1; a few more, 12544 x 1024 -> 256, 784, 12.3 / 13.2 / 12.6 and 10.4 / 9.4 / 9.6).
  return t64 <= 3 * cus ? Tile::kS64K2 : Tile::kR128K2;
}

}  // namespace mxq
#endif  // MXQ_TILES_H_
