// Index arithmetic and launch rules of the kernels that hold without a GPU:
// plain functions of integers, used by the kernels and their launchers.
#pragma once

#include <cstdint>

namespace ihe {

// A result word (an accumulator's int32) plus a torus word, mod 2^32: torus words
// wrap as a matter of course, which a signed sum may not.
constexpr int32_t add_words(int32_t a, uint32_t b) { return (int32_t)((uint32_t)a + b); }

// Ring kernel: word tiles of 32 words (32 of them to a polynomial), and the
// 16-byte runs of u that its B operands are made of.
constexpr uint32_t kRingWordTiles = 32;
constexpr uint32_t kRuns = 2 * 32 * kRingWordTiles - 16;

// The word tile whose B operands a wave's tile `nt` reads. Three tiles a wave
// do not divide the 32 tiles, so the last wave's third one may lie past the
// last word: its result is dropped, and it reads the last tile's runs, where
// its own would start before the table.
constexpr uint32_t ring_operand_tile(uint32_t nt) {
  return nt < kRingWordTiles ? nt : kRingWordTiles - 1;
}

// Run that lane (h, c) reads for word tile nt (nt < kRingWordTiles) at K-block 0;
// K-block ks is 32 ks runs further on.
constexpr uint32_t ring_run(uint32_t nt, uint32_t h, uint32_t c) {
  return 32 * kRingWordTiles - 1 - 32 * nt - c + 16 * h;
}

// Column tiles per workgroup of the LDS-staged 128-row kernel (up to kMfmaLdsNkb
// K-blocks) for a launch of `tiles` tiles: few column tiles make enough
// workgroups of a small launch, many save a large one the start of each. us at
// 8 / 16 / 32, launches of each in turn, at 800 to 1,300 tiles with changing
// inputs and outputs (NS = 1024; 512; 333, whose columns are loaded by dwords):
//   2 K-blocks     61 tiles 15.7 / 20.2 / 34.3; 15.7 / 22.8 / 38.1; 17.2 / 24.1 / 41.7
//                 121: 29.4 / 26.6 / 38.0; 30.0 / 27.4 / 39.2; 29.9 / 30.4 / 42.5
//               1,950: 483 / 486 / 500; 417 / 400 / 397; 408 / 404 / 407
//   3              60: 17.6 / 25.8 / 43.3; 18.4 / 28.2 / 47.6; 21.1 / 30.7 / 53.8
//                 239: 61.0 / 61.4 / 67.5; 62.4 / 63.0 / 69.1; 66.0 / 66.7 / 75.1
//                 846: 244 / 233 / 250; 256 / 245 / 241; 216 / 216 / 223
//               1,238: 356 / 341 / 346; 372 / 356 / 340; 384 / 373 / 372
//               1,933: 562 / 540 / 539; 599 / 576 / 526; 514 / 508 / 511
//   4             116: 37.1 / 40.8 / 50.9; 39.5 / 41.4 / 54.8; 43.4 / 44.6 / 59.0
//                 126: 44.5 / 42.0 / 52.2; 45.1 / 42.5 / 57.9; 50.0 / 46.3 / 59.6
//                 141: 48.4 / 48.9 / 64.8; 48.4 / 51.9 / 66.2; 52.2 / 56.9 / 75.2
//                 182: 58.5 / 56.3 / 69.5; 61.2 / 58.0 / 72.0; 66.8 / 64.8 / 78.6
//                 916: 296 / 280 / 284; 298 / 288 / 286; 307 / 290 / 310
//               1,103: 357 / 340 / 329; 354 / 343 / 334; 377 / 370 / 364
//   5             920: 349 / 337 / 340; 351 / 345 / 348; 365 / 365 / 373
//                 980: 373 / 361 / 357; 372 / 367 / 361; 391 / 390 / 388
//   6             899: 381 / 363 / 364; 377 / 369 / 381; 402 / 398 / 409
//                 978: 413 / 400 / 391; 410 / 405 / 406; 439 / 437 / 434
//               1,907: 819 / 794 / 777; 849 / 821 / 814; 915 / 885 / 873
// Four K-blocks change over twice: 16 column tiles make 4 workgroups a tile, so
// 128 tiles fill 256 CUs with two each and 192 with three, and 8 column tiles
// split more evenly just past either (up to 120 tiles their 8 a tile and the
// variance blocks all fit the chip at once). From 900 tiles on 16 and 32 lie
// within a few per cent of each other, either way by layout, until 32 wins.
constexpr int kMfmaLdsNkb = 6;
constexpr int wide_ntw(int nkb, uint32_t tiles) {
  const bool few = nkb <= 2   ? tiles < 100
                   : nkb != 4 ? tiles < 200
                              : tiles <= 120 || (tiles > 128 && tiles <= 152) ||
                                    (tiles > 192 && tiles < 200);
  if (few) return 8;
  return nkb > 2 && tiles >= 900 ? 32 : 16;
}

// Column tiles of a batch's 128-row family of `tiles` tiles, whose bands run up
// to `most` by themselves, the largest of them with `band_tiles` tiles. A launch
// no larger than a band keeps the band's count (the autotuner may have measured
// it); a larger one goes by its own tiles.
constexpr int family_ntw(int nkb, int most, uint32_t band_tiles, uint32_t tiles) {
  const int rule = wide_ntw(nkb, tiles);
  return tiles > band_tiles && rule > most ? rule : most;
}

}  // namespace ihe
