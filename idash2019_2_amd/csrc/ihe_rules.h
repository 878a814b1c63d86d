// Index arithmetic and launch rules of the kernels that hold without a GPU:
// plain functions of integers, used by the kernels and their launchers.
#pragma once

#include <cstdint>

namespace ihe {

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

}  // namespace ihe
