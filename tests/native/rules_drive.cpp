// The kernels' index arithmetic and launch rules, walked on the CPU over every
// form that they are used in. Prints the first value that is out of place and
// ends with 1; 0 when all hold.
#include <cstdio>
#include <initializer_list>

#include "ihe_rules.h"

using namespace ihe;

// Sums of torus words wrap (an overflowing signed sum is no constant expression,
// so it would not compile here).
static_assert(add_words(INT32_MAX, 1u) == INT32_MIN && add_words(INT32_MIN, 0x80000000u) == 0 &&
              add_words(-1, 1u) == 0 && add_words(INT32_MIN, 0xFFFFFFFFu) == INT32_MAX, "mod 2^32");

// Ring kernel: every B operand that an active wave reads, at every number of
// tiles a wave, lies in the table of runs, and tiles that give results read
// their own.
static int ring_operands() {
  for (uint32_t tpw = 1; tpw <= 4; ++tpw)
    for (uint32_t nt0 = 0; nt0 < kRingWordTiles; nt0 += tpw)
      for (uint32_t t = 0; t < tpw; ++t) {
        const uint32_t nt = ring_operand_tile(nt0 + t);
        if (nt0 + t < kRingWordTiles && nt != nt0 + t)
          return std::printf("%u tiles a wave: tile %u reads tile %u\n", tpw, nt0 + t, nt), 1;
        for (uint32_t h = 0; h < 2; ++h)
          for (uint32_t c = 0; c < 32; ++c) {
            const int64_t first = (int32_t)ring_run(nt, h, c), last = first + 32 * 31;
            if (first < 0 || last >= (int64_t)kRuns)
              return std::printf("%u tiles a wave: tile %u, lane (%u, %u) reads runs %lld .. %lld of %u\n",
                                 tpw, nt0 + t, h, c, (long long)first, (long long)last, kRuns), 1;
          }
      }
  return 0;
}

// Column tiles of 128-row launches where one count was the fastest of the three
// in most layouts measured (the table at wide_ntw).
static int column_tiles() {
  const struct {
    int nkb;
    uint32_t tiles;
    int ntw;
  } measured[] = {{2, 36, 8},   {2, 93, 8},    {2, 177, 16},  {3, 36, 8},    {3, 119, 8},
                  {3, 888, 16}, {3, 1780, 32}, {4, 38, 8},    {4, 120, 8},   {4, 122, 16},
                  {4, 126, 16}, {4, 130, 8},   {4, 150, 8},   {4, 154, 16},  {4, 182, 16},
                  {4, 190, 16}, {4, 251, 16},  {4, 1103, 32}, {4, 2049, 32}, {5, 36, 8},
                  {5, 84, 8},   {5, 980, 32},  {5, 1605, 32}, {6, 36, 8},    {6, 90, 8},
                  {6, 899, 16}, {6, 1223, 32}, {6, 1907, 32}};
  for (const auto &m : measured)
    if (wide_ntw(m.nkb, m.tiles) != m.ntw)
      return std::printf("%d K-blocks, %u tiles: %d column tiles instead of %d\n", m.nkb, m.tiles,
                         wide_ntw(m.nkb, m.tiles), m.ntw), 1;
  return 0;
}

// A batch keeps the count that a band of its own size was tuned to; a launch of
// more tiles than its bands goes by the rule, but not below them.
static int family_column_tiles() {
  for (int nkb = 2; nkb <= kMfmaLdsNkb; ++nkb)
    for (int most : {8, 16, 32})
      for (uint32_t band : {1u, 119u, 378u, 1907u}) {
        if (family_ntw(nkb, most, band, band) != most)
          return std::printf("%d K-blocks: a launch of its band's %u tiles runs %d instead of %d\n",
                             nkb, band, family_ntw(nkb, most, band, band), most), 1;
        for (uint32_t tiles : {band + 1, 2 * band, 16 * band}) {
          const int rule = wide_ntw(nkb, tiles), want = tiles == band || rule < most ? most : rule;
          if (family_ntw(nkb, most, band, tiles) != want)
            return std::printf("%d K-blocks: %u tiles of %u-tile bands run %d instead of %d\n", nkb,
                               tiles, band, family_ntw(nkb, most, band, tiles), want), 1;
        }
      }
  return 0;
}

int main() { return ring_operands() || column_tiles() || family_column_tiles(); }
