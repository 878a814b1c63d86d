// The kernels' index arithmetic and launch rules, walked on the CPU over every
// form that they are used in. Prints the first value that is out of place and
// ends with 1; 0 when all hold.
#include <cstdio>

#include "ihe_rules.h"

using namespace ihe;

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

int main() { return ring_operands(); }
