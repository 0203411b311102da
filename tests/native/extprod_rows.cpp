// Key rows requested by the one-launch external product, one line per request:
// log2n k1 glwes levels r0 rr i rows requested_row
#include <cstdint>
#include <cstdio>

#include "extprod_rows.hpp"

int main() {
  for (uint32_t log2n = 9; log2n <= 11; ++log2n)
    for (uint32_t k1 = 2; k1 <= 4; ++k1)
      for (uint32_t glwes = 1; glwes <= 4; glwes *= 2)
        for (uint32_t levels = 1; levels <= 64; ++levels) {
          // 8 waves; base transforms of at most 1024 points, 64 lanes each
          const uint32_t log2b = log2n < 10 ? log2n : 10, chunks = 1u << (log2n - log2b);
          const uint32_t units = 8 << (10 - log2b), points = chunks * ((1u << log2b) / 512);
          if (glwes * k1 * chunks > units) continue;
          const uint32_t per_round = cfft_dev::rows_per_round(units, chunks, glwes);
          const uint32_t kr = cfft_dev::rows_requested(chunks, points, k1, per_round);
          const uint32_t rows = k1 * levels;
          for (uint32_t r0 = 0; r0 < rows; r0 += per_round) {
            const uint32_t nr = rows - r0 < per_round ? rows - r0 : per_round;
            for (uint32_t rr = 0; rr < nr; rr += kr)
              for (uint32_t i = 0; i < kr; ++i)
                std::printf("%u %u %u %u %u %u %u %u %u\n", log2n, k1, glwes, levels, r0, rr, i,
                            rows, cfft_dev::key_row(r0, rr, i, rows));
          }
        }
  return 0;
}
