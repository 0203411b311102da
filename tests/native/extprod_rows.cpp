// Without arguments: the key rows requested by the one-launch external product,
// one line per request: log2n k1 glwes levels r0 rr i rows requested_row.
// With an argument: for every line "N k1 levels base_log batch cus" of the
// input, 1 if the call runs on that form, else 0.
#include <cstdint>
#include <cstdio>

#include "extprod_rows.hpp"

int main(int argc, char **) {
  if (argc > 1) {
    unsigned N, k1, levels, base_log, cus;
    unsigned long long batch;
    while (std::scanf("%u %u %u %u %llu %u", &N, &k1, &levels, &base_log, &batch, &cus) == 6) {
      uint32_t log2n = 0;
      while ((2u << log2n) < N) ++log2n;
      std::printf("%d\n", cfft_dev::one_launch(log2n, batch, k1, levels, base_log, cus) ? 1 : 0);
    }
    return 0;
  }
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
