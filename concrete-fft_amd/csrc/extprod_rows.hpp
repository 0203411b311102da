// extprod_rows.hpp -- which calls the one-launch external product
// (extprod_fused_kernels.hip) takes, and the key rows it requests for a round's
// multiply-accumulate.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define CFFT_ROWS_FN __host__ __device__ constexpr
#else
#define CFFT_ROWS_FN constexpr
#endif

namespace cfft_dev {

// rows of one GLWE in a round: `units` base transforms in flight, `chunks` of
// them per polynomial, `glwes` per workgroup
CFFT_ROWS_FN uint32_t rows_per_round(uint32_t units, uint32_t chunks, uint32_t glwes) {
  return units / chunks / glwes;
}

// rows whose key points (`points` per row and column) a thread requests
// together: as many as fit beside the sums, at most 8 and a round's
CFFT_ROWS_FN uint32_t rows_requested(uint32_t chunks, uint32_t points, uint32_t k1,
                                     uint32_t per_round) {
  const uint32_t fit = (chunks == 1 ? 24 : 16) / (points * k1);
  const uint32_t some = fit < 1 ? 1 : fit < 8 ? fit : 8;
  return some < per_round ? some : per_round;
}

// The row that request i of a group starting at round row rr reads, in the
// round that starts at row r0 of `rows`: its own, or the key's last one again
// where the group runs past it (those points are never used).
CFFT_ROWS_FN uint32_t key_row(uint32_t r0, uint32_t rr, uint32_t i, uint32_t rows) {
  const uint32_t row = r0 + rr + i;
  return row < rows ? row : rows - 1;
}

// Whether a call runs on the one-launch form (k1 = 2 ... 4: its column sums are
// registers) on a device of `cus` compute units.  Over N = 1024, 2048, 4096, 1 to
// 64 rows and 1 to 2300 GLWEs it measured up to 2.7x faster than the split form,
// whatever the width of the digits, but for three groups of shapes (us, split /
// one launch):
// - Many rows, few GLWEs: one CU runs in rounds the rows that the split form
//   spreads over idle CUs.  From 4 rounds on the split form is ahead below about 2
//   rounds^2 GLWEs (N = 4096, 16 rows, 4 rounds: 51.9 / 60.2 for 8 GLWEs, 64.0 /
//   61.1 for 40; 32 rows, 8 rounds: 100 / 126 for 64, 288 / 251 for 260; N = 2048,
//   32 rows: 52.0 / 56.8 for 24, 57.7 / 57.0 for 40); at 3 rounds below 16 with
//   wide digits (levels * base_log > 31) and k1 = 3 or 4 (N = 2048, k1 = 4, 5 x 7
//   33.2 / 36.4 for 4, 36.4 / 36.8 for 16; N = 4096, k1 = 3, 4 x 10 43.7 / 46.4 for
//   1, 48.3 / 47.3 for 16); and at N = 4096, k1 = 4 from 3 rounds on below twice as
//   many (3 x 10 43.4 / 47.5 for 4, 47.0 / 48.0 for 16, 52.2 / 48.7 for 40; 3 x 11
//   43.1 / 50.7 for 2, 52.2 / 52.0 for 40; 4 x 10 64.1 / 66.0 for 40; 6 x 5 82.0 /
//   88.2 for 72).  k1 = 2 gains at 3 rounds from 2 GLWEs on (N = 4096, 6 x 6 40.5 /
//   42.0 for 1, 49.8 / 42.5 for 2).
// - Wide digits, k1 = 3, and a last pass over the CUs so short that the split
//   form's columns still fill the chip only once (3 batch column waves, 4 per CU at N
//   = 4096): N = 4096, 2 x 16 56.3 / 59.0 for 257, 59.0 / 60.8 for 337, 88.1 / 60.8
//   for 357; 6 x 6 126.6 / 134.4 for 297; one level only below N = 4096: N = 2048,
//   1 x 32 33.8 / 36.8 for 533, 36.0 / 37.2 for 673, 59.1 / 37.3 for 693; N = 1024
//   36.9 / 38.3 for 1160, 64.3 / 39.0 for 1385 (1 x 32 at N = 4096 44.3 / 42.4 for
//   300).
CFFT_ROWS_FN bool one_launch(uint32_t log2n, uint64_t batch, uint32_t k1, uint32_t levels,
                             uint32_t base_log, uint32_t cus) {
  if (log2n < 9 || log2n > 11 || k1 < 2 || k1 > 4) return false;
  const bool wide = levels * base_log > 31;
  const uint64_t per_round = log2n == 9 ? 16 : log2n == 10 ? 8 : 4;
  const uint64_t rounds = (k1 * (uint64_t)levels + per_round - 1) / per_round;
  const bool large4 = log2n == 11 && k1 == 4;
  uint64_t least = 0;
  if (rounds > 3) least = 2 * rounds * rounds;
  else if (rounds == 3 && (large4 || (wide && k1 > 2))) least = 16;
  if (batch < (large4 ? 2 * least : least)) return false;
  const uint64_t fill = (uint64_t)cus << (11 - log2n);
  const bool band = wide && k1 == 3 && (levels > 1) == (log2n == 11);
  return !(band && batch > fill && 3 * batch <= 4 * fill);
}

}  // namespace cfft_dev
