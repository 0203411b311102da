// extprod_rows.hpp -- the key rows that the one-launch external product
// (extprod_fused_kernels.hip) requests for a round's multiply-accumulate.
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

}  // namespace cfft_dev
