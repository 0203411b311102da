// r16s_exec.hpp -- wave-local Dif16 transforms of 256, 512 and 1024 points for
// kernels that fill a CU's LDS: r16l_transform (r16_exec.hpp) with the twiddle
// rows k >= 1 only (T[0] = 1 is never multiplied) and an exchange buffer of
// exactly 2^LB points, point i at i ^ ((i >> 4) & 15) as in r16x_transform.
// With them 8 waves' buffers, the rows and a 1024-entry twist table take 163
// 776 of the 163 840 bytes.
#pragma once

#include "r16_exec.hpp"

namespace cfft_dev {

// the 1024-point r16 block's rows k = 1 ... 15: T[k l] (15 x 64), T[16 k p] (15 x 4)
constexpr uint32_t kSTw1 = 15 * 64, kSTw = kSTw1 + 15 * 4;
// their place in the plan's block, whose rows start at k = 0 (zero past the end:
// any valid entry)
__device__ __forceinline__ uint32_t r16s_block_index(uint32_t i) {
  return i < kSTw1 ? 64 + i : i < kSTw ? 1024 + 4 + (i - kSTw1) : 0;
}

// NV (1 or 2) transforms on T = 2^LB / 16 lanes (64 / T lane groups per wave),
// sharing every twiddle read; layouts and operations as r16l_transform.
template <int LB, bool FWD, int NV>
__device__ __forceinline__ void r16s_transform(c64 *va, c64 *vb, c64 *x, uint32_t l,
                                               const c64 *tw) {
  using S = R16<LB>;
  static_assert(LB >= 8 && LB <= 10, "one transform must fit a wavefront");
  constexpr uint32_t cs = 1u << (10 - LB);  // column stride in the 1024-point block
  const uint32_t p = l >> 4, q = l & 15;
  butterfly<16, FWD>(va);
  if (NV == 2) butterfly<16, FWD>(vb);
  sched_fence();
  twiddle_rows_x2<FWD>(va, vb, NV, tw, 64, l * cs);
#pragma unroll
  for (int t = 0; t < NV; ++t) {
    c64 *v = t == 0 ? va : vb;
    wave_lds_fence();
#pragma unroll
    for (int k = 0; k < 16; ++k) x[16 * l + ((uint32_t)k ^ q)] = v[k];
    wave_lds_fence();
#pragma unroll
    for (int k = 0; k < 16; ++k)
      v[k] = x[S::T * (uint32_t)k + 16 * p + (q ^ ((p + S::T / 16 * (uint32_t)k) & 15))];
  }
  wave_lds_fence();  // last use of x
  butterfly<16, FWD>(va);
  if (NV == 2) butterfly<16, FWD>(vb);
  if constexpr (LB > 8) {
    sched_fence();
    twiddle_rows_x2<FWD>(va, vb, NV, tw + kSTw1, 4, p * cs);
    r16_exchange2_rows<LB>(va);
    if (NV == 2) r16_exchange2_rows<LB>(vb);
#pragma unroll
    for (uint32_t i = 0; i < S::NB; ++i) {
      butterfly<S::REND, FWD>(va + i * S::REND);
      if (NV == 2) butterfly<S::REND, FWD>(vb + i * S::REND);
    }
  }
}

}  // namespace cfft_dev
