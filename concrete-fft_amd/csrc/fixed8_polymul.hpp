// fixed8_polymul.hpp -- the fused negacyclic product on fixed8_exec.hpp's
// eight-point schedule.
//
// What bounds it: latency and LDS exchanges, at 16 waves per CU (eight points
// of a transform are 32 registers; a product's two operands are held to 128, so
// that four waves run per SIMD: up to n = 1024 and for Dif16 some instances spill
// 12 to 28 bytes per lane for it).  Against the same programs with an exchange
// through LDS around every pass and transform, twiddles gathered from the
// n-point table after each butterfly (k_polymul_fixed, us): N = 2048 Dif4 / 512
// 14.6 -> 9.2 (1 product), 25.1 -> 18.7 (1024), 147.8 -> 121 (8192); Dit8 / 512
// 12.3 -> 7.4, 22.8 -> 14.3, 131 -> 108; N = 512 Dif4 / 256 12.6 -> 6.2 (1), 150
// -> 97 (32768); N = 8192 Dit8 / 1024 22.4 -> 18.5 (1), 235 -> 135 (2048); N =
// 16384 Dif8 / 512 38.3 -> 32.3 (1), 225 -> 156 (1024).  The compact table of
// the base transform took N = 8192 Dit8 / 1024 from 147 to 135, N = 16384 Dif8 /
// 1024 from 192 to 170.
#pragma once

#include <hip/hip_runtime.h>

#include "fixed8_exec.hpp"
#include "launch.hpp"
#include "lds_attr.hpp"

namespace {

using namespace cfft_dev;
using cfft_prog::Program;

template <int LOG2N>
struct Geom8 {
  static constexpr uint32_t n = 1u << LOG2N, T = n / 8;
  static constexpr uint32_t G = T < 64 ? 64 / T : 1;  // products per workgroup
  static constexpr uint32_t threads = T * G;
  static constexpr size_t lds = (size_t)G * lds_words(n) * sizeof(c64);
};

// One product per n / 8 threads (one workgroup each, two at n = 256); `tw` as
// in twiddles8.
template <int ALGO, int LOG2N, int LOG2BN>
__global__ void __launch_bounds__(Geom8<LOG2N>::threads) __attribute__((amdgpu_waves_per_eu(4, 4)))
k_polymul_fixed8(const uint64_t *__restrict__ A, const int64_t *__restrict__ B,
                 uint64_t *__restrict__ C, uint64_t batch, const c64 *__restrict__ tw,
                 const c64 *__restrict__ twist, const c64 *__restrict__ untwist) {
  using F = Fixed8<ALGO, LOG2N, LOG2BN, true>;
  using I = Fixed8<ALGO, LOG2N, LOG2BN, false>;
  using Ge = Geom8<LOG2N>;
  // From n = 2048 on a pass's twiddles wait for its points to leave the registers:
  // requested before that, 27 of the 41 instances spilled 12-44 bytes per lane (now
  // Dif16's, 12-20, which measured the same either way).  us, so and now: N = 16384
  // Dif4 / 1024 42.5 / 37.4 (1 product), 196 / 174 (1024), Dit4 / 1024 40.8 / 36.6,
  // 189 / 171; N = 8192 Dif8 / 1024 93 / 85 (1100), Dif4 / 1024 98 / 95; N = 4096
  // Dif8 / 512 39.2 / 37.5.  Up to n = 1024 it made no difference (0.98-1.03x).
  constexpr bool LATE = LOG2N >= 11 && !F::pair;
  constexpr uint32_t n = F::n;
  constexpr int LI = (int)I::prog.npass - 1;
  extern __shared__ c64 smem[];
  const uint32_t g = Ge::G == 1 ? 0 : threadIdx.x / F::T, lt = threadIdx.x % F::T;
  const uint64_t poly = (uint64_t)blockIdx.x * Ge::G + g;
  const uint64_t p = poly < batch ? poly : batch - 1;  // a last group without a product repeats one
  c64 *x = smem + g * lds_words(n);
  const uint64_t *a = A + p * (2ull * n);
  const int64_t *b = B + p * (2ull * n);
  uint64_t *c = C + p * (2ull * n);
  const Lane8<F> L(lt);
  auto settled = [] {  // every thread has read its last points
    if constexpr (F::T <= 64) wave_lds_fence();
    else __syncthreads();
  };
  c64 fa[8], fb[8], w[8];
  int64_t rb[16];
  {
    uint64_t ra[16];
#pragma unroll
    for (uint32_t m = 0; m < 8; ++m) {
      const uint32_t j = linear8<F, 0>(L, m);
      ra[2 * m] = ld_stream(&a[j]);
      ra[2 * m + 1] = ld_stream(&a[j + n]);
    }
    twiddles8<F, 0>(L, tw, w);
#pragma unroll
    for (uint32_t m = 0; m < 8; ++m)
      fa[m] = cmul(twist[linear8<F, 0>(L, m)],
                   mk(torus_to_f64(ra[2 * m]), torus_to_f64(ra[2 * m + 1])));
  }
#pragma unroll
  for (uint32_t m = 0; m < 8; ++m) {
    const uint32_t j = linear8<F, 0>(L, m);
    rb[2 * m] = ld_stream(&b[j]);
    rb[2 * m + 1] = ld_stream(&b[j + n]);
  }
  sched_fence();
  passes8<F, 0, LATE>(fa, w, x, L, tw);
  {
    const Lane8<F> L1(launder_u32(lt));
    const c64 *tz = launder(twist);
    twiddles8<F, 0>(L1, launder(tw), w);
#pragma unroll
    for (uint32_t m = 0; m < 8; ++m)
      fb[m] = cmul(tz[linear8<F, 0>(L1, m)], mk(i64_to_f64(rb[2 * m]), i64_to_f64(rb[2 * m + 1])));
  }
  settled();
  passes8<F, 0, LATE>(fb, w, x, L, tw);
#pragma unroll
  for (int m = 0; m < 8; ++m) fa[m] = cmul(fa[m], fb[m]);
  const Lane8<I> Li(launder_u32(lt));
  twiddles8<I, 0>(Li, launder(tw), w);
  settled();
  passes8<I, 0, LATE>(fa, w, x, Li, tw);
  if (poly >= batch) return;
  const c64 *uz = launder(untwist);
  const Lane8<I> Lo(launder_u32(lt));
#pragma unroll
  for (uint32_t m = 0; m < 8; ++m) {
    const uint32_t j = linear8<I, LI>(Lo, m);
    const c64 r = cmul(uz[j], fa[m]);
    st_stream(from_torus(r.re), &c[j]);
    st_stream(from_torus(r.im), &c[j + n]);
  }
}

// Launch the product of (ALGO, LOG2N, LOG2BN) if the plan's programs are that
// program; false if they are not (nothing launched).
template <int ALGO, int LOG2N, int LOG2BN>
bool fixed8_polymul_try(const Program &fwd, const Program &inv, const uint64_t *a, const int64_t *b,
                        uint64_t *c, uint64_t batch, const c64 *t, const c64 *tws, const c64 *utw,
                        hipStream_t s, hipError_t *e) {
  constexpr Program pf = cfft_prog::fixed_program(ALGO, LOG2N, LOG2BN, true);
  constexpr Program pi = cfft_prog::fixed_program(ALGO, LOG2N, LOG2BN, false);
  if (!cfft_prog::same_passes(fwd, pf) || !cfft_prog::same_passes(inv, pi)) return false;
  using Ge = Geom8<LOG2N>;
  const uint64_t blocks = (batch + Ge::G - 1) / Ge::G;
  const void *k = reinterpret_cast<const void *>(k_polymul_fixed8<ALGO, LOG2N, LOG2BN>);
  *e = cfft_launch::ensure_lds(k, Ge::lds);
  if (*e == hipSuccess)
    hipLaunchKernelGGL((k_polymul_fixed8<ALGO, LOG2N, LOG2BN>), dim3((uint32_t)blocks),
                       dim3(Ge::threads), Ge::lds, s, a, b, c, batch, t, tws, utw);
  if (*e == hipSuccess) *e = hipGetLastError();
  return true;
}

}  // namespace
