// fixed8_fft.hpp -- whole transforms on fixed8_exec.hpp's eight-point schedule for
// host calls of a few transforms.  No table is staged, a transform has n / 8
// threads, and each workgroup tells the polling host when its results are
// written: waiting for the stream instead costs the round trip of a completion
// signal (a one-wave kernel on mapped memory, launch to return: 12.0 us through
// hipStreamSynchronize, 23 polling hipStreamQuery, 7.7 polling a word it wrote).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "fixed8_exec.hpp"
#include "fixed_exec.hpp"
#include "launch.hpp"
#include "lds_attr.hpp"

namespace {

using namespace cfft_dev;
using cfft_prog::Program;

template <int LOG2N>
struct GeomFft8 {
  static constexpr uint32_t n = 1u << LOG2N, T = n / 8;
  static constexpr uint32_t G = T < 64 ? 64 / T : 1;  // transforms per workgroup
  static constexpr uint32_t threads = T * G;
  static constexpr size_t lds = (size_t)G * lds_words(n) * sizeof(c64);
};

// flags[workgroup] (host memory) is set to 1 once the workgroup's results are
// visible to the host.
__device__ __forceinline__ void tell_host(uint32_t *flags) {
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(&flags[blockIdx.x], 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// In place.
template <int ALGO, int LOG2N, int LOG2BN, bool FWD>
__global__ void __launch_bounds__(GeomFft8<LOG2N>::threads)
k_fft_fixed8(c64 *__restrict__ data, uint64_t ntrans, uint64_t stride, const c64 *__restrict__ tw,
             uint32_t *flags) {
  using F = Fixed8<ALGO, LOG2N, LOG2BN, FWD>;
  using Ge = GeomFft8<LOG2N>;
  constexpr int LAST = (int)F::prog.npass - 1;
  extern __shared__ c64 smem[];
  const uint32_t g = Ge::G == 1 ? 0 : threadIdx.x / F::T, lt = threadIdx.x % F::T;
  const uint64_t tr = (uint64_t)blockIdx.x * Ge::G + g;
  const bool active = tr < ntrans;
  c64 *d = data + (active ? tr : ntrans - 1) * stride;
  c64 *x = smem + g * lds_words(F::n);
  const Lane8<F> L(lt);
  c64 v[8], w[8];
#pragma unroll
  for (uint32_t m = 0; m < 8; ++m) v[m] = d[linear8<F, 0>(L, m)];
  twiddles8<F, 0>(L, tw, w);
  passes8<F, 0>(v, w, x, L, tw);
  if (active) {
#pragma unroll
    for (uint32_t m = 0; m < 8; ++m) d[linear8<F, LAST>(L, m)] = v[m];
  }
  tell_host(flags);
}

// The same for programs the eight-point schedule does not take (Dit16, and Dif16
// below 512 points): 16 points per thread through LDS around every pass.
template <int LOG2N>
struct GeomFft16 {
  static constexpr uint32_t n = 1u << LOG2N, T = n / 16;
  static constexpr uint32_t G = T < 64 ? 64 / T : 1;
  static constexpr uint32_t threads = T * G;
  static constexpr size_t lds = (size_t)G * lds_words(n) * sizeof(c64);
};
template <int ALGO, int LOG2N, int LOG2BN, bool FWD>
__global__ void __launch_bounds__(GeomFft16<LOG2N>::threads)
k_fft_fixed16(c64 *__restrict__ data, uint64_t ntrans, uint64_t stride, const c64 *__restrict__ tw,
              uint32_t *flags) {
  using Ge = GeomFft16<LOG2N>;
  extern __shared__ c64 smem[];
  const uint32_t g = threadIdx.x / Ge::T, lt = threadIdx.x % Ge::T;
  const uint64_t tr = (uint64_t)blockIdx.x * Ge::G + g;
  const bool active = tr < ntrans;
  c64 *d = data + (active ? tr : ntrans - 1) * stride;
  auto load = [&](uint32_t pos) -> c64 { return d[pos]; };
  auto store = [&](uint32_t pos, c64 v) {
    if (active) d[pos] = v;
  };
  run_fixed_program<FixedProg<ALGO, LOG2N, LOG2BN, FWD>, 0, 16>(smem + g * lds_words(Ge::n), lt,
                                                                Ge::T, tw, load, store);
  tell_host(flags);
}

// Launch the transform of (ALGO, LOG2N, LOG2BN) if `prog` is its program; false
// if it is not (nothing launched).
template <int ALGO, int LOG2N, int LOG2BN>
bool fixed8_fft_try(const Program &prog, c64 *d, uint64_t ntrans, uint64_t stride, const c64 *t,
                    cfft_launch::HostDone *done, hipStream_t s, hipError_t *e) {
  const bool fwd = prog.npass != 0 && prog.p[0].fwd != 0;
  constexpr Program pf = cfft_prog::fixed_program(ALGO, LOG2N, LOG2BN, true);
  constexpr Program pi = cfft_prog::fixed_program(ALGO, LOG2N, LOG2BN, false);
  if (!cfft_prog::same_passes(prog, fwd ? pf : pi)) return false;
  constexpr bool eight = ALGO < 6 || (ALGO == 6 && LOG2BN >= 9);
  using Ge = typename std::conditional<eight, GeomFft8<LOG2N>, GeomFft16<LOG2N>>::type;
  static_assert(Ge::lds <= 64 * 1024, "no raised LDS limit");
  const uint64_t wgs = (ntrans + Ge::G - 1) / Ge::G;
  if (wgs > done->capacity) return false;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((uint32_t)wgs), dim3(Ge::threads), Ge::lds, s, d, ntrans,
                       stride, t, done->flags);
  };
  if constexpr (eight) {
    if (fwd) launch(k_fft_fixed8<ALGO, LOG2N, LOG2BN, true>);
    else launch(k_fft_fixed8<ALGO, LOG2N, LOG2BN, false>);
  } else {
    if (fwd) launch(k_fft_fixed16<ALGO, LOG2N, LOG2BN, true>);
    else launch(k_fft_fixed16<ALGO, LOG2N, LOG2BN, false>);
  }
  *e = hipGetLastError();
  if (*e == hipSuccess) done->used = (uint32_t)wgs;
  return true;
}

}  // namespace
