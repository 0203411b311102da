// fixed8_exec.hpp -- a plan's pass program fixed at compile time, on eight
// points per thread held in registers between the first and the last pass.
//
// A transform of n points runs on n / 8 threads.  Each base chunk (base_n
// points) belongs to base_n / 8 consecutive threads, so with base_n = 512 the
// base passes of a chunk stay within one wavefront and exchange through LDS
// without a workgroup barrier; depth passes run over the whole transform.  A
// pass takes its butterflies' inputs from registers (first pass) or LDS,
// requests the next pass's twiddles as soon as it has used its own (or has stored
// its outputs, passes8), so that they arrive during the exchange, and leaves its outputs in LDS or (last
// pass) in registers.  Every thread's inputs and outputs of a whole transform
// are the same eight points, so loads, twist, pointwise product and the
// hand-over from a forward to an inverse transform need no exchange.
//
// Radix-16 butterflies (Dif16) are shared by the lanes l and l + 32 of a
// wavefront: lane half o holds the inputs k of parity o.  The radix-16
// butterfly is two radix-8 butterflies, on its even and its odd inputs, whose
// outputs A_k and B_k combine as A_k +- w_k B_k (device_math.hpp, bf16): each
// half runs one of them, the halves then swap four outputs
// (v_permlane32_swap) and lower lanes combine k = 0 ... 3, upper lanes k = 4
// ... 7.  The operations are bf16's, so are the bits.
//
// Operations, operand order and twiddle table entries are the runtime
// executor's (stockham_exec.hpp).
#pragma once

#include "device_math.hpp"
#include "program.hpp"
#include "r16_exec.hpp"
#include "stockham_exec.hpp"

namespace cfft_dev {

// the pass program of (ALGO, 2^LOG2N points, base 2^LOG2BN) in one direction
template <int ALGO, int LOG2N, int LOG2BN, bool FWD>
struct Fixed8 {
  static_assert(ALGO != 7, "Dit16 outputs do not come back to their threads");
  static constexpr Program prog = cfft_prog::fixed_program(ALGO, LOG2N, LOG2BN, FWD);
  static constexpr bool fwd = FWD;
  static constexpr bool pair = ALGO == 6;  // radix-16 cores on lane pairs
  static constexpr uint32_t n = 1u << LOG2N, b = 1u << LOG2BN;
  static constexpr uint32_t T = n / 8, TC = b / 8;  // threads per transform, per chunk
  static_assert(!pair || TC >= 64, "lane pairs need whole wavefronts");
};

template <class F, int PI>
struct Pass8 {
  static constexpr Pass P = F::prog.p[PI];
  static constexpr int R = P.radix;
  static constexpr bool depth = P.kind == cfft_prog::DEPTH_FWD || P.kind == cfft_prog::DEPTH_INV;
  static constexpr bool core = P.kind == cfft_prog::DIF_CORE || P.kind == cfft_prog::DIT_CORE;
  static constexpr bool p16 = R == 16 && F::pair;
  static constexpr int NB = p16 ? 1 : 8 / R;  // butterflies per thread
  static constexpr uint32_t lr = RadixLog<R>::value;
  static constexpr uint32_t log2m = P.log2len - lr, m = 1u << log2m;
  static constexpr bool pre = P.kind == cfft_prog::DIT_CORE || P.kind == cfft_prog::DEPTH_INV;
  static constexpr bool post = P.kind == cfft_prog::DIF_CORE || P.kind == cfft_prog::DEPTH_FWD;
  static constexpr int NT = !(pre || post) ? 0 : p16 ? 8 : NB * (R - 1);  // twiddles per thread
};

// the thread's place: chunk start, index in the chunk and, for lane pairs,
// the butterfly and the half
template <class F>
struct Lane8 {
  uint32_t lt, base, lc, bb, o;
  __device__ __forceinline__ explicit Lane8(uint32_t t) {
    lt = t;
    base = (t / F::TC) * F::b;
    lc = t % F::TC;
    bb = (lc & 31) + 32 * (lc >> 6);
    o = (lc >> 5) & 1;
  }
};

// butterfly i of the thread in pass P: start of its chunk and index in it
template <class F, class Q>
__device__ __forceinline__ void butterfly8(const Lane8<F> &L, int i, uint32_t &base, uint32_t &bb) {
  if constexpr (Q::depth) {
    const uint32_t B = L.lt + F::T * (uint32_t)i;
    base = (B >> Q::log2m) << Q::P.log2len;
    bb = B & (Q::m - 1);
  } else if constexpr (F::pair) {
    // an end butterfly of a Dif16 plan keeps to the points of the lane's parity
    base = L.base;
    bb = L.bb + (Q::p16 ? 0 : F::b / 16 * (2 * (uint32_t)i + L.o));
  } else {
    base = L.base;
    bb = L.lc + F::TC * (uint32_t)i;
  }
}

// LDS point of input / output k of butterfly (base, bb)
template <class F, class Q>
__device__ __forceinline__ uint32_t in_point(uint32_t base, uint32_t bb, uint32_t k) {
  if constexpr (Q::P.kind == cfft_prog::DIT_CORE) {
    const uint32_t p = bb >> Q::P.s, q = bb & ((1u << Q::P.s) - 1);
    return base + (p << (Q::lr + Q::P.s)) + (k << Q::P.s) + q;
  } else if constexpr (Q::P.kind == cfft_prog::DEPTH_INV) {
    return base + ((uint32_t)bitrev_digit<Q::R>((int)k) << Q::log2m) + bb;
  } else {
    return base + (k << Q::log2m) + bb;
  }
}
template <class F, class Q>
__device__ __forceinline__ uint32_t out_point(uint32_t base, uint32_t bb, uint32_t k) {
  if constexpr (Q::P.kind == cfft_prog::DIF_CORE) {
    const uint32_t p = bb >> Q::P.s, q = bb & ((1u << Q::P.s) - 1);
    return base + q + (((p << Q::lr) + k) << Q::P.s);
  } else if constexpr (Q::P.kind == cfft_prog::DEPTH_FWD) {
    return base + ((uint32_t)bitrev_digit<Q::R>((int)k) << Q::log2m) + bb;
  } else {
    return base + (k << Q::log2m) + bb;
  }
}
// outputs of a lane pair's radix-16 butterfly: sum r is output k, difference r
// output k ^ 8
template <class F>
__device__ __forceinline__ uint32_t pair_out(const Lane8<F> &L, int j) {
  const uint32_t r = (uint32_t)(j & 3), diff = (uint32_t)(j >> 2);
  return r + (L.o ? 12 - 8 * diff : 8 * diff);
}

// the twiddles of a pass, requested.  `tw`: T[j] of the n-point transform (n
// entries), then for the core passes the base transform's own T[j n / b] (b
// entries: neighbouring lanes' factors lie n / b times closer together)
template <class F, int PI>
__device__ __forceinline__ void twiddles8(const Lane8<F> &L, const c64 *__restrict__ tw, c64 *w) {
  using Q = Pass8<F, PI>;
  if constexpr (Q::NT > 0) {
    if constexpr (Q::core && F::b < F::n) tw += F::n;
    if constexpr (Q::p16) {
      static_assert(!Q::p16 || Q::post, "Dif16 cores multiply after the butterfly");
      const uint32_t p = L.bb >> Q::P.s;
#pragma unroll
      for (int j = 0; j < 8; ++j) w[j] = tw[(pair_out(L, j) * p) << Q::P.s];
    } else {
#pragma unroll
      for (int i = 0; i < Q::NB; ++i) {
        uint32_t base, bb;
        butterfly8<F, Q>(L, i, base, bb);
        const uint32_t p = Q::core ? bb >> Q::P.s : bb, sh = Q::core ? Q::P.s : Q::P.tw_mul;
#pragma unroll
        for (int k = 1; k < Q::R; ++k)
          w[i * (Q::R - 1) + k - 1] = tw[((uint32_t)k * p) << sh];
      }
    }
    if constexpr (!F::fwd) {
#pragma unroll
      for (int j = 0; j < Q::NT; ++j) w[j].im = -w[j].im;
    }
  }
}

// radix-16 butterfly of a lane pair: v[j] = input 2 j + o on entry, sums in
// v[0..3] and differences in v[4..7] on exit
template <bool FWD>
__device__ __forceinline__ void bf16_pair(c64 *v, uint32_t o) {
  bf8<FWD>(v);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    swap_rows32(v[r].re, v[4 + r].re);
    swap_rows32(v[r].im, v[4 + r].im);
  }
  // v[r] = A_k, v[4 + r] = B_k with k = r (o = 0) or r + 4 (o = 1)
  const bool up = o != 0;
  // B_0, or j B_4
  const c64 j4 = mul_j<FWD>(v[4]);
  const c64 t0 = up ? j4 : v[4];
  // exp(-+ i pi / 8) B_1, or exp(-+ 5 i pi / 8) B_5 (mul_exp_pi_over_16, mul_exp_17pi_over_16)
  const c64 w1 = up ? mk(-kH1Y, FWD ? kH1X : -kH1X) : mk(kH1X, FWD ? kH1Y : -kH1Y);
  const c64 t1 = cmul(w1, v[5]);
  // mul_exp_pi_over_8: (re -+ im, im +- re) scaled
  const c64 a = mul_j<!FWD>(v[6]), b = mul_j<FWD>(v[6]);
  const c64 s2 = cadd(v[6], up ? b : a);
  const c64 t2 = mk(kFrac1Sqrt2 * s2.re, kFrac1Sqrt2 * s2.im);
  const c64 w3 = up ? mk(kH1X, FWD ? -kH1Y : kH1Y) : mk(-kH1Y, FWD ? -kH1X : kH1X);
  const c64 t3 = cmul(w3, v[7]);
  const c64 t[4] = {t0, t1, t2, t3};
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const c64 x = v[r];
    v[r] = cadd(x, t[r]);
    v[4 + r] = csub(x, t[r]);
  }
}

// passes PI ... of F: v[m] holds the thread's point m on entry of the first
// pass (slot order of `linear8`) and on exit of the last; w holds pass PI's
// twiddles.  `x`: n + n / 16 points of LDS; the caller's earlier reads of it
// by other threads must be complete.  LATE: the next pass's twiddles are
// requested once its points are in LDS and no longer in registers (for callers
// that hold another transform meanwhile), else before those are stored.
template <class F, int PI, bool LATE = false>
__device__ __forceinline__ void passes8(c64 *v, c64 *w, c64 *x, const Lane8<F> &L0,
                                        const c64 *__restrict__ tw) {
  using Q = Pass8<F, PI>;
  constexpr bool first = PI == 0, last = PI + 1 == (int)F::prog.npass;
  constexpr bool wave_in = !first && !Q::depth && F::TC <= 64;
  const Lane8<F> L(launder_u32(L0.lt));
  c64 y[8];
  if constexpr (first) {
    // (i, k) <- point i + k 8 / R; a lane pair's input 2 j + o is its point j
#pragma unroll
    for (int i = 0; i < Q::NB; ++i)
#pragma unroll
      for (int k = 0; k < 8 / Q::NB; ++k) y[i * (8 / Q::NB) + k] = v[i + k * Q::NB];
  } else {
#pragma unroll
    for (int i = 0; i < Q::NB; ++i) {
      uint32_t base, bb;
      butterfly8<F, Q>(L, i, base, bb);
#pragma unroll
      for (int k = 0; k < 8 / Q::NB; ++k)
        y[i * (8 / Q::NB) + k] =
            x[lds_pad(in_point<F, Q>(base, bb, Q::p16 ? 2 * (uint32_t)k + L.o : (uint32_t)k))];
    }
  }
  // pre-multiplied twiddles, butterflies, post-multiplied ones
  if constexpr (Q::p16) {
    bf16_pair<F::fwd>(y, L.o);
    if constexpr (Q::post) {
      const c64 y0 = y[0];
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = cmul(w[j], y[j]);
      if (L.o == 0) y[0] = y0;  // output 0 is not multiplied
    }
  } else {
#pragma unroll
    for (int i = 0; i < Q::NB; ++i) {
      c64 *u = y + i * Q::R;
      if constexpr (Q::pre) {
#pragma unroll
        for (int k = 1; k < Q::R; ++k) u[k] = cmul(w[i * (Q::R - 1) + k - 1], u[k]);
      }
      butterfly<Q::R, F::fwd>(u);
      if constexpr (Q::post) {
#pragma unroll
        for (int k = 1; k < Q::R; ++k) u[k] = cmul(w[i * (Q::R - 1) + k - 1], u[k]);
      }
    }
  }
  sched_fence();
  if constexpr (last) {
#pragma unroll
    for (int i = 0; i < Q::NB; ++i)
#pragma unroll
      for (int k = 0; k < 8 / Q::NB; ++k) v[i + k * Q::NB] = y[i * (8 / Q::NB) + k];
  } else {
    c64 wn[8];
    if constexpr (!LATE) twiddles8<F, PI + 1>(L, pass_opaque(tw), wn);
    // every reader of the exchange's previous contents is done
    if constexpr (!first) {
      if constexpr (wave_in) wave_lds_fence();
      else __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < Q::NB; ++i) {
      uint32_t base, bb;
      butterfly8<F, Q>(L, i, base, bb);
#pragma unroll
      for (int k = 0; k < 8 / Q::NB; ++k)
        x[lds_pad(out_point<F, Q>(base, bb, Q::p16 ? pair_out(L, k) : (uint32_t)k))] =
            y[i * (8 / Q::NB) + k];
    }
    if constexpr (LATE) {
      sched_fence();
      twiddles8<F, PI + 1>(Lane8<F>(launder_u32(L0.lt)), pass_opaque(tw), wn);
    }
    constexpr bool wave_out = !Q::depth && !Pass8<F, PI + 1>::depth && F::TC <= 64;
    if constexpr (wave_out) wave_lds_fence();
    else __syncthreads();
    passes8<F, PI + 1, LATE>(v, wn, x, L0, tw);
  }
}

// point (of the transform) that v[m] of a thread holds on the side of pass PI
// (0: inputs of the whole transform, npass - 1: its outputs)
template <class F, int PI>
__device__ __forceinline__ uint32_t linear8(const Lane8<F> &L, uint32_t m) {
  using Q = Pass8<F, PI>;
  if constexpr (Q::depth) return L.lt + F::T * m;
  else if constexpr (F::pair) return L.base + L.bb + F::b / 16 * (2 * m + L.o);
  else return L.base + L.lc + F::TC * m;
}

}  // namespace cfft_dev
