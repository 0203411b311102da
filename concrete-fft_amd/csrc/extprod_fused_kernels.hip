// extprod_fused_kernels.hip -- the external product (GGSW (x) GLWE) in one
// launch on Dif16 plans with n = 512 (base 512), 1024 and 2048 (base 1024).
//
// One 8-wave workgroup takes P GLWEs through all of it, so no spectrum
// leaves the CU: a round transforms 8 units (16 at n = 512, two per wave),
// each unit one base transform of a digit polynomial, and leaves the spectra
// in the waves' exchange buffers; all 512 threads then add key * spectrum of
// the round's rows to the sums of their n / 512 points (P x K1 columns in
// registers, rows in ascending order); after the last round the sums go back
// through the buffers and the first P * K1 units run the columns' inverse
// transforms and store.  At n = 2048 a polynomial is two units, its two
// 1024-point chunks: the plan's radix-2 depth butterflies swap their
// partners through the two waves' buffers.
//
// Operations and their order are the split kernels' (extprod_kernels.hip),
// and so the bits: the same digits, twist, transforms, cmul(key, spectrum)
// summed from zero in ascending row order, untwist and rounding.
//
// What bounds it: two waves per SIMD (a transform's registers, and 16 KB of
// exchange buffer per wave) that neither the FP64 units nor LDS wait for
// alone; a round of eight 1024-point transforms, digits and sums takes 8.5-9
// us, in which by the counters (N = 4096 x 512) the SIMDs issue VALU instructions
// for 44 % of the time and LDS is busy for 27 %, while a wave waits for data or
// barriers 41 % of its time (one GLWE of N = 2048: 30, 19 and 53 %).  With one GLWE
// on a CU its key points come through that CU's one L2 port (196 KB at N =
// 2048, k1 = 2, l = 3: 2.6 of 13 us), hence their early request.  Measured
// against the split form (two launches, spectra through HBM), us per call,
// k1 = 2, l = 3: N = 1024 18.7 -> 10.2 (1 GLWE), 31.6 -> 11.7 (256), 75.5 ->
// 40.0 (2000); N = 2048 19.9 -> 13.1, 37.8 -> 15.3, 127 -> 71; N = 4096 34.2
// -> 24.1, 54.6 -> 28.6, 285 -> 167.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "extprod_rows.hpp"
#include "gadget.hpp"
#include "launch.hpp"
#include "lds_attr.hpp"
#include "r16s_exec.hpp"

using namespace cfft_dev;
using cfft_launch::dc64;

namespace {

constexpr uint32_t kFWaves = 8;

template <int LOG2N>
struct FGeom {
  static constexpr int LB = LOG2N == 11 ? 10 : LOG2N;  // base transform
  static constexpr uint32_t n = 1u << LOG2N, nb = 1u << LB;
  static constexpr uint32_t CH = n / nb;         // chunks (units) per polynomial
  static constexpr uint32_t T = nb / 16;         // lanes per unit
  static constexpr uint32_t G = 64 / T;          // units per wave
  static constexpr uint32_t U = kFWaves * G;     // units in flight
  static constexpr uint32_t PB = nb / (64 * kFWaves);  // points per thread and chunk
  // the twist table, or at n = 2048 its entries 0 ... 1024 (twist_point)
  static constexpr uint32_t zw = n <= 1024 ? n : 1025;
  static constexpr uint32_t head = kSTw + zw;
  static constexpr size_t lds = (size_t)(head + U * nb) * sizeof(c64);
  static_assert(lds <= 160 * 1024, "one workgroup per CU");
};

// Twist factor of point i of chunk ch.  zeta_j = exp(i pi j / 2n), so that at
// n = 2048 the second chunk's factors are the first one's mirrored at j =
// 1024 with re and im exchanged (the plan checks its table for that, entry
// for entry); j = 1024 itself is stored.
template <uint32_t CH>
__device__ __forceinline__ c64 twist_point(const c64 *ltz, uint32_t ch, uint32_t i) {
  if constexpr (CH == 1) {
    return ltz[i];
  } else {
    const c64 z = ltz[ch ? 1024 - i : i];
    const bool swap = ch && i;
    return swap ? mk(z.im, z.re) : z;
  }
}

// A buffer descriptor over `points` points: loads take a 32-bit offset per lane
// and a scalar one in place of a 64-bit address.  Every load stays inside the
// `points`.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t point_buffer(const c64 *base, uint32_t points) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<c64 *>(base), 0, (int)(points * 16u),
                                           0x00027000);
}
__device__ __forceinline__ c64 load_point(__amdgpu_buffer_rsrc_t r, uint32_t point,
                                          uint32_t from = 0) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const u32x4 w = __builtin_amdgcn_raw_buffer_load_b128(r, (int)(point * 16u), (int)(from * 16u), 0);
  return mk(__builtin_bit_cast(double, ((uint64_t)w.y << 32) | w.x),
            __builtin_bit_cast(double, ((uint64_t)w.w << 32) | w.z));
}

// NARROW: the digits need the coefficients' high words only (gadget32_digit),
// which are the words then loaded: half the registers and loaded bytes.
// glwe_tab / out_tab (optional): one address per GLWE in place of the
// contiguous glwe / out.
template <int LOG2N, int K1, int P, bool NARROW>
__global__ void __launch_bounds__(64 * kFWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_extprod_fused(const c64 *__restrict__ keyf, const uint64_t *glwe, const uint64_t *glwe_tab,
                uint64_t *out, const uint64_t *out_tab, uint64_t batch, uint32_t levels,
                uint32_t base_log, const c64 *__restrict__ tw, const c64 *__restrict__ tw_blk,
                const c64 *__restrict__ twist) {
  using F = FGeom<LOG2N>;
  using S = R16<F::LB>;
  constexpr uint32_t n = F::n, T = F::T, CH = F::CH;
  constexpr uint32_t RG = rows_per_round(F::U, CH, P);
  static_assert(RG >= 1 && P * K1 * CH <= F::U, "the columns must fit the units");
  extern __shared__ c64 smem[];
  c64 *ltw = smem, *ltz = smem + kSTw, *xs = smem + F::head;
  const uint32_t rows = K1 * levels;
  const uint32_t tid = threadIdx.x;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t u = wave * F::G + (tid & 63u) / T;  // this lane's unit
  c64 *x = xs + u * F::nb;
  const c64 *xp = xs + (u ^ 1u) * F::nb;  // the other chunk's unit (n = 2048)
  const uint32_t ch = u % CH;

  // the coefficients of unit u's row of the round at r0, for the GLWEs from
  // g0: always 32 loads (the compiler would wait at a branch), from the
  // L2-resident twist table where the unit has no row
  using Word = typename std::conditional<NARROW, uint32_t, uint64_t>::type;
  Word w[32];
  auto fetch = [&](uint64_t g0, uint32_t r0) {
    const uint32_t row = r0 + (u / CH) % RG;
    const uint64_t gq = g0 + u / (CH * RG);
    const uint32_t l = launder_u32(tid) & (T - 1);
    const uint64_t *src = reinterpret_cast<const uint64_t *>(twist);
    if (row < rows && gq < batch)
      src = (glwe_tab ? reinterpret_cast<const uint64_t *>(glwe_tab[gq])
                      : glwe + gq * (K1 * 2ull * n)) +
            (row / levels) * 2ull * n;
    src += ch * 1024 + l;
    const Word *sw = reinterpret_cast<const Word *>(src) + (NARROW ? 1 : 0);
    constexpr uint32_t st = sizeof(uint64_t) / sizeof(Word);
#pragma unroll
    for (uint32_t m = 0; m < 16; ++m) {
      w[2 * m] = ld_stream(&sw[st * (T * m)]);
      w[2 * m + 1] = ld_stream(&sw[st * (T * m + n)]);
    }
  };

  uint64_t g0 = (uint64_t)blockIdx.x * P;
  {
    // the twiddle block's loads, then the first coefficients', in flight together
    // (rows k = 1 ... 15 start at 64 and at 1024 + 4 in the plan's block)
    static_assert(kSTw > 512 && kSTw <= 1024, "two entries per thread");
    const auto blk = point_buffer(tw_blk, 16 * 64 + 16 * 4), zt = point_buffer(twist, n);
    auto entry = [&](uint32_t i) { return load_point(blk, r16s_block_index(i)); };
    const c64 t0 = entry(tid), t1 = entry(tid + 512);
    // (n = 512: one twist entry per thread; n = 2048: entry 1024 as well; entry 0
    // where there is none)
    const c64 z0 = load_point(zt, tid), z1 = load_point(zt, F::zw > 512 ? tid + 512 : 0);
    const c64 z2 = load_point(zt, F::zw > 1024 ? 1024 : 0);
    fetch(g0, 0);
    sched_fence();
    ltw[tid] = t0;
    if (tid + 512 < kSTw) ltw[tid + 512] = t1;
    ltz[tid] = z0;
    if constexpr (F::zw > 512) ltz[tid + 512] = z1;
    if (F::zw > 1024 && tid == 0) ltz[1024] = z2;
  }
  __syncthreads();

  for (; g0 < batch; g0 += (uint64_t)gridDim.x * P) {
    c64 acc[P][CH * F::PB][K1];
#pragma unroll
    for (int g = 0; g < P; ++g)
#pragma unroll
      for (uint32_t e = 0; e < CH * F::PB; ++e)
#pragma unroll
        for (int c = 0; c < K1; ++c) acc[g][e][c] = mk(0.0, 0.0);

    for (uint32_t r0 = 0; r0 < rows; r0 += RG) {
      // ---- forward: unit u transforms row r0 + (u / CH) % RG of GLWE g0 + u / (CH RG) ----
      const uint32_t row = r0 + (u / CH) % RG;
      // a wave without a row skips the work, not the barriers
      const bool on = __ballot(row < rows && g0 + u / (CH * RG) < batch) != 0;
      const uint32_t l = launder_u32(tid) & (T - 1);
      c64 v[16];
      if (on) {
        auto twisted = [&](auto digit) {
#pragma unroll
          for (uint32_t m = 0; m < 16; ++m) {
            v[m] = cmul(twist_point<CH>(ltz, ch, l + T * m),
                        mk((double)digit(w[2 * m]), (double)digit(w[2 * m + 1])));
            if (CH == 2 && (m & 3) == 3) sched_fence();
          }
        };
        if constexpr (NARROW) {
          const Gadget32 gd = gadget32_of(row % levels, levels, base_log);
          twisted([&](uint32_t h) { return gadget32_digit(gd, h); });
        } else {
          const Gadget gd = gadget_of(row % levels, levels, base_log);
          twisted([&](uint64_t x) { return (int32_t)gadget_digit(gd, x); });
        }
      }
      if constexpr (CH == 2) {
        // DEPTH_FWD radix 2: (a + b) to chunk 0, (a - b) T[j] to chunk 1
        if (on) {
#pragma unroll
          for (uint32_t m = 0; m < 16; ++m) x[m * 64 + l] = v[m];
        }
        __syncthreads();
        if (on) {
          if (ch == 0) {
#pragma unroll
            for (uint32_t m = 0; m < 16; ++m) v[m] = cadd(v[m], xp[m * 64 + l]);
          } else {
            const c64 *tj = launder(tw) + l;
            c64 z[2][4];
#pragma unroll
            for (uint32_t m = 0; m < 4; ++m) z[0][m] = tj[64 * m];
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
              if (k < 3) {
#pragma unroll
                for (uint32_t m = 0; m < 4; ++m) z[(k + 1) & 1][m] = tj[64 * (4 * k + 4 + m)];
              }
              sched_fence();
#pragma unroll
              for (uint32_t m = 0; m < 4; ++m)
                v[4 * k + m] = cmul(z[k & 1][m], csub(xp[(4 * k + m) * 64 + l], v[4 * k + m]));
              sched_fence();
            }
          }
        }
        __syncthreads();  // the partner has read this buffer
      }
      // the key points of the multiply-accumulate, KR rows requested together;
      // the first ones before the transform that hides them where they fit
      // beside it and the sums (spilling cost more)
      constexpr uint32_t PT = CH * F::PB;
      constexpr uint32_t KR = rows_requested(CH, PT, K1, RG);
      // and the next coefficients before the sums where they fit beside the key
      // points, after them elsewhere.  Requested before them by every form, 64-bit
      // words spilled 28-196 bytes per lane at k1 = 3 and 4, 32-bit ones 68 at N =
      // 2048, k1 = 4, P = 2 (us, so and now, N = 2048: k1 = 3, 1 level of 32 bits,
      // 600 GLWEs 46.2 / 37.0; 4 levels of 10, 1100 162.9 / 110.7; k1 = 4, 8 levels
      // of 8, 257 160.9 / 101.5; 3 levels of 8, 600 113.4 / 83.6).
      constexpr uint32_t KREGS = 4 * (P + KR) * PT * K1;  // key points and sums
      constexpr bool EARLY = CH == 1 && P <= 2 && KREGS <= 120;
      constexpr bool AHEAD = NARROW ? KREGS <= 144 : CH == 1 && KREGS <= (PT == 1 ? 108 : 112);
      const uint32_t nr = rows - r0 < RG ? rows - r0 : RG;
      c64 kv[KR][PT][K1];
      auto key_rows = [&](uint32_t rr) {
        const uint32_t t = launder_u32(tid);
        uint32_t q[PT];
#pragma unroll
        for (uint32_t e = 0; e < PT; ++e) {
          const uint32_t idx = t + 64 * kFWaves * (e % F::PB);
          q[e] = (e / F::PB) * 1024 + (idx & (T - 1)) + T * S::end_m(idx / T);
        }
#pragma unroll
        for (uint32_t i = 0; i < KR; ++i) {
          const auto key = point_buffer(keyf + (uint64_t)key_row(r0, rr, i, rows) * (K1 * n),
                                        K1 * n);
#pragma unroll
          for (uint32_t e = 0; e < PT; ++e)
#pragma unroll
            for (int c = 0; c < K1; ++c) kv[i][e][c] = load_point(key, q[e], c * n);
        }
      };
      if constexpr (EARLY) {
        key_rows(0);
        sched_fence();
      }
      if (on) {
        r16s_transform<F::LB, true, 1>(v, v, x, l, ltw);
        wave_lds_fence();
#pragma unroll
        for (uint32_t s = 0; s < 16; ++s) x[s * T + l] = v[s];
      }
      sched_fence();
      // ---- multiply-accumulate: this thread's points of every unit's buffer ----
      if constexpr (!EARLY) key_rows(0);
      const bool more = r0 + RG < rows;
      auto fetch_next = [&]() {
        fetch(more ? g0 : g0 + (uint64_t)gridDim.x * P, more ? r0 + RG : 0);
      };
      if constexpr (AHEAD) fetch_next();
      sched_fence();
      __syncthreads();
      const uint32_t t = launder_u32(tid);
      for (uint32_t rr = 0; rr < (KR < RG ? nr : 1); rr += KR) {
        if (KR < RG && rr) key_rows(rr);
#pragma unroll
        for (uint32_t i = 0; i < KR; ++i) {
          if (rr + i >= nr) break;
          sched_fence();
#pragma unroll
          for (uint32_t e = 0; e < PT; ++e) {
            const uint32_t idx = t + 64 * kFWaves * (e % F::PB);
#pragma unroll
            for (int g = 0; g < P; ++g) {
              const c64 sv = xs[((g * RG + rr + i) * CH + e / F::PB) * F::nb + idx];
#pragma unroll
              for (int c = 0; c < K1; ++c)
                acc[g][e][c] = cadd(acc[g][e][c], cmul(kv[i][e][c], sv));
            }
          }
        }
      }
      if constexpr (!AHEAD) {
        sched_fence();
        fetch_next();
      }
      __syncthreads();  // every spectrum of the round read
    }
    // ---- columns: sums to unit (g, c, chunk)'s buffer, in point order ----
    {
      const uint32_t t = launder_u32(tid);
#pragma unroll
      for (uint32_t e = 0; e < CH * F::PB; ++e) {
        const uint32_t idx = t + 64 * kFWaves * (e % F::PB), c2 = e / F::PB;
        const uint32_t q = (idx & (T - 1)) + T * S::end_m(idx / T);
#pragma unroll
        for (int g = 0; g < P; ++g)
#pragma unroll
          for (int c = 0; c < K1; ++c) xs[((g * K1 + c) * CH + c2) * F::nb + q] = acc[g][e][c];
      }
    }
    __syncthreads();
    const uint32_t l = launder_u32(tid) & (T - 1);
    // unit u has GLWE u / (CH K1)'s column; waves without one skip the transform
    const bool busy = __ballot(u < P * K1 * CH && g0 + u / (CH * K1) < batch) != 0;
    c64 v[16];
    if (busy) {
#pragma unroll
      for (uint32_t m = 0; m < 16; ++m) v[m] = x[l + T * m];
      r16s_transform<F::LB, false, 1>(v, v, x, l, ltw);
    }
    // untwist = conj(twist) / n (an exact scaling: the plan's untwist table)
    auto put = [&](uint64_t *o, uint32_t c2, uint32_t i, c64 y) {
      const c64 z = twist_point<CH>(ltz, c2, i);
      const c64 r = cmul(mk(z.re * (1.0 / n), (-z.im) * (1.0 / n)), y);
      st_stream(from_torus(r.re), &o[c2 * 1024 + i]);
      st_stream(from_torus(r.im), &o[c2 * 1024 + i + n]);
    };
    auto column = [&](uint64_t q, uint32_t c) {
      return (out_tab ? reinterpret_cast<uint64_t *>(out_tab[q]) : out + q * (K1 * 2ull * n)) +
             c * 2ull * n;
    };
    // every wave stores a share of the columns: the depth butterflies meet in
    // LDS anyway, and with half of the units idle one wave's rounding of a
    // whole column took longer than its transform
    if (busy) {
      wave_lds_fence();
#pragma unroll
      for (uint32_t s = 0; s < 16; ++s) x[s * T + l] = v[s];
    }
    __syncthreads();
    const uint32_t t = launder_u32(tid);
#pragma unroll
    for (uint32_t e = 0; e < F::PB; ++e) {
      const uint32_t idx = t + 64 * kFWaves * e;
      const uint32_t q = (idx & (T - 1)) + T * S::end_m(idx / T);
      const c64 zq = CH == 2 ? tw[q] : mk(0.0, 0.0);
#pragma unroll
      for (int g = 0; g < P; ++g) {
        if (g0 + g >= batch) break;
#pragma unroll
        for (int c = 0; c < K1; ++c) {
          uint64_t *o = column(g0 + g, c);
          const c64 *y = xs + (g * K1 + c) * CH * F::nb + idx;
          if constexpr (CH == 1) {
            put(o, 0, q, y[0]);
          } else {
            // DEPTH_INV radix 2: conj(T[q]) on chunk 1's point, then the butterfly
            const c64 b = cmul(conj(zq), y[F::nb]);
            put(o, 0, q, cadd(y[0], b));
            put(o, 1, q, csub(y[0], b));
          }
        }
      }
    }
    __syncthreads();  // the buffers are read
  }
}

struct FArgs {
  const c64 *keyf;
  const uint64_t *glwe, *glwe_tab;
  uint64_t *out;
  const uint64_t *out_tab;
  uint64_t batch;
  uint32_t levels, base_log;
  const c64 *tw, *tw_blk, *twist;
};

template <int LOG2N, int K1, int P, bool NARROW>
hipError_t launch_fused_n(const FArgs &a, int cus, hipStream_t s) {
  using F = FGeom<LOG2N>;
  const void *k = reinterpret_cast<const void *>(k_extprod_fused<LOG2N, K1, P, NARROW>);
  const hipError_t e = cfft_launch::ensure_lds(k, F::lds);
  if (e != hipSuccess) return e;
  const uint64_t groups = (a.batch + P - 1) / P;
  const uint32_t grid = (uint32_t)(groups < (uint64_t)cus ? groups : (uint64_t)cus);
  hipLaunchKernelGGL((k_extprod_fused<LOG2N, K1, P, NARROW>), dim3(grid), dim3(64 * kFWaves), F::lds, s,
                     a.keyf, a.glwe, a.glwe_tab, a.out, a.out_tab, a.batch, a.levels, a.base_log,
                     a.tw, a.tw_blk, a.twist);
  return hipGetLastError();
}

template <int LOG2N, int K1, int P>
hipError_t launch_fused(const FArgs &a, int cus, hipStream_t s) {
  return a.levels * a.base_log <= 31 ? launch_fused_n<LOG2N, K1, P, true>(a, cus, s)
                                     : launch_fused_n<LOG2N, K1, P, false>(a, cus, s);
}

// GLWEs per workgroup: the fewest rounds, inverse included, over the
// workgroups' passes (one workgroup per CU at a time); fewer GLWEs on a tie
template <int LOG2N, int K1>
hipError_t launch_fused_p(const FArgs &a, hipStream_t s) {
  using F = FGeom<LOG2N>;
  constexpr int PMAX = LOG2N == 9 && K1 > 2 ? 2 : (int)(F::U / (F::CH * K1));
  int cus = 0;
  const hipError_t e = cfft_launch::cu_count(&cus);
  if (e != hipSuccess) return e;
  auto cost = [&](uint64_t p) -> uint64_t {
    if (p > (uint64_t)PMAX) return ~(uint64_t)0;
    const uint64_t groups = (a.batch + p - 1) / p, rg = F::U / F::CH / p;
    const uint64_t passes = (groups + (uint64_t)cus - 1) / (uint64_t)cus;
    return passes * ((K1 * (uint64_t)a.levels + rg - 1) / rg + 1);
  };
  const uint64_t c1 = cost(1), c2 = cost(2), c4 = cost(4);
  if constexpr (PMAX >= 4)
    if (c4 < c1 && c4 < c2) return launch_fused<LOG2N, K1, 4>(a, cus, s);
  if constexpr (PMAX >= 2)
    if (c2 < c1) return launch_fused<LOG2N, K1, 2>(a, cus, s);
  return launch_fused<LOG2N, K1, 1>(a, cus, s);
}

template <int LOG2N>
hipError_t launch_fused_k(const FArgs &a, uint32_t k1, hipStream_t s) {
  switch (k1) {
    case 2: return launch_fused_p<LOG2N, 2>(a, s);
    case 3: return launch_fused_p<LOG2N, 3>(a, s);
    case 4: return launch_fused_p<LOG2N, 4>(a, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

namespace cfft_launch {

hipError_t external_product_fused(uint32_t log2n, const dc64 *keyf, const uint64_t *glwe,
                                  const uint64_t *glwe_tab, uint64_t *out,
                                  const uint64_t *out_tab, uint64_t batch, uint32_t k1,
                                  uint32_t levels, uint32_t base_log, const dc64 *tw,
                                  const dc64 *tw_blk, const dc64 *twist, hipStream_t s) {
  if (batch == 0) return hipSuccess;
  const FArgs a{reinterpret_cast<const c64 *>(keyf), glwe, glwe_tab, out, out_tab, batch, levels,
                base_log, reinterpret_cast<const c64 *>(tw),
                reinterpret_cast<const c64 *>(tw_blk), reinterpret_cast<const c64 *>(twist)};
  switch (log2n) {
    case 9: return launch_fused_k<9>(a, k1, s);
    case 10: return launch_fused_k<10>(a, k1, s);
    case 11: return launch_fused_k<11>(a, k1, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace cfft_launch
