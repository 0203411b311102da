// gadget.hpp -- the external product's gadget decomposition on the device:
// round x to the nearest multiple of 2^(64 - levels*base_log) (ties up), then
// balanced digits in [-2^(B-1), 2^(B-1)) from the least significant level up,
// carrying; level 0 is the most significant.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cfft_dev {

// One level of the gadget decomposition, without branches or loops: the
// balanced digits of the rounded value st (rep = levels * base_log bits) are
// the plain base-2^B digits of st + (half in every digit position), each
// minus half -- the carry loop of the decomposition done by one addition
// (the same digits; the wrap-around past rep bits is the top digit's carry,
// which the decomposition drops as well).
struct Gadget {
  uint32_t shift;   // 64 - rep: the rounding position (0: no rounding)
  uint32_t down;    // base_log * (levels - 1 - level): this level's digit position
  uint64_t keep;    // the low rep bits
  uint64_t offset;  // half in every digit position
  uint64_t mask;    // one digit
  int64_t half;
};

__device__ __forceinline__ Gadget gadget_of(uint32_t level, uint32_t levels, uint32_t base_log) {
  Gadget g;
  const uint32_t rep = levels * base_log;
  g.shift = 64 - rep;
  g.down = base_log * (levels - 1 - level);
  g.keep = rep < 64 ? ((uint64_t)1 << rep) - 1 : ~(uint64_t)0;
  g.mask = ((uint64_t)1 << base_log) - 1;
  g.half = (int64_t)1 << (base_log - 1);
  g.offset = 0;
  for (uint32_t i = 0; i < levels; ++i) g.offset = (g.offset << base_log) | (uint64_t)g.half;
  return g;
}

__device__ __forceinline__ int64_t gadget_digit(const Gadget &g, uint64_t x) {
  const uint64_t up = g.shift ? (x >> (g.shift - 1)) & 1u : 0;  // ties round up
  const uint64_t st = ((x >> g.shift) + up) & g.keep;
  return (int64_t)(((st + g.offset) >> g.down) & g.mask) - g.half;
}

// The same digit for rep = levels * base_log <= 31, from the high word of the
// coefficient alone and in 32-bit operations: with h = x >> 32 and s = 32 - rep
// >= 1, the rounded value is ((h >> (s - 1)) + 1) >> 1, and its digits are the
// bit fields of (h >> (s - 1)) + 1 + 2 offset from bit 1 up, each minus half
// (bits past rep, the top digit's carry, lie above every field).  5 operations
// and a conversion against about 20 in 64 bits.
struct Gadget32 {
  uint32_t shift;   // s - 1
  uint32_t add;     // 1 + 2 offset
  uint32_t down;    // this level's field
  uint32_t width;   // base_log
  uint32_t half;
};

__device__ __forceinline__ Gadget32 gadget32_of(uint32_t level, uint32_t levels,
                                                uint32_t base_log) {
  Gadget32 g;
  g.shift = 31 - levels * base_log;
  g.half = 1u << (base_log - 1);
  uint32_t offset = 0;
  for (uint32_t i = 0; i < levels; ++i) offset = (offset << base_log) | g.half;
  g.add = 1 + 2 * offset;
  g.down = base_log * (levels - 1 - level) + 1;
  g.width = base_log;
  return g;
}

__device__ __forceinline__ int32_t gadget32_digit(const Gadget32 &g, uint32_t h) {
  const uint32_t st = (h >> g.shift) + g.add;
  return (int32_t)(__builtin_amdgcn_ubfe(st, g.down, g.width) - g.half);
}

}  // namespace cfft_dev
