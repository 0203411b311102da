// fixed8_fft.hip -- the transforms of fixed8_fft.hpp for every algo's plans with
// n = 64 ... 1024 on base n, and n = 1024 on base 512.
#include "fixed8_fft.hpp"

namespace {

struct Call {
  const Program &prog;
  c64 *d;
  uint64_t ntrans, stride;
  const c64 *t;
  cfft_launch::HostDone *done;
  hipStream_t s;
  hipError_t *e;
};

template <int ALGO, int LOG2N, int LOG2BN>
bool one(const Call &c) {
  return fixed8_fft_try<ALGO, LOG2N, LOG2BN>(c.prog, c.d, c.ntrans, c.stride, c.t, c.done, c.s,
                                             c.e);
}
template <int LOG2N, int LOG2BN>
bool any(const Call &c) {
  return one<0, LOG2N, LOG2BN>(c) || one<1, LOG2N, LOG2BN>(c) || one<2, LOG2N, LOG2BN>(c) ||
         one<3, LOG2N, LOG2BN>(c) || one<4, LOG2N, LOG2BN>(c) || one<5, LOG2N, LOG2BN>(c) ||
         one<6, LOG2N, LOG2BN>(c) || one<7, LOG2N, LOG2BN>(c);
}

}  // namespace

namespace cfft_launch {

bool fft_fixed8(const cfft_prog::Program &prog, dc64 *data, uint64_t ntrans, uint64_t stride,
                const dc64 *tw, HostDone *done, hipStream_t s, hipError_t *e) {
  const Call c{prog, reinterpret_cast<c64 *>(data), ntrans, stride,
               reinterpret_cast<const c64 *>(tw), done, s, e};
  switch (prog.log2n) {
    case 6: return any<6, 6>(c);
    case 7: return any<7, 7>(c);
    case 8: return any<8, 8>(c);
    case 9: return any<9, 9>(c);
    case 10: return any<10, 10>(c) || any<10, 9>(c);
    default: return false;
  }
}

}  // namespace cfft_launch
