// Each line of the input is "bytes m in_0 out_0 ... in_{m-1} out_{m-1}"; prints
// 1 if an output overlaps another request's input (serve_overlap.hpp), else 0.
#include <cstdio>

#include "serve_overlap.hpp"

int main() {
  unsigned long long bytes, m;
  while (std::scanf("%llu %llu", &bytes, &m) == 2) {
    std::vector<uint64_t> in(m), out(m);
    for (size_t i = 0; i < m; ++i) {
      unsigned long long a, b;
      if (std::scanf("%llu %llu", &a, &b) != 2) return 1;
      in[i] = a;
      out[i] = b;
    }
    std::printf("%d\n", cfft_internal::outputs_meet_other_inputs(in, out, bytes) ? 1 : 0);
  }
  return 0;
}
