// serve_overlap.hpp -- whether the requests of a device batch overwrite each
// other's inputs.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <utility>
#include <vector>

namespace cfft_internal {

// in[i], out[i]: addresses of request i's `bytes`-long buffers.  True if the
// output of a request overlaps the input of another one; a request's own input
// does not count.  O(m log m): each output looks up its neighbours among the
// sorted inputs and stops at the first that is not its own.
inline bool outputs_meet_other_inputs(const std::vector<uint64_t> &in,
                                      const std::vector<uint64_t> &out, uint64_t bytes) {
  std::vector<std::pair<uint64_t, size_t>> at(in.size());
  for (size_t i = 0; i < in.size(); ++i) at[i] = {in[i], i};
  std::sort(at.begin(), at.end());
  for (size_t i = 0; i < out.size(); ++i) {
    // the inputs that start less than `bytes` before or after out[i]
    const uint64_t first = out[i] < bytes ? 0 : out[i] - bytes + 1;
    for (auto p = std::lower_bound(at.begin(), at.end(), std::make_pair(first, (size_t)0));
         p != at.end() && p->first < out[i] + bytes; ++p)
      if (p->second != i) return true;
  }
  return false;
}

}  // namespace cfft_internal
