// launch_shape.h -- the launch shapes of the fused step that the autotuner
// tries (internal to the library; host code alone).
#pragma once

#include <algorithm>
#include <cstddef>
#include <utility>
#include <vector>

namespace colphys {

// (block, live levels of Thomas state in LDS) pairs that fit lds_max bytes
// with nq quantities a level: the shape that the handle has (which need not be
// one of the others, and would otherwise go untimed), then 64, 128 and 256
// threads with a range of levels.
inline std::vector<std::pair<int, int>> shape_candidates(int lds_max, size_t nq, int block, int levels) {
  std::vector<std::pair<int, int>> c{{block, levels}};
  for (int b : {64, 128, 256}) {
    const int most = (int)((size_t)lds_max / ((size_t)b * nq * 8));
    for (int m : {0, 4, 8, 12, 16, 24, 32}) {
      const std::pair<int, int> s{b, m};
      if (m <= most && std::find(c.begin(), c.end(), s) == c.end()) c.push_back(s);
    }
  }
  return c;
}

}  // namespace colphys
