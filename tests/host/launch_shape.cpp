// C entry over colphys::shape_candidates for tests/test_launch_shape.py.
#include "../../roundabout_amd/csrc/launch_shape.h"

extern "C" int ls_candidates(int lds_max, int nq, int block, int levels, int* out, int cap) {
  const auto c = colphys::shape_candidates(lds_max, (size_t)nq, block, levels);
  for (size_t i = 0; i < c.size() && (int)i < cap; ++i) {
    out[2 * i] = c[i].first;
    out[2 * i + 1] = c[i].second;
  }
  return (int)c.size();
}
