// The one-pass forward kernel of all the shapes of six final-state particles ([22, 64) of the shape
// table), the launch of every group of two or more of them unless merge_below is 0.
#include "phs_forward.h"

namespace gphs {
namespace fwd {

FwdKernel pick_shapes_2(int block) {
  static_assert(kShapes[22].n_out == 6 && kShapes[63].n_out == 6 && 64 <= kNumShapes, "shape range");
  return block == 64 ? forward_shapes_kernel<22, 64, 3, false, 64> : nullptr;
}

}  // namespace fwd
}  // namespace gphs
