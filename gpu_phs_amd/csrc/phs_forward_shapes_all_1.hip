// The one-pass forward kernel of all the shapes of five final-state particles ([8, 22) of the shape
// table), the launch of every group of two or more of them unless merge_below is 0.
#include "phs_forward.h"

namespace gphs {
namespace fwd {

FwdKernel pick_shapes_1(int block) {
  static_assert(kShapes[8].n_out == 5 && kShapes[21].n_out == 5 && 22 <= kNumShapes, "shape range");
  return block == 64 ? forward_shapes_kernel<8, 22, 3, false, 64> : nullptr;
}

}  // namespace fwd
}  // namespace gphs
