// The adjoint of the trees of six final-state particles (shapes [22, 64)), the built-in loss (loss mode 1).
#include "phs_adjoint_shape.h"

namespace gphs {
namespace adj {

Kernel pick_6_1() {
  static_assert(kShapes[22].n_out == 6 && kShapes[63].n_out == 6 && 64 == kNumShapes, "shape range");
  return shapes_kernel<22, 64, 1, 2>;
}

}  // namespace adj
}  // namespace gphs
