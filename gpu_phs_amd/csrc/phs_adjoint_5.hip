// The adjoint of the trees of five final-state particles (shapes [8, 22)).
#include "phs_adjoint_shape.h"

namespace gphs {
namespace adj {

Kernel pick_5(int loss_mode) {
  static_assert(kShapes[8].n_out == 5 && kShapes[21].n_out == 5, "shape range");
  return loss_mode ? shapes_kernel<8, 22, 1, 2> : shapes_kernel<8, 22, 0, 2>;
}

}  // namespace adj
}  // namespace gphs
