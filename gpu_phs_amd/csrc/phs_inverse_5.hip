// The inverse kernel of the trees of five final-state particles, specialised per tree shape.
#include "phs_inverse.h"

namespace gphs {
namespace inv {

SharedKernel shared_kernel_5() { return inverse_kernel_shared<false, 5, false, 2>; }

}  // namespace inv
}  // namespace gphs
