// The inverse kernel of the trees of six final-state particles, specialised per tree shape.
#include "phs_inverse.h"

namespace gphs {
namespace inv {

SharedKernel shared_kernel_6() { return inverse_kernel_shared<false, 6, false, 2>; }

}  // namespace inv
}  // namespace gphs
