// Shape-specialised forward kernels of shapes [36, 50) of the shape table (phs_shapes.h);
// one translation unit per range so that they compile in parallel.  Trees of five and six
// final-state particles: one-pass (one workgroup per sub-tile) and looping (persistent grids)
// variants for the 64-thread workgroups their launches take, at the compiler's register budget; other
// workgroup sizes run a looping variant with a run-time size.
#include "phs_forward.h"

namespace gphs {
namespace fwd {

namespace {

template <int SID>
FwdKernel pick_one(int block, bool* one) {
  static_assert(kShapes[SID].n_out > 4, "trees of five and six final-state particles");
  if (*one && block == 64) return shape_kernel<SID, 0, 64, true>();
  *one = false;
  return block == 64 ? shape_kernel<SID, 0, 64>() : shape_kernel<SID, 0, 0>();
}

template <int... S>
FwdKernel pick_seq(int sid, int block, bool* one, std::integer_sequence<int, S...>) {
  FwdKernel k = nullptr;
  (void)((sid == 36 + S ? (k = pick_one<36 + S>(block, one), true) : false) || ...);
  return k;
}

}  // namespace

FwdKernel pick_shape_36_50(int sid, int, int block, bool* one) {
  static_assert(50 <= kNumShapes, "shape range");
  return pick_seq(sid, block, one, std::make_integer_sequence<int, 14>{});
}

}  // namespace fwd
}  // namespace gphs
