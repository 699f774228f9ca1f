// Shape-specialised forward kernels for per-event beam energies, shapes [0, 8) of the shape
// table (the trees of 2-4 final-state particles): each event's sqrt(s), lab boost and
// sqrt(s)-dependent map constants formed in the kernel, as in the generic kernel's per-event
// variant, with the walk unrolled for the shape.  One-pass variants (one workgroup per sub-tile)
// for workgroups of 64, 128 and 256 threads at the compiler's register budget, a one-pass kernel of
// all the shapes (128 VGPRs, four waves per SIMD; 1e6 events of 2->4 46 us, 53 while the maps' constants
// went through scratch memory and a branch's were loaded where they are used), and looping ones (persistent grids, other workgroup sizes) at
// the compiler's budget or one for 3 waves per SIMD (asked for 4 or 5, the kernel takes 3).
// Larger trees with per-event beams run the generic kernel.
#include "phs_forward.h"

namespace gphs {
namespace fwd {

namespace {

template <int SID, int BLK>
FwdKernel pick_wpe(int wpe) {
  return wpe >= 3 ? shape_kernel<SID, 3, BLK, false, true>() : shape_kernel<SID, 0, BLK, false, true>();
}

template <int SID>
FwdKernel pick_one(int wpe, int block, bool* one) {
  static_assert(kShapes[SID].n_out <= 4, "per-event beam shape kernels cover trees of up to four particles");
  if (*one) {
    if (block == 64) return shape_kernel<SID, 0, 64, true, true>();
    if (block == 128) return shape_kernel<SID, 0, 128, true, true>();
    if (block == 256) return shape_kernel<SID, 0, 256, true, true>();
  }
  *one = false;
  if (block == 64) return pick_wpe<SID, 64>(wpe);
  if (block == 128) return pick_wpe<SID, 128>(wpe);
  if (block == 256) return pick_wpe<SID, 256>(wpe);
  return pick_wpe<SID, 0>(wpe);
}

template <int... S>
FwdKernel pick_seq(int sid, int wpe, int block, bool* one, std::integer_sequence<int, S...>) {
  FwdKernel k = nullptr;
  (void)((sid == S ? (k = pick_one<S>(wpe, block, one), true) : false) || ...);
  return k;
}

}  // namespace

FwdKernel pick_shape_pev_0_8(int sid, int wpe, int block, bool* one) {
  return pick_seq(sid, wpe, block, one, std::make_integer_sequence<int, kPevShapes>{});
}

FwdKernel pick_shapes_pev_0(int block) {
  if (block == 64) return forward_shapes_kernel<0, kPevShapes, 3, true, 64>;
  if (block == 128) return forward_shapes_kernel<0, kPevShapes, 3, true, 128>;
  if (block == 256) return forward_shapes_kernel<0, kPevShapes, 3, true, 256>;
  return nullptr;
}

}  // namespace fwd
}  // namespace gphs
