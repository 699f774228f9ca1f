// Shape-specialised forward kernels of shapes [0, 8) of the shape table (phs_shapes.h);
// one translation unit per range so that they compile in parallel.  Trees of up to four
// final-state particles have one-pass variants (one workgroup per sub-tile) for workgroups of 64,
// 128 and 256 threads at the compiler's register budget, which is then within four waves per SIMD
// (90-118 VGPRs), looping ones (persistent grids) for every budget, a one-pass kernel of all the
// shapes, and for other workgroup sizes looping ones with a run-time size.
#include "phs_forward.h"

namespace gphs {
namespace fwd {

namespace {

template <int SID, int BLK>
FwdKernel pick_wpe(int wpe) {
  if (wpe == 3) return shape_kernel<SID, 3, BLK>();
  if (wpe == 4) return shape_kernel<SID, 4, BLK>();
  if (wpe == 5) return shape_kernel<SID, 5, BLK>();
  return shape_kernel<SID, 0, BLK>();
}

template <int SID>
FwdKernel pick_one(int wpe, int block, bool* one) {
  if (*one && wpe != 5) {
    if (block == 64) return shape_kernel<SID, 0, 64, true>();
    if (block == 128) return shape_kernel<SID, 0, 128, true>();
    if (block == 256) return shape_kernel<SID, 0, 256, true>();
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
  (void)((sid == 0 + S ? (k = pick_one<0 + S>(wpe, block, one), true) : false) || ...);
  return k;
}

}  // namespace

FwdKernel pick_shape_0_8(int sid, int wpe, int block, bool* one) {
  static_assert(8 <= kNumShapes, "shape range");
  return pick_seq(sid, wpe, block, one, std::make_integer_sequence<int, 8>{});
}

FwdKernel pick_shapes_0(int block) {
  if (block == 64) return forward_shapes_kernel<0, 8, 4, false, 64>;
  if (block == 128) return forward_shapes_kernel<0, 8, 4, false, 128>;
  if (block == 256) return forward_shapes_kernel<0, 8, 4, false, 256>;
  return nullptr;
}

}  // namespace fwd
}  // namespace gphs
