// Adjoint kernels: per event, the forward pass with a tape, then the reverse sweep (phs_adjoint.h; for a
// tree shape with fixed beams phs_adjoint_shape.h).  One workgroup = one wavefront = 64 events of one tile;
// the tape, the stash and the lane's (M, Gamma) accumulators live in LDS, lane-strided so every access is
// conflict-free.  The parameter adjoints of a tile are reduced across the wavefront and written as one
// partial per unit; a second kernel sums the partials of each channel in a fixed order, so results do not
// depend on scheduling.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <utility>

#include "phs_adjoint.h"
#include "phs_adjoint_shape.h"
#include "phs_kernels.h"
#include "phs_shapes.h"

namespace gphs {

namespace {

using adj::wave_sums;

// COMPACT: the stash keeps 15 of its 19 words (only the root defers; phs_adjoint.h).  Word w
// of a lane is at base[w * 64] (one wavefront per workgroup: consecutive lanes, consecutive
// words).
template <bool COMPACT>
struct LdsStore {
  static constexpr int stride = 64;
  double* base;
  int off_in, off_st;
  __device__ double& T(int node, int k) { return base[(node * 6 + k) * stride]; }
  __device__ double& in(int node, int k) { return base[(off_in + node * 2 + k) * stride]; }
  __device__ __forceinline__ void st_put(int level, int k, double v) {
    if constexpr (COMPACT) {
      const int c = compact_stash_slot(k);
      if (c >= 0) base[(off_st + level * kAdjCompactStashWords + c) * stride] = v;
    } else {
      base[(off_st + level * kAdjStashWords + k) * stride] = v;
    }
  }
  __device__ __forceinline__ double st_get(int level, int k) const {
    if constexpr (COMPACT) {
      const int c = compact_stash_slot(k);
      return c >= 0 ? base[(off_st + level * kAdjCompactStashWords + c) * stride] : 0.0;
    } else {
      return base[(off_st + level * kAdjStashWords + k) * stride];
    }
  }
};

struct LdsAcc {
  double* base;
  __device__ double& operator[](int i) { return base[i * 64]; }
};

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

constexpr int kAdjXReg = 8;             // n_x <= 8 <=> n_out <= 4
constexpr int kSmallParams = 2 * 3;     // (M, Gamma) of the 3 branches of an n_out = 4 tree

// One 64-event unit of the adjoint: sub-tile `sub` of tile t, events [64 sub, 64 sub + 64).
// XN > 0: every channel has at most XN randoms, and each event's row is held in registers.
// SID >= 0: the tile's channel has that compile-time tree shape (XN is then its n_x).
// Partials go to the tile's global unit.
template <int XN, bool COMPACT, int SID, int LM, bool PEV, bool FR>
__device__ __forceinline__ void adjoint_unit(int t, int sub, int n_sub, const TileDesc& td, const SegDesc& sd,
                                             const ChannelDesc& cd, const NodeCmd* __restrict__ prog,
                                             double* __restrict__ gpart, int part_stride, const AdjLayout& lay,
                                             double* lds) {
  const int lane = threadIdx.x;
  LdsStore<COMPACT> S{lds + lane, lay.off_in, lay.off_st};
  // the (M, Gamma) accumulators: in registers for the small programs (XN > 0: n_out <= 4, at
  // most kSmallParams), else in LDS after the tape
  double accv[XN > 0 ? kSmallParams : 1];
  LdsAcc acc_lds{lds + lay.off_acc * 64 + lane};
  const int np = 2 * cd.n_nodes;
  if constexpr (XN > 0) {
#pragma unroll
    for (int v = 0; v < kSmallParams; v++) accv[v] = 0;
  } else {
    for (int v = 0; v < np; v++) acc_lds[v] = 0;
  }
  const int end = min(td.count, 64 * (sub + 1));
  // a unit has at most 64 events: one per lane, no loop (constants are not hoisted out of one)
  if (const int local = 64 * sub + lane; local < end) {
    const int64_t e = td.e0 + local;
    const double* xg = sd.x + e * cd.n_x;
    const double* gp = sd.g_p ? sd.g_p + e * (int64_t)cd.n_out * 4 : nullptr;
    const double gf = sd.g_f ? sd.g_f[e] : 0.0;
    double* p_out = sd.p ? sd.p + e * (int64_t)cd.n_out * 4 : nullptr;
    double F = 0, L = 0;
    bool ok;
    EvBeams eb;
    if constexpr (PEV) eb = event_beams(cd, sd.e1[e], sd.e2[e]);
    else eb = fixed_beams(cd);
    if constexpr (XN > 0) {
      double xv[XN];
#pragma unroll
      for (int k = 0; k < XN; k++) xv[k] = xg[SID >= 0 || k < cd.n_x ? k : cd.n_x - 1];   // entries past n_x are never read
      ok = event_adjoint<SID, LM, PEV, FR>(cd, eb, prog, xv, gp, gf, p_out, &F, &L, sd.g_x + e * cd.n_x, accv, S);
    } else {
      ok = event_adjoint<SID, LM, PEV, FR>(cd, eb, prog, xg, gp, gf, p_out, &F, &L, sd.g_x + e * cd.n_x, acc_lds, S);
    }
    if (sd.factor) sd.factor[e] = F;
    if (sd.volume) sd.volume[e] = eb.volume;
    if (sd.ok) sd.ok[e] = ok ? 1 : 0;
    if (sd.loss) sd.loss[e] = L;
  }
  double* part = gpart + ((int64_t)t * n_sub + sub) * part_stride;
  if constexpr (XN > 0) {
    wave_sums(accv);
#pragma unroll
    for (int v = 0; v < kSmallParams; v++)
      if (lane == 0 && v < np) part[v] = accv[v];
  } else {
    for (int v = 0; v < np; v++) {
      const double tot = wave_sum(acc_lds[v]);
      if (lane == 0) part[v] = tot;
    }
  }
}

// The generic adjoint, and the one with per-event beam energies of the trees of up to four final-state
// particles.  The launch covers tiles [t_begin, t_begin + n_units / n_sub): unit u is sub-tile (u % n_sub)
// of tile t_begin + u / n_sub.  SID = kAdjMulti: every tile's channel has one of the shapes of up to four
// final-state particles, and each workgroup takes the specialised code of its tile's shape.  The register
// budget keeps two waves per SIMD (at most 256 VGPRs).  PEV: per-event beam energies (loss mode 0).  FR:
// plans with friend branches (the generic walk, randoms read from memory, accumulators in LDS).
constexpr int kAdjMulti = 1000;
template <int XN, bool COMPACT, int SID, int LM, bool PEV = false, bool FR = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void adjoint_kernel(
    const TileDesc* __restrict__ tiles, int t_begin, int n_units, int n_sub, const SegDesc* __restrict__ segs,
    const ChannelDesc* __restrict__ chans, const NodeCmd* __restrict__ nodes, double* __restrict__ gpart,
    int part_stride, AdjLayout lay) {
  extern __shared__ double lds[];
  // one workgroup per unit (the host launches n_units workgroups): no loop
  if (const int u = (int)blockIdx.x; u < n_units) {
    const int tl = u / n_sub, sub = u - tl * n_sub, t = t_begin + tl;
    const TileDesc td = tiles[t];
    const SegDesc sd = segs[td.seg];
    const ChannelDesc cd = chans[sd.channel];
    const NodeCmd* prog = nodes + cd.node0;
    if constexpr (SID == kAdjMulti) {
      switch (cd.shape) {
        case 0: adjoint_unit<kShapes[0].n_x, COMPACT, 0, LM, PEV, false>(t, sub, n_sub, td, sd, cd, prog, gpart, part_stride, lay, lds); break;
        case 1: adjoint_unit<kShapes[1].n_x, COMPACT, 1, LM, PEV, false>(t, sub, n_sub, td, sd, cd, prog, gpart, part_stride, lay, lds); break;
        case 2: adjoint_unit<kShapes[2].n_x, COMPACT, 2, LM, PEV, false>(t, sub, n_sub, td, sd, cd, prog, gpart, part_stride, lay, lds); break;
        case 3: adjoint_unit<kShapes[3].n_x, COMPACT, 3, LM, PEV, false>(t, sub, n_sub, td, sd, cd, prog, gpart, part_stride, lay, lds); break;
        case 4: adjoint_unit<kShapes[4].n_x, COMPACT, 4, LM, PEV, false>(t, sub, n_sub, td, sd, cd, prog, gpart, part_stride, lay, lds); break;
        case 5: adjoint_unit<kShapes[5].n_x, COMPACT, 5, LM, PEV, false>(t, sub, n_sub, td, sd, cd, prog, gpart, part_stride, lay, lds); break;
        case 6: adjoint_unit<kShapes[6].n_x, COMPACT, 6, LM, PEV, false>(t, sub, n_sub, td, sd, cd, prog, gpart, part_stride, lay, lds); break;
        case 7: adjoint_unit<kShapes[7].n_x, COMPACT, 7, LM, PEV, false>(t, sub, n_sub, td, sd, cd, prog, gpart, part_stride, lay, lds); break;
        default: break;   // not reached: the host launches only tiles of shapes 0-7 here
      }
    } else {
      adjoint_unit<XN, COMPACT, SID, LM, PEV, FR>(t, sub, n_sub, td, sd, cd, prog, gpart, part_stride, lay, lds);
    }
  }
}

// gparam[2 * slot + w] = sum over the sub-tiles of the tiles of the slot's channel (every slot
// is written, channels without events get 0).  A channel's units are split into ranges of
// kRangeUnits, at most kSplit, one workgroup each: thread t adds units t, t + 256, ..., then a fixed
// tree (a butterfly within each wave, the four waves in order).  The one range of a small channel is
// its sum; otherwise the workgroup that finishes the channel's last range adds the range sums in order.
// Every sum has a fixed order, so results do not depend on scheduling.  `done` counts the finished
// ranges per channel; the last workgroup resets it to 0, so it is 0 again when the launch ends.
//
// Bound by latency.  Range sums are published with device-scope stores and read with device-scope
// loads: a release fence would write back the L2's dirty lines, the gradients the adjoint has just
// written.  The sums of all parameters go through the wave together (wave_sums).  15,627 units of 3
// channels 12 -> 9 us, 3,150 units of 16 channels of 10 parameters 25 -> 6.5 us.
constexpr int kRangeUnits = 512;
constexpr int kReduceThreads = 256;
constexpr int kSplit = kAdjRanges;
constexpr int kMaxParams = 2 * (kMaxOut - 1);
// NP: parameters of the largest channel, at least (the entries past a channel's own are not used).
template <int NP>
__global__ __launch_bounds__(kReduceThreads) void param_reduce(
    const double* __restrict__ gpart, int part_stride, int n_sub, const int* __restrict__ chan_tiles,
    const int* __restrict__ chan_tile_off, const ChannelDesc* __restrict__ chans, int n_chans,
    double* __restrict__ granges, unsigned int* __restrict__ done, double* __restrict__ gparam) {
  __shared__ double red[kReduceThreads / 64][NP];
  const int c = blockIdx.x / kSplit, r = blockIdx.x % kSplit;
  if (c >= n_chans) return;
  const int np = 2 * chans[c].n_nodes;
  const int t0 = chan_tile_off[c];
  const int n_units = (chan_tile_off[c + 1] - t0) * n_sub;
  const int n_ranges = max(1, min(kSplit, (n_units + kRangeUnits - 1) / kRangeUnits));
  if (r >= n_ranges) return;
  const int chunk = (n_units + n_ranges - 1) / n_ranges;
  const int u0 = r * chunk, u1 = min(n_units, u0 + chunk);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  double sum[NP];
#pragma unroll
  for (int v = 0; v < NP; v++) sum[v] = 0;
  for (int k = u0 + tid; k < u1; k += kReduceThreads) {
    const int tile = chan_tiles[t0 + k / n_sub];
    const double* src = gpart + ((int64_t)tile * n_sub + k % n_sub) * part_stride;
#pragma unroll
    for (int v = 0; v < NP; v++) sum[v] += src[v < part_stride ? v : 0];
  }
  wave_sums(sum);
#pragma unroll
  for (int v = 0; v < NP; v++)
    if (lane == 0) red[wv][v] = sum[v];
  __syncthreads();
  // (np < 64: what follows is the first wave's)
  const double mine = tid < np ? ((red[0][tid] + red[1][tid]) + red[2][tid]) + red[3][tid] : 0.0;
  double* out = gparam + 2 * chans[c].param0;
  if (n_ranges == 1) {
    if (tid < np) out[tid] = mine;
    return;
  }
  if (wv != 0) return;
  // publish this range, then count it; the workgroup that counts the channel's last range sees every
  // range: each store has reached the device's coherence point before its workgroup counts
  unsigned long long* sums = (unsigned long long*)granges + (int64_t)c * kSplit * part_stride;
  if (tid < np)
    __hip_atomic_store(sums + r * part_stride + tid, __builtin_bit_cast(unsigned long long, mine), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  unsigned int before = 0;
  if (lane == 0) before = __hip_atomic_fetch_add(&done[c], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (__builtin_amdgcn_readfirstlane(before) != (unsigned int)(n_ranges - 1)) return;
  asm volatile("" ::: "memory");
  if (tid < np) {
    double s = 0;
    for (int q = 0; q < n_ranges; q++)
      s += __builtin_bit_cast(double, __hip_atomic_load(sums + q * part_stride + tid, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT));
    out[tid] = s;
  }
  if (tid == 0) done[c] = 0;
}

using AdjKernel = adj::Kernel;

// The kernel of the shapes [lo, hi] that a launch has (of one group): those of one number of final-state
// particles, or of all of two to four.  Waves per SIMD: as many as the registers hold without spills, so two
// for the trees of four with given cotangents (10^6 events: 96 us; at three, with 108 bytes of scratch per
// lane, 129).  The trees of six with given cotangents take all 256 registers that two leave a lane, and
// 44 bytes of scratch.
template <int LM>
adj::Kernel pick_shapes(int lo, int hi) {
  if (hi < 1) return adj::shapes_kernel<0, 1, LM, 4>;
  if (lo >= 1 && hi < 3) return adj::shapes_kernel<1, 3, LM, 3>;
  if (lo >= 3 && hi < 8) return adj::shapes_kernel<3, 8, LM, LM ? 3 : 2>;
  if (hi < 8) return adj::shapes_kernel<0, 8, LM, LM ? 3 : 2>;
  if (hi < 22) return adj::pick_5(LM);
  return LM ? adj::pick_6_1() : adj::pick_6_0();
}

template <int LM>
AdjKernel adj_generic(const DevicePlan& dp, const AdjLayout& lay) {
  if (dp.has_friends) {   // the host sets no compact stash and keeps the accumulators in LDS
    if constexpr (LM == 0) {
      if (dp.per_event_beams) return adjoint_kernel<0, false, -1, 0, true, true>;
    }
    return adjoint_kernel<0, false, -1, LM, false, true>;
  }
  if constexpr (LM == 0) {   // per-event beams: the external cotangents only (the built-in loss assumes equal beams)
    if (dp.per_event_beams)
      return dp.nx_max > kAdjXReg ? adjoint_kernel<0, false, -1, 0, true>
             : lay.compact ? adjoint_kernel<kAdjXReg, true, -1, 0, true> : adjoint_kernel<kAdjXReg, false, -1, 0, true>;
  }
  return dp.nx_max > kAdjXReg ? adjoint_kernel<0, false, -1, LM>
         : lay.compact ? adjoint_kernel<kAdjXReg, true, -1, LM> : adjoint_kernel<kAdjXReg, false, -1, LM>;
}

}  // namespace

hipError_t launch_adjoint(const DevicePlan& dp, const AdjLayout& lay, const TileRun* runs, int n_runs, int loss_mode,
                          double* gpart, int part_stride, int n_sub, double* granges, unsigned int* done,
                          const int* chan_tiles, const int* chan_tile_off, int n_chans, double* gparam,
                          hipStream_t stream) {
  const size_t shmem = (size_t)lay.words * 64 * sizeof(double);
  if (shmem > forward_lds_limit() || n_sub < 1) return hipErrorInvalidValue;
  if ((int64_t)dp.n_tiles * n_sub > 0x7fffffff) return hipErrorInvalidValue;
  if (dp.per_event_beams && loss_mode != 0) return hipErrorInvalidValue;
  AdjKernel generic = loss_mode ? adj_generic<1>(dp, lay) : adj_generic<0>(dp, lay);
  AdjKernel multi_pev = lay.compact ? adjoint_kernel<kAdjXReg, true, kAdjMulti, 0, true>
                                    : adjoint_kernel<kAdjXReg, false, kAdjMulti, 0, true>;
  auto group = [](int sid) { return sid < 0 ? -1 : shape_group(kShapes[sid].n_out); };
  for (int r = 0; r < n_runs;) {
    // consecutive runs of shapes of one group: one launch (a launch lasts at least one wave's lifetime)
    int r1 = r + 1, end = runs[r].end, lo = runs[r].sid, hi = lo;
    for (; r1 < n_runs && runs[r].sid >= 0 && group(runs[r1].sid) == group(runs[r].sid) && runs[r1].begin == end; r1++) {
      end = runs[r1].end;
      lo = std::min(lo, runs[r1].sid);
      hi = std::max(hi, runs[r1].sid);
    }
    const int units = (end - runs[r].begin) * n_sub;
    const bool shapes = lo >= 0 && !dp.has_friends, own = shapes && !dp.per_event_beams;   // own: LDS of its own
    AdjKernel k = !shapes ? generic
                  : !own  ? (hi < kAdjPevShapes ? multi_pev : generic)
                          : (loss_mode ? pick_shapes<1>(lo, hi) : pick_shapes<0>(lo, hi));
    if (units > 0) {
      hipLaunchKernelGGL(k, dim3(units), dim3(64), own ? 0 : shmem, stream, dp.tiles, runs[r].begin, units, n_sub, dp.segs,
                         dp.chans, dp.nodes, gpart, part_stride, lay);
      hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
    }
    r = r1;
  }
  if (n_chans > 0) {
    // (the trees of up to four and of up to six final-state particles, and all)
    auto reduce = part_stride <= 6 ? param_reduce<6> : part_stride <= 10 ? param_reduce<10> : param_reduce<kMaxParams>;
    hipLaunchKernelGGL(reduce, dim3(n_chans * kSplit), dim3(kReduceThreads), 0, stream, gpart, part_stride,
                       n_sub, chan_tiles, chan_tile_off, dp.chans, n_chans, granges, done, gparam);
  }
  return hipGetLastError();
}

}  // namespace gphs
