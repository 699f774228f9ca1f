// Inverse mapping (device code shared by the translation units that instantiate it: phs_inverse.hip,
// and phs_inverse_5.hip and phs_inverse_6.hip for the trees of five and six final-state particles):
// for every event and every channel of its process, the randoms and the phase-space factor under
// which that channel would have produced the event's momenta (what Whizard's multi-channel weight
// needs; reference phs.cu:626-675, 924-1284, driven per channel by phs.cu:1499-1554 with 2 + 2(n-1)
// dependent launches per channel).
//
// One lane = one event, one launch for all channels: a wave takes 64 events of one generating channel,
// stages their momenta (boosted back to the centre-of-mass frame) in an LDS column per lane, and walks
// every channel's tree in turn (wave-uniform: all lanes invert into the same channel at the same time,
// reading its records with scalar loads).  The generating channel's slot gets the forward pass's own
// factor and randoms, as the reference's _move_factors / _move_x do (phs.cu:1495-1497).
//
// The steps per branch follow the GPU reference with its defects corrected (the oracle's
// inverse lists them): the msq of both daughters from sums of final-state momenta (added as
// the reference adds them, daughter by daughter), x and the
// map factor of each internal daughter from its msq, lambda and the decay momentum, then the
// angles of the first daughter in B_z(-bg) G, where G = L_parent^-1 is carried down the tree
// (a branch with a friend measures them from the friend beam), x_phi = atan2 / 2 pi, x of
// cos theta from its map, and G <- R_y(-theta) R_z(-phi) B_z(-bg) G for the daughters.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "phs_device.h"
#include "phs_kernels.h"
#include "phs_walk.h"

namespace gphs {
namespace inv {

constexpr int kInvBankWords = 19;

// The lane's column of the sub-tile's randoms table x[k][event] (rows of `stride` doubles).
struct XColumn {
  double* p;
  int stride;
  __device__ __forceinline__ double& operator[](int k) const { return p[k * stride]; }
};

extern __shared__ double inv_lds[];

// x and the map factor of an internal daughter from its msq (mappings_gpu.hpp:15-172; STEP_H
// as phs_cpu.cpp:95-101, whose root of the quadratic is the right one).
__device__ __forceinline__ void x_from_msq(const ChildCmd& c, double msq, double s, double& x, double& f) {
  switch (c.kind) {
    case MK_LINEAR:
      x = (msq - c.msq_min) / (c.msq_max - c.msq_min);
      f = c.f_lin;
      break;
    case MK_BREIT_WIGNER: {
      const double z = (msq - c.m * c.m) / (c.m * c.w);
      // (the device library's atan keeps its coefficients in forty vector registers)
      x = (math::atan_radians(z) - c.a0) / (c.a1 - c.a0);
      f = c.a2 * (1 + z * z);
      break;
    }
    case MK_EXP: {
      const double z = msq - c.msq_min + c.a0;
      x = math::log_bounded(z / c.a0) / c.a1;
      f = c.a2 * z;
      break;
    }
    case MK_TU: {
      const bool lo = msq < (c.msq_max + c.msq_min) / 2;
      const double z = lo ? msq - c.msq_min + c.a0 : c.msq_max - msq + c.a0;
      const double l = math::log_bounded(z / c.a0) / c.a1;
      x = lo ? l : 1 - l;
      f = c.a2 * z;
      break;
    }
    case MK_STEP_H: {
      const double z = (msq - c.msq_min) / (c.msq_max - c.msq_min);
      const double t = c.a1 / (c.a0 * c.a2);
      const double u = c.a0 + z / c.a2, v = c.a0 - z / c.a2;
      x = ((u + t) - math::sqrt_phys(v * v + 2 * t * u + t * t)) / 2;
      f = (c.a1 / (c.a0 - x) / (c.a0 - x) + c.a2) * (c.msq_max - c.msq_min) / s;
      break;
    }
    default: {  // MK_STEP_E
      const double z = (msq - c.msq_min) / (c.msq_max - c.msq_min);
      const double t = 1 + c.a1 * math::exp_bounded(z / c.a2);
      x = (z - c.a2 * math::log_bounded(t / (1 + c.a1))) / c.a0;
      f = c.a0 * t * (c.msq_max - c.msq_min) / s;
      break;
    }
  }
}

// x and factor of cos theta (mappings_gpu.hpp:181-219).
__device__ __forceinline__ void x_from_ct(int kind, double ct, double b0, double b1, double& x, double& f) {
  if (kind == CK_FLAT) {
    x = (ct + 1) / 2;
    f = 1;
  } else {
    const bool neg = ct < 0;
    const double t = neg ? ct + b0 + 1 : -ct + b0 + 1;
    const double l = math::log_bounded(t / b0) / (2 * b1);
    x = neg ? l : 1 - l;
    f = t * b1;
  }
}

// The same from an InvNode: every constant formed on the host, and the quotients by constants through
// their reciprocals (the same bits).
__device__ __forceinline__ void x_from_map(int kind, const InvMap& m, double msq, double s, double& x, double& f) {
  using math::divide;
  const math::Divisor d0{m.p1, m.inv0}, d1{m.q1, m.inv1};
  switch (kind) {
    case MK_LINEAR:   // msq_min, msq_max - msq_min; f
      x = divide(msq - m.p0, d0);
      f = m.c;
      break;
    case MK_BREIT_WIGNER: {   // M^2, M Gamma; a0, a1 - a0; a2
      const double z = divide(msq - m.p0, d0);
      x = divide(math::atan_radians(z) - m.q0, d1);
      f = m.c * (1 + z * z);
      break;
    }
    case MK_EXP: {   // msq_min, a0; msq_max, a1; a2 (also below)
      const double z = msq - m.p0 + m.p1;
      x = divide(math::log_bounded(divide(z, d0)), d1);
      f = m.c * z;
      break;
    }
    case MK_TU: {
      const bool lo = msq < (m.q0 + m.p0) / 2;
      const double z = lo ? msq - m.p0 + m.p1 : m.q0 - msq + m.p1;
      const double l = divide(math::log_bounded(divide(z, d0)), d1);
      x = lo ? l : 1 - l;
      f = m.c * z;
      break;
    }
    case MK_STEP_H: {
      const double z = (msq - m.p0) / (m.q0 - m.p0);
      const double t = m.q1 / (m.p1 * m.c);
      const double u = m.p1 + z / m.c, v = m.p1 - z / m.c;
      x = ((u + t) - math::sqrt_phys(v * v + 2 * t * u + t * t)) / 2;
      f = (m.q1 / (m.p1 - x) / (m.p1 - x) + m.c) * (m.q0 - m.p0) / s;
      break;
    }
    default: {  // MK_STEP_E
      const double z = (msq - m.p0) / (m.q0 - m.p0);
      const double t = 1 + m.q1 * math::exp_bounded(z / m.c);
      x = (z - m.c * math::log_bounded(t / (1 + m.q1))) / m.p1;
      f = m.p1 * t * (m.q0 - m.p0) / s;
      break;
    }
  }
}
__device__ __forceinline__ void x_from_ct(const InvNode& nd, double ct, double& x, double& f) {
  if (nd.ct_kind == CK_FLAT) {
    x = (ct + 1) / 2;
    f = 1;
  } else {
    const bool neg = ct < 0;
    const double t = neg ? ct + nd.b0 + 1 : -ct + nd.b0 + 1;
    const double l = math::divide(math::log_bounded(math::divide(t, {nd.b0, nd.inv_b0})), {2 * nd.b1, nd.inv_2b1});
    x = neg ? l : 1 - l;
    f = t * nd.b1;
  }
}

// An InvNode in scalar registers: read as a whole before the first branch on what it holds, so that the
// wave waits for it once (loads left where they are used cost a wait each: some 29 per event and
// channel of a 2->4 tree, 39% of the waves' time).
__device__ __forceinline__ InvNode load_node(const InvNode* __restrict__ p) { return *p; }
template <bool MAP0, bool MAP1>
__device__ __forceinline__ void arrived(InvNode& nd) {
  keep_scalar(nd.ct_kind);
  keep_scalar(nd.b0); keep_scalar(nd.b1); keep_scalar(nd.inv_b0); keep_scalar(nd.inv_2b1);
#pragma unroll
  for (int d = 0; d < 2; d++) {
    if (!(d == 0 ? MAP0 : MAP1)) continue;
    keep_scalar(nd.kind[d]);
    InvMap& m = nd.map[d];
    keep_scalar(m.p0); keep_scalar(m.p1); keep_scalar(m.inv0); keep_scalar(m.q0); keep_scalar(m.q1);
    keep_scalar(m.inv1); keep_scalar(m.c);
  }
}

// Sum of the staged final-state momenta in `leaves` (lane column pl, stride S).
__device__ __forceinline__ void leaf_sum(const double* __restrict__ pl, int S, int n_out, uint32_t leaves,
                                         double (&q)[4]) {
  q[0] = q[1] = q[2] = q[3] = 0;
  for (int j = 0; j < n_out; j++) {
    if ((leaves >> j) & 1u) {
      const double* r = pl + 4 * j * S;
      q[0] = q[0] + r[0]; q[1] = q[1] + r[S]; q[2] = q[2] + r[2 * S]; q[3] = q[3] + r[3 * S];
    }
  }
}

// A daughter's four-momentum: its sum program (ChildCmd::sum_code) over the staged final-state
// momenta, which adds them in the reference's association, daughter sums first; the index
// order of `leaves` where the subtree has no program.
__device__ __forceinline__ void branch_sum(const double* __restrict__ pl, int S, int n_out, const ChildCmd& c,
                                           double (&q)[4]) {
  if (c.sum_len <= 0) {
    leaf_sum(pl, S, n_out, c.leaves, q);
    return;
  }
  double a[4] = {0, 0, 0, 0}, b[4] = {0, 0, 0, 0};
  bool second = false;
  uint64_t code = c.sum_code;
  for (int t = 0; t < c.sum_len; t++, code >>= 4) {
    const int op = (int)(code & 15u);
    if (op == kSumPush) {
      second = true;
      b[0] = b[1] = b[2] = b[3] = 0;
    } else if (op == kSumMerge) {
      a[0] = a[0] + b[0]; a[1] = a[1] + b[1]; a[2] = a[2] + b[2]; a[3] = a[3] + b[3];
      second = false;
    } else {
      const double* r = pl + 4 * op * S;
      if (second) {
        b[0] = b[0] + r[0]; b[1] = b[1] + r[S]; b[2] = b[2] + r[2 * S]; b[3] = b[3] + r[3 * S];
      } else {
        a[0] = a[0] + r[0]; a[1] = a[1] + r[S]; a[2] = a[2] + r[2 * S]; a[3] = a[3] + r[3 * S];
      }
    }
  }
  q[0] = a[0]; q[1] = a[1]; q[2] = a[2]; q[3] = a[3];
}

// G <- R_y(-theta) R_z(-phi) G (rows 1..3)
__device__ __forceinline__ void rotate_back(double (&G)[16], double ct, double st, double cp, double sp) {
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const double w1 = G[4 + j], w2 = G[8 + j], w3 = G[12 + j];
    const double t1 = cp * w1 + sp * w2;
    G[4 + j] = ct * t1 - st * w3;
    G[8 + j] = -sp * w1 + cp * w2;
    G[12 + j] = st * t1 + ct * w3;
  }
}

// One branch's decay from its own msq and mass and its daughters' msq (phs.cu:658-664):
// p_decay, the factor sqrt(lambda) / msq (0 where lambda <= 0, phs_cpu.cpp:275-279), and the
// boost bg = p_parent / m.  The quotients are correctly rounded, as the reference's divisions
// are: they feed the frames of the daughters and so the cosines that the peaked maps take near
// +-1, where an ulp of cos theta is amplified by up to sqrt(s) / m^2 in the map's factor.
struct Decay {
  double pk, lam, bg;
};
__device__ __forceinline__ Decay decay(const math::Divisor& by_msq, const math::Divisor& m, double cur_p, double msq0,
                                       double msq1) {
  const double cur_msq = by_msq.d, cur_m = m.d;
  const double lda = (cur_msq - msq0 - msq1) * (cur_msq - msq0 - msq1) - 4 * msq0 * msq1;
  const bool pos = lda > 0;
  const double sl = pos ? math::sqrt_phys(lda) : 0.0;
  Decay d;
  d.pk = math::divide(sl, {2 * cur_m, 0.5 * m.r});
  d.lam = pos ? math::divide(sl, by_msq) : 0.0;
  d.bg = cur_m > 0 ? math::divide(cur_p, m) : 0.0;
  return d;
}
__device__ __forceinline__ Decay decay(double cur_msq, double cur_m, double cur_p, double msq0, double msq1) {
  return decay(math::divisor(cur_msq), math::divisor(cur_m), cur_p, msq0, msq1);
}

// Polar and azimuthal angles of the direction v (mappings_gpu.hpp:196-219 inverted): the
// cosines and sines of both angles (correctly rounded quotients, as above) and
// x_phi = atan2(v1, v0) / 2 pi in [0, 1], formed in turns by math::atan2_turns.
struct Dir {
  double xphi, ct, st, cp, sp;
};
__device__ __forceinline__ Dir direction(double v0, double v1, double v2) {
  math::Divisor dr, dv;
  const double rho = math::sqrt_phys(v0 * v0 + v1 * v1, dr);
  math::sqrt_phys(v0 * v0 + v1 * v1 + v2 * v2, dv);
  Dir d;
  d.xphi = math::atan2_turns(v1, v0);
  d.cp = rho > 0 ? math::divide(v0, dr) : 1.0;
  d.sp = rho > 0 ? math::divide(v1, dr) : 0.0;
  d.ct = math::divide(v2, dv);
  d.st = math::divide(rho, dv);
  return d;
}

// ---- shared roots --------------------------------------------------------------------------
//
// The root of every channel sits in the centre-of-mass frame (G = 1, p_decay = 0, so its boost
// is the identity and v = the first daughter's momentum, bit for bit), and what it computes from
// the event -- both daughters' msq, lambda, p_decay and the first daughter's angles -- depends
// only on which final-state particles each daughter holds and in which association they are
// added.  Channels whose roots agree in both (the same root split up to the orientation of the
// subtrees below it) share one evaluation: the host orders the channels so that they follow one
// another, and the kernel evaluates the root when a new group starts.  Each channel then only
// applies its own maps to the shared numbers (x and factor of its internal daughters' msq, x
// and factor of cos theta) and walks the rest of its tree from the root's frame, which is the
// rotation R_y(-theta) R_z(-phi) of the identity, re-formed from four numbers.  That frame and
// the group's msq, m and p_decay also stand in for a subtree the root defers, so the save bank
// holds only subtrees deferred below the root.

struct RootGeo {
  double msq[2];          // msq of the daughters, from the sums of their final-state momenta
  math::Divisor m[2];     // sqrt(msq) of an internal daughter (unused for a final-state one)
  double lam;             // sqrt(lambda) / s, 0 where lambda <= 0 (phs_cpu.cpp:275-279)
  double pk;              // p_decay = sqrt(lambda) / (2 sqrt(s))
  double xphi;            // phi / 2 pi of daughter 0
  double ct, st, cp, sp;  // cos and sin of its polar and azimuthal angles
};

// (by_s, by_sqrts: the event's s and sqrt(s))
__device__ __forceinline__ RootGeo root_geometry(const double (&q0)[4], const double (&q1)[4], bool leaf0, bool leaf1,
                                                 const math::Divisor& by_s, const math::Divisor& by_sqrts) {
  RootGeo r;
  r.msq[0] = q0[0] * q0[0] - q0[1] * q0[1] - q0[2] * q0[2] - q0[3] * q0[3];
  r.msq[1] = q1[0] * q1[0] - q1[1] * q1[1] - q1[2] * q1[2] - q1[3] * q1[3];
  if (!leaf0) math::sqrt_phys(r.msq[0], r.m[0]);
  if (!leaf1) math::sqrt_phys(r.msq[1], r.m[1]);
  const Decay dk = decay(by_s, by_sqrts, 0.0, r.msq[0], r.msq[1]);
  r.pk = dk.pk;
  r.lam = dk.lam;
  // G = 1 and bg = 0 at the root: v is daughter 0's momentum
  const Dir dr = direction(q0[1], q0[2], q0[3]);
  r.xphi = dr.xphi;
  r.ct = dr.ct; r.st = dr.st; r.cp = dr.cp; r.sp = dr.sp;
  return r;
}

// G of the root's daughters: the root's rotation R_y(-theta) R_z(-phi) of the identity, without
// the products by 0 and 1 (rotate_back's bits, up to the sign of a zero).
__device__ __forceinline__ void root_frame(double (&G)[16], const RootGeo& g) {
  G[0] = 1; G[1] = 0;            G[2] = 0;            G[3] = 0;
  G[4] = 0; G[5] = g.ct * g.cp;  G[6] = g.ct * g.sp;  G[7] = -g.st;
  G[8] = 0; G[9] = -g.sp;        G[10] = g.cp;        G[11] = 0;
  G[12] = 0; G[13] = g.st * g.cp; G[14] = g.st * g.sp; G[15] = g.ct;
}

template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// ---- walks specialised per tree shape --------------------------------------------------------
//
// The trees of two to six final-state particles (InvStep::shape, of the compile-time table): every
// branch's structure is a constant, the final-state slots come from InvStep::outs, and what a channel's
// maps need of a branch from its InvNode (or, with per-event beams, for up to four particles, from
// its NodeCmd).  No branch has a friend.

// Final-state momentum of daughter C of branch I.
template <int I, int C>
__device__ __forceinline__ void leaf_momentum(uint64_t outs, const double* __restrict__ pl, double (&q)[4]) {
  const double* r = pl + 4 * 64 * (int)((outs >> (4 * (2 * I + C))) & 15u);
  q[0] = r[0]; q[1] = r[64]; q[2] = r[128]; q[3] = r[192];
}

// Momentum of daughter C of branch I, in the reference's association (each branch the sum of its two
// daughters, phs.cu:1262-1275; the sum programs of branch_sum add the same pairs, in an order that
// differs only by commutation).
template <int SID, int I, int C>
__device__ __forceinline__ void daughter_sum(uint64_t outs, const double* __restrict__ pl, double (&q)[4]) {
  constexpr ShapeNode N = kShapes[SID].node[I];
  if constexpr (C == 0 ? N.leaf0 : N.leaf1) {
    leaf_momentum<I, C>(outs, pl, q);
  } else {
    constexpr int V = (C == 0 ? N.node0 : N.node1) < 0 ? 0 : (C == 0 ? N.node0 : N.node1);
    double a[4], b[4];
    daughter_sum<SID, V, 0>(outs, pl, a);
    daughter_sum<SID, V, 1>(outs, pl, b);
    q[0] = a[0] + b[0]; q[1] = a[1] + b[1]; q[2] = a[2] + b[2]; q[3] = a[3] + b[3];
  }
}

// A channel's records: what its maps read (nodes with per-event beams, else maps).
struct Records {
  const NodeCmd* nodes;
  const InvNode* maps;
};

// One channel's maps of branch I's geometry, in the order of the walk: x and factor of its internal
// daughters' msq, sqrt(lambda) / msq, and x and factor of its angles.
template <int SID, int I, bool PEV, class XO>
__device__ __forceinline__ void branch_maps(const ChannelDesc& cd, const EvBeams& eb, const Records& rec, double msq0,
                                            double msq1, double lam, double xphi, double ct, XO xo, double& factor) {
  constexpr ShapeNode N = kShapes[SID].node[I];
  InvNode nd;
  if constexpr (!PEV) {
    nd = load_node(rec.maps + I);
    arrived<!N.leaf0, !N.leaf1>(nd);
  }
  auto msq_map = [&](int d, double msq, int xi) {
    double x, f;
    if constexpr (PEV) x_from_msq(child_at(rec.nodes[I].k[d], eb.sqrts, eb.s, cd.m_tot), msq, eb.s, x, f);
    else x_from_map(nd.kind[d], nd.map[d], msq, eb.s, x, f);
    xo[xi] = x;
    factor *= f;
  };
  if constexpr (!N.leaf0) msq_map(0, msq0, N.xi0);
  if constexpr (!N.leaf1) msq_map(1, msq1, N.xi1);
  factor *= lam;
  xo[N.xphi] = xphi;
  double x, f;
  if constexpr (PEV) {
    double m_max, b0, b1;
    node_at(rec.nodes[I], I == 0, eb, cd.m_tot, m_max, b0, b1);
    x_from_ct(rec.nodes[I].ct_kind, ct, b0, b1, x, f);
  } else {
    x_from_ct(nd, ct, x, f);
  }
  xo[N.xphi + 1] = x;
  factor *= f;
}

template <int SID>
__device__ __forceinline__ RootGeo root_of(uint64_t outs, const math::Divisor& by_s, const math::Divisor& by_sqrts,
                                           const double* __restrict__ pl) {
  constexpr ShapeNode N = kShapes[SID].node[0];
  double q0[4], q1[4];
  daughter_sum<SID, 0, 0>(outs, pl, q0);
  daughter_sum<SID, 0, 1>(outs, pl, q1);
  return root_geometry(q0, q1, N.leaf0, N.leaf1, by_s, by_sqrts);
}

// The rows of G that a branch below the root measures its angles in: v = rows 1 to 3 of B_z(-bg) G on
// q; G becomes B_z(-bg) G.  ROOT: G is root_frame, whose zeros (rows 1 and 2 of column 0, [2][3]) and
// ones are left out of the sums.
template <bool ROOT>
__device__ __forceinline__ void boost_back(double (&G)[16], double gm, double bg, const double (&q)[4], double (&v)[3]) {
  if constexpr (ROOT) {
    G[0] = gm;
    G[12] = -bg;
#pragma unroll
    for (int j = 1; j < 4; j++) {
      const double r3 = G[12 + j];
      G[j] = -(bg * r3);
      G[12 + j] = gm * r3;
    }
    v[0] = G[5] * q[1] + G[6] * q[2] + G[7] * q[3];
    v[1] = G[9] * q[1] + G[10] * q[2];
  } else {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const double r0 = G[j], r3 = G[12 + j];
      G[j] = gm * r0 - bg * r3;
      G[12 + j] = -bg * r0 + gm * r3;
    }
    v[0] = G[4] * q[0] + G[5] * q[1] + G[6] * q[2] + G[7] * q[3];
    v[1] = G[8] * q[0] + G[9] * q[1] + G[10] * q[2] + G[11] * q[3];
  }
  v[2] = G[12] * q[0] + G[13] * q[1] + G[14] * q[2] + G[15] * q[3];
}

// rotate_back after boost_back<true>: the zeros of G (rows 1 and 2 of column 0, [2][3]) left out.
__device__ __forceinline__ void rotate_back_root(double (&G)[16], double ct, double st, double cp, double sp) {
  const double w3 = G[12];
  G[4] = -(st * w3);
  G[8] = 0;
  G[12] = ct * w3;
#pragma unroll
  for (int j = 1; j < 4; j++) {
    const double w1 = G[4 + j], w2 = G[8 + j], w3j = G[12 + j];
    const double t1 = j == 3 ? cp * w1 : cp * w1 + sp * w2;
    G[4 + j] = ct * t1 - st * w3j;
    G[8 + j] = j == 3 ? -(sp * w1) : -sp * w1 + cp * w2;
    G[12 + j] = st * t1 + ct * w3j;
  }
}

// The inverse of one event into one channel of shape SID from its root group's geometry `g`, branch by
// branch: the randoms go to xo[0..n_x), returns the factor.  One subtree at a time is deferred below
// the root, in registers (the root's own deferred daughter starts from `g` again).
template <int SID, bool PEV, class XO>
__device__ __forceinline__ double inverse_walk(const ChannelDesc& cd, const EvBeams& eb, const Records& rec,
                                               uint64_t outs, const RootGeo& g, const double* __restrict__ pl, XO xo) {
  constexpr const ShapeProg& sh = kShapes[SID];
  static_assert(sh.banks <= 1, "one deferred subtree at a time");
  double factor = 1;
  branch_maps<SID, 0, PEV>(cd, eb, rec, g.msq[0], g.msq[1], g.lam, g.xphi, g.ct, xo, factor);
  double G[16], cur_msq = 0, cur_p = 0;
  math::Divisor cur_m{};
  double bank[16], bank_msq = 0, bank_p = 0;
  static_for<1, sh.n_nodes>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    constexpr ShapeNode N = sh.node[i];
    constexpr bool on_root = N.parent == 0;
    if constexpr (on_root) {
      constexpr int slot = sh.node[0].node0 == i ? 0 : 1;
      root_frame(G, g);
      cur_msq = g.msq[slot];
      cur_m = g.m[slot];
      cur_p = slot == 0 ? g.pk : -g.pk;
    } else if constexpr (sh.node[i - 1].desc < 0) {   // the subtree deferred below the root
#pragma unroll
      for (int j = 0; j < 16; j++) G[j] = bank[j];
      cur_msq = bank_msq; cur_p = bank_p;
      math::sqrt_phys(cur_msq, cur_m);
    }
    double q0[4], q1[4];
    daughter_sum<SID, i, 0>(outs, pl, q0);
    daughter_sum<SID, i, 1>(outs, pl, q1);
    const double msq0 = q0[0] * q0[0] - q0[1] * q0[1] - q0[2] * q0[2] - q0[3] * q0[3];
    const double msq1 = q1[0] * q1[0] - q1[1] * q1[1] - q1[2] * q1[2] - q1[3] * q1[3];
    const Decay dk = decay(math::divisor(cur_msq), cur_m, cur_p, msq0, msq1);
    double v[3];
    boost_back<on_root>(G, math::sqrt_phys(1 + dk.bg * dk.bg), dk.bg, q0, v);
    const Dir dr = direction(v[0], v[1], v[2]);
    branch_maps<SID, i, PEV>(cd, eb, rec, msq0, msq1, dk.lam, dr.xphi, dr.ct, xo, factor);
    if constexpr (!N.leaf0 || !N.leaf1) {
      if constexpr (on_root) rotate_back_root(G, dr.ct, dr.st, dr.cp, dr.sp);
      else rotate_back(G, dr.ct, dr.st, dr.cp, dr.sp);
      if constexpr (N.push >= 0) {
#pragma unroll
        for (int j = 0; j < 16; j++) bank[j] = G[j];
        bank_msq = N.push == 0 ? msq0 : msq1;
        bank_p = N.push == 0 ? dk.pk : -dk.pk;
      }
      cur_msq = N.desc == 0 ? msq0 : msq1;
      math::sqrt_phys(cur_msq, cur_m);
      cur_p = N.desc == 0 ? dk.pk : -dk.pk;
    }
  });
  return factor;
}

// ---- shared branches (trees of up to four final-state particles) ---------------------------
//
// Below the root the same holds branch by branch: what a branch computes from the event depends on
// its ancestors' final-state particles and daughter order, its own daughters' and their
// association, and not on any map.  The host orders the channels by the branches of their trees, root
// first, and marks in each step which branches differ from the last ones evaluated
// (InvStep::eval); the others keep their numbers, and the channel only applies its maps.  The 120
// channels of random 2->4 trees evaluate 30 roots and 129 branches instead of 240 (680 VALU
// instructions per event and channel instead of 897).  Where few branches repeat, the tests keep the
// compiler from interleaving a branch's evaluation with the maps and cost more than they save (the
// three 2->4 resonance channels, which share nothing: 134 against 120 us for 1e6 events when the branches
// were first shared), so inverse_walk runs, which also leaves out the generating channel's branches.

// What a branch below the root leaves behind: msq of its internal daughter (if any), sqrt(lambda) /
// msq, the first daughter's angles, and what its daughters' frame is formed from.
struct BranchGeo {
  double msqi, lam, xphi, ct, st, cp, sp, bg, gm, pk;
};

// Geometry of branch I >= 1 of shape SID from the root's and, for a branch below branch 1, branch 1's.
template <int SID, int I>
__device__ __forceinline__ BranchGeo branch_geometry(uint64_t outs, const RootGeo& g, const BranchGeo& up,
                                                     const double* __restrict__ pl) {
  constexpr ShapeNode N = kShapes[SID].node[I];
  constexpr ShapeNode P = kShapes[SID].node[N.parent < 0 ? 0 : N.parent];
  constexpr int slot = P.node0 == I ? 0 : 1;   // which daughter of its parent the branch is
  double q0[4], q1[4], G[16], v[3];
  daughter_sum<SID, I, 0>(outs, pl, q0);
  daughter_sum<SID, I, 1>(outs, pl, q1);
  const double msq0 = q0[0] * q0[0] - q0[1] * q0[1] - q0[2] * q0[2] - q0[3] * q0[3];
  const double msq1 = q1[0] * q1[0] - q1[1] * q1[1] - q1[2] * q1[2] - q1[3] * q1[3];
  root_frame(G, g);
  Decay dk;
  if constexpr (N.parent == 0) {
    // (the reciprocals of the root's two masses, kept from one branch to the next, took 16 bytes of scratch)
    dk = decay(g.msq[slot], g.m[slot].d, slot == 0 ? g.pk : -g.pk, msq0, msq1);
  } else {
    boost_back<true>(G, up.gm, up.bg, q0, v);
    rotate_back_root(G, up.ct, up.st, up.cp, up.sp);
    math::Divisor m;
    math::sqrt_phys(up.msqi, m);
    dk = decay(math::divisor(up.msqi), m, slot == 0 ? up.pk : -up.pk, msq0, msq1);
  }
  BranchGeo r;
  r.gm = math::sqrt_phys(1 + dk.bg * dk.bg);
  boost_back<N.parent == 0>(G, r.gm, dk.bg, q0, v);
  const Dir dr = direction(v[0], v[1], v[2]);
  r.msqi = !N.leaf0 ? msq0 : msq1;
  r.pk = dk.pk; r.lam = dk.lam; r.bg = dk.bg;
  r.xphi = dr.xphi; r.ct = dr.ct; r.st = dr.st; r.cp = dr.cp; r.sp = dr.sp;
  return r;
}

// As inverse_walk, with the branches that `eval` marks evaluated and the others as they are; for the
// generating channel (own) nothing else.
template <int SID, bool PEV, class XO>
__device__ __forceinline__ double inverse_shared(const ChannelDesc& cd, const EvBeams& eb, const Records& rec,
                                                 uint64_t outs, int eval, bool own, const RootGeo& g, BranchGeo& g1,
                                                 BranchGeo& g2, const double* __restrict__ pl, XO xo) {
  constexpr const ShapeProg& sh = kShapes[SID];
  static_assert(sh.n_nodes <= 3, "trees of up to four final-state particles");
  if constexpr (sh.n_nodes > 1) {
    if (eval & 2) g1 = branch_geometry<SID, 1>(outs, g, g1, pl);
  }
  if constexpr (sh.n_nodes > 2) {
    if (eval & 4) g2 = branch_geometry<SID, 2>(outs, g, g1, pl);
  }
  double factor = 1;
  if (own) return factor;
  branch_maps<SID, 0, PEV>(cd, eb, rec, g.msq[0], g.msq[1], g.lam, g.xphi, g.ct, xo, factor);
  static_for<1, sh.n_nodes>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    const BranchGeo& b = i == 1 ? g1 : g2;
    branch_maps<SID, i, PEV>(cd, eb, rec, b.msqi, b.msqi, b.lam, b.xphi, b.ct, xo, factor);
  });
  return factor;
}

// The inverse of one event into the channel of program `prog` from its root group's geometry `g`,
// the tree's structure read from the program: the randoms go to xo[0..n_x), returns the factor.  No
// branch has a friend.  `cd` is any channel of the process (only what its channels share is read).
template <bool PEV, class XO>
__device__ __forceinline__ double inverse_channel(const ChannelDesc& cd, const EvBeams& eb,
                                                  const NodeCmd* __restrict__ prog, const RootGeo& g,
                                                  const double* __restrict__ pl, int S, double* bank, int B,
                                                  XO xo) {
  double factor = 1;
  // the root: this channel's maps of the shared numbers
  auto map_msq = [&](const NodeCmd& nc, int d, double msq) {
    double x, f;
    if constexpr (PEV) x_from_msq(child_at(nc.k[d], eb.sqrts, eb.s, cd.m_tot), msq, eb.s, x, f);
    else x_from_msq(nc.k[d], msq, eb.s, x, f);
    xo[nc.k[d].xi] = x;
    factor *= f;
  };
  auto map_angles = [&](const NodeCmd& nc, bool root, double xphi, double ct) {
    xo[nc.x_phi] = xphi;
    double x, f, m_max, b0 = nc.b0, b1 = nc.b1;
    if constexpr (PEV) node_at(nc, root, eb, cd.m_tot, m_max, b0, b1);
    x_from_ct(nc.ct_kind, ct, b0, b1, x, f);
    xo[nc.x_phi + 1] = x;
    factor *= f;
  };
#pragma unroll
  for (int d = 0; d < 2; d++)
    if (!prog[0].k[d].leaf) map_msq(prog[0], d, g.msq[d]);
  factor *= g.lam;
  map_angles(prog[0], true, g.xphi, g.ct);
  if (cd.n_nodes == 1) return factor;

  // the root's frame, and the daughter the walk descends into
  double G[16];
  root_frame(G, g);
  const int rdesc = prog[0].desc;
  double cur_msq = rdesc == 0 ? g.msq[0] : g.msq[1], cur_m = rdesc == 0 ? g.m[0].d : g.m[1].d, cur_p = rdesc == 0 ? g.pk : -g.pk;
  bool root_pending = prog[0].push >= 0;
  int depth = 0;   // save-bank entries of subtrees deferred below the root

  for (int i = 1; i < cd.n_nodes; ++i) {
    const NodeCmd& nc = prog[i];
    double q0[4], q1[4];
    branch_sum(pl, S, cd.n_out, nc.k[0], q0);
    branch_sum(pl, S, cd.n_out, nc.k[1], q1);
    const double msq0 = q0[0] * q0[0] - q0[1] * q0[1] - q0[2] * q0[2] - q0[3] * q0[3];
    const double msq1 = q1[0] * q1[0] - q1[1] * q1[1] - q1[2] * q1[2] - q1[3] * q1[3];
#pragma unroll
    for (int d = 0; d < 2; d++)
      if (!nc.k[d].leaf) map_msq(nc, d, d == 0 ? msq0 : msq1);
    const Decay dk = decay(cur_msq, cur_m, cur_p, msq0, msq1);
    const double pk = dk.pk, bg = dk.bg;
    factor *= dk.lam;

    const double gm = math::sqrt_phys(1 + bg * bg);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const double r0 = G[j], r3 = G[12 + j];
      G[j] = gm * r0 - bg * r3;
      G[12 + j] = -bg * r0 + gm * r3;
    }
    const double v0 = G[4] * q0[0] + G[5] * q0[1] + G[6] * q0[2] + G[7] * q0[3];
    const double v1 = G[8] * q0[0] + G[9] * q0[1] + G[10] * q0[2] + G[11] * q0[3];
    const double v2 = G[12] * q0[0] + G[13] * q0[1] + G[14] * q0[2] + G[15] * q0[3];
    const Dir dr = direction(v0, v1, v2);
    map_angles(nc, false, dr.xphi, dr.ct);
    rotate_back(G, dr.ct, dr.st, dr.cp, dr.sp);

    const int push = nc.push, desc = nc.desc;
    if (push >= 0) {
      const double mp = push == 0 ? msq0 : msq1;
      double* b = bank + kInvBankWords * depth * B;
#pragma unroll
      for (int j = 0; j < 16; j++) b[j * B] = G[j];
      b[16 * B] = mp;
      b[17 * B] = math::sqrt_phys(mp);
      b[18 * B] = push == 0 ? pk : -pk;
      depth++;
    }
    if (desc >= 0) {
      cur_msq = desc == 0 ? msq0 : msq1;
      cur_m = math::sqrt_phys(cur_msq);
      cur_p = desc == 0 ? pk : -pk;
    } else if (depth > 0) {
      depth--;
      const double* b = bank + kInvBankWords * depth * B;
#pragma unroll
      for (int j = 0; j < 16; j++) G[j] = b[j * B];
      cur_msq = b[16 * B];
      cur_m = b[17 * B];
      cur_p = b[18 * B];
    } else if (root_pending) {
      // the subtree the root deferred: the root's frame again, re-formed bit for bit
      root_pending = false;
      const int rp = 1 - rdesc;
      root_frame(G, g);
      cur_msq = rp == 0 ? g.msq[0] : g.msq[1];
      cur_m = rp == 0 ? g.m[0].d : g.m[1].d;
      cur_p = rp == 0 ? g.pk : -g.pk;
    }
  }
  return factor;
}

// Shared roots (processes without friends): the channels in the order of `steps`, a root evaluated
// where a group starts.  NOUT: the final-state particles of the process, whose channels run the walks
// specialised per tree shape; 0 for the walk that reads its structure from the program (larger
// trees, and those of five and six with per-event beams).  SHARE: inverse_shared.  WPE: waves per SIMD
// the register allocation aims at (0: the compiler's choice).
//
// Bound by FP64 issue and latency.  Every wavefront works alone, without barriers, on one unit: 64
// events of a tile times one of n_chunks ranges of `steps`, so that a batch of few events still
// gives every SIMD its waves (the launch picks n_chunks); all units of one range come before the next
// range's, so that the waves of a CU mostly read the same records and run the same code (16 channels
// of 2->6 trees 157 against 168 us for 1e5 events, 120 2->4 channels equal).  Its lanes exchange data
// only through the wave's own randoms table.  1e6 events x 3 channels: 102 us (116 with each constant
// loaded where it is used), the vector units 60% busy; 2e5 x 120: 0.69 ms cold, the clock falling under a
// sustained load (0.80), 75% busy; 1e5 x 16 of 2->6: 146 us, 51% busy (310 on the walk that reads its
// structure from the program, whose LDS bank held it to one wave per SIMD).
// LDS per wave: the momenta column (4 n_out rows of 64 doubles), the generic walk's save banks of
// subtrees deferred below the root (19 rows of 64 doubles per level), then the randoms table of the
// channel being inverted (n_x rows of kInvRow doubles).
constexpr int kInvRow = 68;   // lanes that read one another's columns meet different LDS banks

// LDS of one wave, in doubles.
__host__ __device__ inline int inverse_wave_words(int n_out, int n_x, int rest_banks) {
  return 64 * (4 * n_out + kInvBankWords * rest_banks) + kInvRow * n_x;
}

// The wave's randoms table to rows [0, cnt) of dst [..][n_x], one contiguous run of streaming
// stores: 16-byte words where rows are even and dst is aligned.
template <int NX>
__device__ __forceinline__ void store_rows(const double* __restrict__ xs, int cnt, int n_x_rt, bool aligned,
                                           gdouble* __restrict__ dst) {
  const int lane = (int)threadIdx.x & 63;
  if constexpr (NX > 0 && NX % 2 == 0) {
    if (aligned) {
      gdouble2* d2 = (gdouble2*)dst;
#pragma unroll
      for (int u = 0; u < NX / 2; u++) {   // word w: doubles 2 w and 2 w + 1, of one row
        const int w = lane + 64 * u, r = 2 * w / NX, k = 2 * w - r * NX;
        if (cnt == 64 || r < cnt) {
          dvec2 v;
          v.x = xs[k * kInvRow + r];
          v.y = xs[(k + 1) * kInvRow + r];
          __builtin_nontemporal_store(v, d2 + w);
        }
      }
      return;
    }
  }
  const int n_x = NX > 0 ? NX : n_x_rt;
  int r = lane / n_x, k = lane - r * n_x;
  const int dr = 64 / n_x, dk = 64 - dr * n_x;
  for (int q = lane; q < cnt * n_x; q += 64) {
    __builtin_nontemporal_store(xs[k * kInvRow + r], dst + q);
    r += dr;
    k += dk;
    if (k >= n_x) { k -= n_x; r++; }
  }
}

// Lanes read LDS words that other lanes of the wave wrote before (the accesses of one wave stay in
// order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Calls f(integral_constant<int, shape>) for a shape of [LO, HI).
template <int LO, int HI, class F>
__device__ __forceinline__ void for_shape(int shape, F&& f) {
  if constexpr (HI - LO == 1) {
    f(std::integral_constant<int, LO>{});
  } else {
    constexpr int MID = (LO + HI) / 2;
    if (shape < MID) for_shape<LO, MID>(shape, f);
    else for_shape<MID, HI>(shape, f);
  }
}
constexpr int first_shape(int n_out) { return n_out == 2 ? 0 : n_out == 3 ? 1 : n_out == 4 ? 3 : n_out == 5 ? 8 : 22; }
constexpr bool shapes_of(int n_out) {
  for (int k = 0; k < kNumShapes; k++)
    if ((kShapes[k].n_out == n_out) != (k >= first_shape(n_out) && k < (n_out == 6 ? kNumShapes : first_shape(n_out + 1))))
      return false;
  return true;
}
static_assert(shapes_of(2) && shapes_of(3) && shapes_of(4) && shapes_of(5) && shapes_of(6), "shapes by n_out");

template <bool PEV, int NOUT, bool SHARE, int WPE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE))) void inverse_kernel_shared(
    const TileDesc* __restrict__ tiles, int n_units, int n_sub, int n_chunks, const SegDesc* __restrict__ segs,
    const InvSeg* __restrict__ isegs, const InvStep* __restrict__ steps, const ChannelDesc* __restrict__ chans,
    const NodeCmd* __restrict__ nodes, const InvNode* __restrict__ maps, int n_ch, int n_out_rt, int n_x_rt,
    int64_t n_rows, int rest_banks, int aligned, double* __restrict__ factors, double* __restrict__ x_out) {
  constexpr int NX = NOUT > 0 ? 3 * NOUT - 4 : 0;
  const int n_x = NX > 0 ? NX : n_x_rt, n_out = NOUT > 0 ? NOUT : n_out_rt;
  const int lane = (int)threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int u = (int)blockIdx.x * ((int)blockDim.x >> 6) + wave;
  if (u >= n_units) return;
  const int n_us = n_units / n_chunks, chunk = u / n_us, us = u - chunk * n_us;
  const int t = us / n_sub, base = 64 * (us - t * n_sub);
  const TileDesc td = tiles[t];
  if (base >= td.count) return;
  const SegDesc sd = segs[td.seg];
  const InvSeg is = isegs[td.seg];
  double* ps = inv_lds + wave * inverse_wave_words(n_out, n_x, rest_banks);
  double* pl = ps + lane;
  double* bank = ps + 64 * 4 * n_out + lane;
  double* xs = ps + 64 * (4 * n_out + kInvBankWords * rest_banks);
  const XColumn xl{xs + lane, kInvRow};
  const int cnt = min(64, td.count - base);
  const bool valid = lane < cnt;   // lanes past the end stage the last event and store nothing
  const int64_t e = td.e0 + base + (valid ? lane : cnt - 1);
  const int64_t row = is.row0 + e;
  const ChannelDesc cd = chans[0];   // only what all channels of the process share is read
  EvBeams eb;
  if constexpr (PEV) eb = event_beams(cd, as_global(sd.e1)[e], as_global(sd.e2)[e]);
  else eb = fixed_beams(cd);
  gdouble* f_row = as_global(factors) + row * n_ch;
  gdouble* x_rows = as_global(x_out) + (is.row0 + td.e0 + base) * n_x;
  // the generating channel's slot: the forward pass's factor, and its randoms, whose rows lie as
  // x_out's do (loaded here, beside the momenta, and stored below)
  const gdouble* x_own = as_global(sd.x) + (td.e0 + base) * n_x;
  gdouble* x_dst = x_rows + (int64_t)is.own * n_rows * n_x;
  const int n_own = chunk == 0 ? cnt * n_x : 0;
  double xo[NX > 0 ? NX : 1], f_own = 0;
  if constexpr (NX > 0) {
#pragma unroll
    for (int q = 0; q < NX; q++)
      if (lane + 64 * q < n_own) xo[q] = x_own[lane + 64 * q];
    if (n_own > 0) f_own = as_global((const double*)sd.factor)[e];
  }
  const gdouble* pe = as_global((const double*)sd.p) + e * 4 * n_out;
  for (int j = 0; j < n_out; j++) {
    double q0 = pe[4 * j], q1 = pe[4 * j + 1], q2 = pe[4 * j + 2], q3 = pe[4 * j + 3];
    if (eb.bg_lab != 0) {
      const double a = eb.g_lab * q0 - eb.bg_lab * q3;
      const double b = -eb.bg_lab * q0 + eb.g_lab * q3;
      q0 = a; q3 = b;
    }
    pl[(4 * j) * 64] = q0; pl[(4 * j + 1) * 64] = q1; pl[(4 * j + 2) * 64] = q2; pl[(4 * j + 3) * 64] = q3;
  }
  if constexpr (NX > 0) {
#pragma unroll
    for (int q = 0; q < NX; q++)
      if (lane + 64 * q < n_own) __builtin_nontemporal_store(xo[q], x_dst + lane + 64 * q);
  } else {
    for (int q = lane; q < n_own; q += 64) __builtin_nontemporal_store(x_own[q], x_dst + q);
    if (n_own > 0) f_own = as_global((const double*)sd.factor)[e];
  }
  if (n_own > 0 && valid) f_row[is.own] = f_own;
  const int k_begin = (int)((int64_t)n_ch * chunk / n_chunks), k_end = (int)((int64_t)n_ch * (chunk + 1) / n_chunks);
  math::Divisor by_s = math::divisor(eb.s), by_sqrts = math::divisor(eb.sqrts);
  if constexpr (!PEV) {   // the same for all lanes: in scalar registers
    by_s.r = uniform(by_s.r);
    by_sqrts.r = uniform(by_sqrts.r);
  }
  RootGeo geo{};
  BranchGeo g1, g2;
  for (int k = k_begin; k < k_end; k++) {
    const InvStep st = steps[k];
    const int c = st.channel;
    const int eval = k == k_begin ? ~0 : st.eval;
    const bool own = c == is.own;
    double f = 0;
    if constexpr (NOUT == 0) {
      const NodeCmd* prog = nodes + st.node0;
      if (eval & 1) {
        double q0[4], q1[4];
        branch_sum(pl, 64, n_out, prog[0].k[0], q0);
        branch_sum(pl, 64, n_out, prog[0].k[1], q1);
        geo = root_geometry(q0, q1, prog[0].k[0].leaf, prog[0].k[1].leaf, by_s, by_sqrts);
      }
      if (!own) f = inverse_channel<PEV>(cd, eb, prog, geo, pl, 64, bank, 64, xl);
    } else {
      const Records rec{nodes + st.node0, maps + st.node0};
      for_shape<first_shape(NOUT), NOUT == 6 ? kNumShapes : first_shape(NOUT + 1)>(st.shape, [&](auto sid) {
        constexpr int SID = decltype(sid)::value;
        if (eval & 1) geo = root_of<SID>(st.outs, by_s, by_sqrts, pl);
        if constexpr (SHARE) f = inverse_shared<SID, PEV>(cd, eb, rec, st.outs, eval, own, geo, g1, g2, pl, xl);
        else if (!own) f = inverse_walk<SID, PEV>(cd, eb, rec, st.outs, geo, pl, xl);
      });
    }
    if (own) continue;
    if (valid) f_row[c] = f;
    wave_sync();
    store_rows<NX>(xs, cnt, n_x, aligned != 0, x_rows + (int64_t)c * n_rows * n_x);
    wave_sync();
  }
}

using SharedKernel = void (*)(const TileDesc*, int, int, int, const SegDesc*, const InvSeg*, const InvStep*,
                              const ChannelDesc*, const NodeCmd*, const InvNode*, int, int, int, int64_t, int, int, double*,
                              double*);
// The specialised kernels of five and six final-state particles (a translation unit each).
SharedKernel shared_kernel_5();
SharedKernel shared_kernel_6();

}  // namespace inv
}  // namespace gphs
