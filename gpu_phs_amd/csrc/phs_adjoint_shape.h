// The adjoint of one event specialised for a compile-time tree shape (phs_shapes.h), fixed beams: the
// computation of phs_adjoint.h (event_adjoint) with both sweeps unrolled, and the kernel that runs it
// (instantiated per range of shapes in phs_adjoint.hip and phs_adjoint_5.hip, _6.hip and _6_loss.hip).
//
// What bounds it: FP64 instruction issue and, at two waves per SIMD, the latencies between the
// instructions; the tape in LDS decides how many waves a CU holds.  So
//  - the root is a rotation (its parent boost is the identity and its p_decay 0): nothing is multiplied by
//    its zeros and ones, and its boost's gamma and beta gamma take no part in the sweep;
//  - the tangent or exponential of every msq map is kept from the forward sweep, in the four words of
//    the tape that the root does not need;
//  - the adjoint of a deferred subtree waits in the tape words of its own branches, which nothing reads
//    after they are reversed: eight words per branch are all the LDS there is (20 KB per wave for five
//    branches, eight waves per CU; 35 KB with a stash and the (M, Gamma) sums in LDS: four waves);
//  - products with structural zeros are left out (masks below): with the built-in loss two of the four rows
//    of every adjoint of a boost;
//  - square roots give the reciprocals too, and a quotient by s or m is a product.
// Measured, the generic adjoint or the one specialised without these, and this one: 2 x 10^5 events of 16
// channels of 2 -> 6, given cotangents: 101 -> 52 us (3,980 -> 3,090 vector instructions per wave; two waves
// per SIMD, which the tape allows, are two rounds of 3,164 waves); 10^6 events of 3 channels of 2 -> 4 with
// the built-in loss: 97 -> 70 us (1,820 -> 1,380 instructions, 196 -> 161 registers and so three waves per
// SIMD), with given cotangents 118 -> 96 us; 10^6 events of five particles, built-in loss: 247 -> 119 us; of
// three: 69 -> 44 us.
#pragma once
#include <hip/hip_runtime.h>

#include <utility>

#include "phs_adjoint.h"
#include "phs_kernels.h"
#include "phs_shapes.h"

namespace gphs {

namespace adj {

// Structural zeros, as masks over the entries 4 row + column of a matrix.  With the built-in loss (LM = 1) the
// cotangents of energies and longitudinal momenta are zero, and so are rows 0 and 3 of every adjoint of a
// boost; a final-state daughter reads columns 0 and 3 of its parent's; the root reads the adjoint of its
// rotation only; and L1 has zeros of its own.
constexpr unsigned kRowsOf[2] = {0xffff, 0x0ff0};   // by loss mode
constexpr unsigned kLeafCols = 0x9999;
constexpr unsigned kRootEntries = 1u << 5 | 1u << 6 | 1u << 7 | 1u << 9 | 1u << 10 | 1u << 11 | 1u << 13 | 1u << 15;
constexpr unsigned kL1Row[4] = {0xb, 0xe, 0xe, 0xb};   // non-zero columns of each row of L1
constexpr unsigned kRotCol[4] = {0x1, 0xe, 0x6, 0xe};  // non-zero rows of each column of the root's rotation

// The non-zeros of what branch j >= 1 hands to its parent (G L1^T) and of the adjoint G of its own boost.
template <int SID, int LM>
constexpr unsigned handed_mask(int j);
template <int SID, int LM>
constexpr unsigned adjoint_mask(int i) {
  const ShapeNode sn = kShapes[SID].node[i];
  unsigned m = sn.leaf0 || sn.leaf1 ? kLeafCols & kRowsOf[LM] : 0;
  if (!sn.leaf0) m |= handed_mask<SID, LM>(sn.node0);
  if (!sn.leaf1) m |= handed_mask<SID, LM>(sn.node1);
  return i == 0 ? m & kRootEntries : m;
}
template <int SID, int LM>
constexpr unsigned handed_mask(int j) {
  const unsigned g = adjoint_mask<SID, LM>(j);
  unsigned m = 0;
  for (int q = 0; q < 16; q++)
    if ((g >> (q & 12)) & kL1Row[q & 3]) m |= 1u << q;
  return kShapes[SID].node[j].parent == 0 ? m & kRootEntries : m;
}
constexpr int bits(unsigned m) { return __builtin_popcount(m); }

// Branch i is a deferred one (its predecessor has no daughter that is visited next).
template <int SID>
constexpr bool popped(int i) { return i > 0 && kShapes[SID].node[i > 0 ? i - 1 : 0].desc < 0; }

// A deferred subtree hands its parent the non-zero entries and the adjoints of msq and p_decay.  The words
// that do not fit the tape of its own branches are in registers.
template <int SID, int LM>
constexpr int extra_words() {
  int extra = 0;
  const ShapeProg& sh = kShapes[SID];
  for (int j = 1; j < sh.n_nodes; j++)
    if (popped<SID>(j)) {
      const int over = bits(handed_mask<SID, LM>(j)) + 2 - 8 * (sh.n_nodes - j);
      extra = over > extra ? over : extra;
    }
  return extra;
}

// sum of a[k] b[k] over the k in MASK, in order (0 if there are none)
template <unsigned MASK>
__device__ __forceinline__ double dot(const double (&a)[4], const double (&b)[4]) {
#pragma clang fp contract(fast)
  double acc = 0;
#pragma unroll
  for (int k = 0; k < 4; k++)
    if (MASK >> k & 1) acc = MASK & ((1u << k) - 1) ? __builtin_fma(a[k], b[k], acc) : a[k] * b[k];
  return acc;
}

// sqrt(x) and its reciprocal for x > 0: the estimate that the square root has, refined as recip refines its
// own (two instructions instead of a reciprocal's five, the first of which takes as long as four).
__device__ __forceinline__ double sqrt_recip(double x, double& inv) {
  const double r = math::sqrt_phys(x);
  double h = __builtin_amdgcn_rsq(x);
  h = __builtin_fma(h, __builtin_fma(-r, h, 1.0), h);
  inv = __builtin_fma(h, __builtin_fma(-r, h, 1.0), h);
  return r;
}

// Eight words per branch, lane-strided (one wavefront per workgroup: consecutive lanes, consecutive words).
template <int SID, int LM>
struct ShapeTape {
  static constexpr int kNodes = kShapes[SID].n_nodes;
  static_assert(kNodes <= 5, "the root's four free words hold the maps of at most four internal daughters");
  double* base;
  double extra[extra_words<SID, LM>() > 0 ? extra_words<SID, LM>() : 1];
  __device__ __forceinline__ double& word(int w) { return base[w * 64]; }
  __device__ __forceinline__ double& T(int node, int k) { return word(8 * node + k); }        // gamma, bg, ct, st, cp, sp
  __device__ __forceinline__ double& in(int node, int k) { return word(8 * node + 6 + k); }   // msq, p_decay
  // the root keeps no gamma, bg, msq and p_decay: the map values t (MapEval) of branches 1..4
  __device__ __forceinline__ double& t(int node) { return word(node <= 2 ? node - 1 : 3 + node); }
  // word w of what the subtree of branch j hands to its parent
  __device__ __forceinline__ void put(int j, int w, double v) {
    if (8 * j + w < 8 * kNodes) word(8 * j + w) = v;
    else extra[8 * j + w - 8 * kNodes] = v;
  }
  __device__ __forceinline__ double get(int j, int w) {
    return 8 * j + w < 8 * kNodes ? word(8 * j + w) : extra[8 * j + w - 8 * kNodes];
  }
};

// A map's value from its kept tangent or exponential (the operations of msq_eval); the step maps, which
// keep nothing, are evaluated again.
__device__ __forceinline__ MapEval msq_eval_kept(const ChildCmd& c, double x, double s, double t) {
  MapEval r{0, 0, t, 0, true};
  switch (c.kind) {
    case MK_BREIT_WIGNER: {
      const double z = (1 - x) * c.a0 + x * c.a1;
      r.in = (-kPi / 2 < z) && (z < kPi / 2);
      r.msq = r.in ? c.m * (c.m + c.w * t) : 0.0;
      r.f = r.in ? c.a2 * (1 + t * t) : 0.0;
      return r;
    }
    case MK_EXP: {
      const double m1 = c.a0 * t;
      r.msq = m1 - c.a0 + c.msq_min;
      r.f = c.a2 * m1;
      return r;
    }
    case MK_TU: {
      const bool lo = x < 0.5;
      r.aux = lo ? 1.0 : -1.0;
      const double m1 = c.a0 * t;
      r.msq = lo ? (m1 - c.a0 + c.msq_min) : (-(m1 - c.a0) + c.msq_max);
      r.f = c.a2 * m1;
      return r;
    }
    default: return msq_eval(c, x, s);
  }
}

// P = product of the boosts of branch A and of its ancestors (phs_adjoint.h parent_boost), for a branch A
// below the root; rot: the root's angles.
template <int SID, int A, class Tape>
__device__ __forceinline__ void boosts_to(Tape& S, const RootRot& rot, double (&P)[16]) {
  if constexpr (A > 0) {
    constexpr int parent = kShapes[SID].node[A].parent;
    boosts_to<SID, parent>(S, rot, P);
    const double g = S.T(A, 0), bg = S.T(A, 1), ct = S.T(A, 2), st = S.T(A, 3), cp = S.T(A, 4), sp = S.T(A, 5);
    if constexpr (parent == 0) compose_on_root<false>(P, rot, g, bg, ct, st, cp, sp);
    else compose_l1(P, g, bg, ct, st, cp, sp);
  }
}

// f(0), ..., f(N - 1) (or N - 1 first) with compile-time arguments.
template <class F, int... I>
__device__ __forceinline__ void for_each(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <class F, int... I>
__device__ __forceinline__ void for_each_reversed(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, (int)sizeof...(I) - 1 - I>{}), ...);
}

// event_adjoint (phs_adjoint.h) for tree shape SID.
// xr: the event's randoms (registers); xg: the same in memory, from where the reverse sweep loads each
// branch's again (held to the end, they took the registers that hold the sweep at two waves per SIMD).
template <int SID, int LM, class GPar, class XR>
__device__ __forceinline__ bool shape_adjoint(const ChannelDesc& cd, const EvBeams& eb, const NodeCmd* __restrict__ prog,
                                              const XR& xr, const gdouble* xg, const double* __restrict__ gp, double gf_in,
                                              double* __restrict__ p_out, double* f_out, double* loss_out,
                                              double* __restrict__ gx, GPar& gpar, ShapeTape<SID, LM>& S) {
  constexpr int N = kShapes[SID].n_nodes;
  const double s = eb.s;
  // ---------------- forward, with the tape
  double M[16] = {1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1};
  double cur_msq = s, cur_m = eb.sqrts, cur_p = 0, F = 1, S2 = 0;
  bool ok = true;
  RootRot rot{};
  auto fwd_branch = [&](auto branch) {
    constexpr int i = branch.value;
    constexpr ShapeNode sn = kShapes[SID].node[i];
    constexpr bool leaf[2] = {sn.leaf0 != 0, sn.leaf1 != 0};
    constexpr int xi[2] = {sn.xi0, sn.xi1}, child[2] = {sn.node0, sn.node1};
    constexpr bool root = i == 0, on_root = sn.parent == 0;
    const NodeCmd nc = load_branch(prog + i, leaf[0], leaf[1]);
    if constexpr (popped<SID>(i)) {   // the deferred branch: its boost is re-formed
      rot = RootRot{S.T(0, 2), S.T(0, 3), S.T(0, 4), S.T(0, 5)};
      boosts_to<SID, sn.parent>(S, rot, M);
      cur_msq = S.in(i, 0); cur_p = S.in(i, 1); cur_m = math::sqrt_phys(cur_msq);
    }
    double msq[2], f[2], mk[2];
#pragma unroll
    for (int c = 0; c < 2; c++) {
      if (leaf[c]) { msq[c] = nc.k[c].msq_leaf; f[c] = 1; mk[c] = nc.k[c].m_leaf; }
      else {
        const MapEval r = msq_eval(nc.k[c], xr[xi[c]], s);
        msq[c] = r.msq; f[c] = r.f; mk[c] = math::sqrt_phys(r.msq);
        S.t(child[c]) = r.t;
      }
    }
    const double m = cur_m;
    const double lda = (cur_msq - msq[0] - msq[1]) * (cur_msq - msq[0] - msq[1]) - 4 * msq[0] * msq[1];
    ok = ok && (lda > 0 && m > mk[0] + mk[1] && m <= nc.m_max);
    // 1 / m serves pk = sl / (2 m) and bg = p / m (math::quot(a, b) is a times this reciprocal)
    const double sl = math::sqrt_phys(lda), rm = math::recip(m), pk = sl * (0.5 * rm);
    F *= f[0] * f[1] * math::quot(sl, cur_msq);
    const double bg = root ? 0.0 : m > 0 ? cur_p * rm : 0.0, g = root ? 1.0 : math::sqrt_phys(1 + bg * bg);
    double sp, cp;
    math::sincos_turns(xr[sn.xphi], sp, cp);
    const CtEval ce = ct_eval(nc.ct_kind, xr[sn.xphi + 1], nc.b0, nc.b1);
    F *= ce.f;
    if (root) rot = RootRot{ce.ct, ce.st, cp, sp};
    else if (on_root) compose_on_root<false>(M, rot, g, bg, ce.ct, ce.st, cp, sp);
    else compose_l1(M, g, bg, ce.ct, ce.st, cp, sp);
    if (!root) { S.T(i, 0) = g; S.T(i, 1) = bg; }
    S.T(i, 2) = ce.ct; S.T(i, 3) = ce.st; S.T(i, 4) = cp; S.T(i, 5) = sp;
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const double pc = c == 0 ? pk : -pk;
      if (!leaf[c]) {
        S.in(child[c], 0) = msq[c];
        S.in(child[c], 1) = pc;
        continue;
      }
      const double E = nc.k[c].msq_leaf == 0 ? fabs(pc) : math::sqrt_phys(nc.k[c].msq_leaf + pc * pc);
      double q0 = root ? E : __builtin_fma(M[3], pc, M[0] * E);
      const double q1 = root ? ce.st * cp * pc : __builtin_fma(M[7], pc, M[4] * E);
      const double q2 = root ? ce.st * sp * pc : __builtin_fma(M[11], pc, M[8] * E);
      double q3 = root ? ce.ct * pc : __builtin_fma(M[15], pc, M[12] * E);
      if (LM == 0 && eb.bg_lab != 0) {
        const double b0 = eb.g_lab * q0 + eb.bg_lab * q3, b3 = eb.bg_lab * q0 + eb.g_lab * q3;
        q0 = b0; q3 = b3;
      }
      S2 += q1 * q1 + q2 * q2;
      if (p_out) {
        double* o = p_out + 4 * nc.k[c].out;
        o[0] = q0; o[1] = q1; o[2] = q2; o[3] = q3;
      }
    }
    if constexpr (sn.desc >= 0) {
      cur_msq = msq[sn.desc]; cur_m = mk[sn.desc]; cur_p = sn.desc == 0 ? pk : -pk;
    }
  };
  for_each(fwd_branch, std::make_integer_sequence<int, N>{});
  *f_out = F;
  const math::Divisor by_s = math::divisor(s);
  if (loss_out) *loss_out = ok && LM == 1 ? math::divide(F * S2, by_s) : 0.0;
  if (!ok) {
#pragma unroll
    for (int k = 0; k < kShapes[SID].n_x; k++) gx[k] = 0;
    return false;
  }
  {
  // derivatives only from here on: products and sums may fuse (the outputs above are final)
#pragma clang fp contract(fast)
  const double gF = LM == 1 ? S2 * by_s.r : gf_in;
  const double W = gF * F;           // adjoint of log(term) for every factor of the product
  const double F2s = F * 2 * by_s.r;   // (LM = 1) d loss / d q1 = F2s q1, and the same for q2

  // ---------------- reverse sweep (an ok event: every m and lambda is positive)
  double Gc[16];             // adjoint of the parent boost, from the branch just reversed
  double gc_msq = 0, gc_p = 0;
  asm volatile("" : "+v"(xg));   // not the values loaded before
  auto rev_branch = [&](auto branch) {
    constexpr int i = branch.value;
    constexpr ShapeNode sn = kShapes[SID].node[i];
    constexpr bool leaf[2] = {sn.leaf0 != 0, sn.leaf1 != 0};
    constexpr int xi[2] = {sn.xi0, sn.xi1}, child[2] = {sn.node0, sn.node1}, push = sn.push, desc = sn.desc;
    constexpr bool root = i == 0, on_root = sn.parent == 0;
    constexpr unsigned gm = adjoint_mask<SID, LM>(i), rows = kRowsOf[LM];
    const NodeCmd nc = load_branch<true>(prog + i, leaf[0], leaf[1]);
    const double xct = xg[sn.xphi + 1], xk[2] = {xi[0] < 0 ? 0.0 : xg[xi[0] < 0 ? 0 : xi[0]],
                                                xi[1] < 0 ? 0.0 : xg[xi[1] < 0 ? 0 : xi[1]]};
    // cotangents of the final-state daughters' lab momenta: loaded before anything else
    double gq[2][4] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
    if (LM == 0 && gp) {
#pragma unroll
      for (int c = 0; c < 2; c++)
        if (leaf[c])
#pragma unroll
          for (int mu = 0; mu < 4; mu++) gq[c][mu] = as_global(gp)[4 * nc.k[c].out + mu];
    }
    // the adjoint of this branch's boost (entries gm), of its daughters' msq and of pk
    double G[4][4] = {{0}}, g_msq[2] = {0, 0}, g_pk = 0;
    unsigned have = 0;   // entries of G so far (constant, once unrolled)
    auto add = [&](int q, double v) {
      G[q >> 2][q & 3] = have >> q & 1 ? G[q >> 2][q & 3] + v : v;
      have |= 1u << q;
    };
    auto add_product = [&](int q, double u, double v) {
      G[q >> 2][q & 3] = have >> q & 1 ? __builtin_fma(u, v, G[q >> 2][q & 3]) : u * v;
      have |= 1u << q;
    };
    if constexpr (desc >= 0) {
      constexpr unsigned hm = handed_mask<SID, LM>(child[desc]);
#pragma unroll
      for (int q = 0; q < 16; q++)
        if (hm >> q & 1) add(q, Gc[q]);
      g_msq[desc] = gc_msq; g_pk = desc == 0 ? gc_p : -gc_p;
    }
    if constexpr (push >= 0) {
      constexpr int j = child[push];
      constexpr unsigned hm = handed_mask<SID, LM>(j);
#pragma unroll
      for (int q = 0; q < 16; q++)
        if (hm >> q & 1) add(q, S.get(j, bits(hm & ((1u << q) - 1))));
      g_msq[push] = S.get(j, bits(hm));
      g_pk += push == 0 ? S.get(j, bits(hm) + 1) : -S.get(j, bits(hm) + 1);
    }
    const double a = root ? s : S.in(i, 0), p0 = root ? 0.0 : S.in(i, 1);
    double inv_m = 0;
    if constexpr (root) inv_m = math::recip(eb.sqrts);
    else sqrt_recip(a, inv_m);
    const double g = root ? 1.0 : S.T(i, 0), bg = root ? 0.0 : S.T(i, 1), cp = S.T(i, 4), sp = S.T(i, 5);
    const RootRot rr = root ? RootRot{} : RootRot{S.T(0, 2), S.T(0, 3), S.T(0, 4), S.T(0, 5)};
    MapEval r[2];
    double msq[2], f[2];
#pragma unroll
    for (int c = 0; c < 2; c++) {
      if (leaf[c]) { msq[c] = nc.k[c].msq_leaf; f[c] = 1; }
      else {
        r[c] = msq_eval_kept(nc.k[c], xk[c], s, S.t(child[c]));
        msq[c] = r[c].msq; f[c] = r[c].f;
      }
    }
    const double d = a - msq[0] - msq[1];
    double inv_sl;
    const double sl = sqrt_recip(d * d - 4 * msq[0] * msq[1], inv_sl), pk = 0.5 * (sl * inv_m);
    if (!(sl > 0)) inv_sl = 0;   // lambda rounded differently at the threshold
    CtEval ce;
    if (nc.ct_kind == CK_FLAT) {   // sin theta as the forward sweep formed it
      ce.tmp = 2 * (1 - xct);
      ce.ct = 1 - ce.tmp;
      ce.st = S.T(i, 3);
      ce.f = 1;
      ce.e = 0;
      ce.in = true;
      ce.lo = false;
    } else {
      ce = ct_eval(nc.ct_kind, xct, nc.b0, nc.b1);
    }
    // the parent boost P (below the root: 1 (+) its rotation) and columns 0 and 3 of Ma = P L1
    double P[16] = {1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1}, Ma[16];
    if constexpr (root) {
      Ma[0] = 1; Ma[4] = 0; Ma[8] = 0; Ma[12] = 0;
      Ma[3] = 0; Ma[7] = ce.st * cp; Ma[11] = ce.st * sp; Ma[15] = ce.ct;
    } else if constexpr (on_root) {
      P[5] = rr.ct * rr.cp; P[6] = -rr.sp; P[7] = rr.st * rr.cp;
      P[9] = rr.ct * rr.sp; P[10] = rr.cp; P[11] = rr.st * rr.sp;
      P[13] = -rr.st;       P[14] = 0;     P[15] = rr.ct;
      compose_on_root<true>(Ma, rr, g, bg, ce.ct, ce.st, cp, sp);
    } else {
      boosts_to<SID, (root ? 0 : sn.parent)>(S, rr, P);
      compose_l1_to(P, Ma, g, bg, ce.ct, ce.st, cp, sp);
    }

    // final-state daughters: q = Ma[:,0] E + Ma[:,3] pc
#pragma unroll
    for (int c = 0; c < 2; c++) {
      if (!leaf[c]) continue;
      const double pc = c == 0 ? pk : -pk;
      const double E = nc.k[c].msq_leaf == 0 ? fabs(pc) : math::sqrt_phys(nc.k[c].msq_leaf + pc * pc);
      if (LM == 1) {
        gq[c][1] = F2s * (root ? Ma[7] * pc : __builtin_fma(Ma[7], pc, Ma[4] * E));
        gq[c][2] = F2s * (root ? Ma[11] * pc : __builtin_fma(Ma[11], pc, Ma[8] * E));
      } else if (eb.bg_lab != 0) {   // back through the (linear) lab boost
        const double a0 = gq[c][0], a3 = gq[c][3];
        gq[c][0] = eb.g_lab * a0 + eb.bg_lab * a3;
        gq[c][3] = eb.bg_lab * a0 + eb.g_lab * a3;
      }
#pragma unroll
      for (int mu = 0; mu < 4; mu++) {
        if (gm >> (4 * mu) & 1) add_product(4 * mu, gq[c][mu], E);
        if (gm >> (4 * mu + 3) & 1) add_product(4 * mu + 3, gq[c][mu], pc);
      }
      constexpr unsigned col = (rows >> 0 & 1) | (rows >> 4 & 1) << 1 | (rows >> 8 & 1) << 2 | (rows >> 12 & 1) << 3;
      const double c0[4] = {Ma[0], Ma[4], Ma[8], Ma[12]}, c3[4] = {Ma[3], Ma[7], Ma[11], Ma[15]};
      const double gE = dot<col & (root ? 0x1 : 0xf)>(gq[c], c0);
      double gpc = dot<col & (root ? 0xe : 0xf)>(gq[c], c3);
      if (!(root && LM == 1) && E > 0) gpc += math::quot(gE * pc, E);
      g_pk += c == 0 ? gpc : -gpc;
    }
    // Ma = P L1: gP = G L1^T, gL1 = P^T G (structural non-zeros of L1 only)
    const double st = ce.st, ct = ce.ct;
    double gbg = 0, gct, gst, gcp, gsp;
    if constexpr (root) {
      gct = G[1][1] * cp + G[2][1] * sp;
      gst = G[1][3] * cp + G[2][3] * sp;
      gcp = G[1][1] * ct + G[1][3] * st + G[2][2];
      gsp = -G[1][2] + G[2][1] * ct + G[2][3] * st;
      if (LM == 0) { gct += G[3][3]; gst -= G[3][1]; }
    } else {
      const double L[4][4] = {{g, -bg * st, 0, bg * ct}, {0, ct * cp, -sp, st * cp}, {0, ct * sp, cp, st * sp},
                              {bg, -g * st, 0, g * ct}};
      // entry (k, j) of gL1: over the rows of G that can be non-zero in column j and of P in column k
      auto gl = [&](auto ck, auto cj) {
        constexpr int k = ck.value, j = cj.value;
        constexpr unsigned col = (gm >> j & 1) | (gm >> (4 + j) & 1) << 1 | (gm >> (8 + j) & 1) << 2 |
                                 (gm >> (12 + j) & 1) << 3;
        const double pc[4] = {P[k], P[4 + k], P[8 + k], P[12 + k]}, gc[4] = {G[0][j], G[1][j], G[2][j], G[3][j]};
        if constexpr (on_root && k == 0) return col & 1 ? gc[0] : 0.0;
        else return dot<col & (on_root ? kRotCol[k] : 0xf)>(pc, gc);
      };
      constexpr std::integral_constant<int, 0> c0{};
      constexpr std::integral_constant<int, 1> c1{};
      constexpr std::integral_constant<int, 2> c2{};
      constexpr std::integral_constant<int, 3> c3{};
      // columns 1 and 2 of G are zero for a branch of two final-state particles
      constexpr bool inner = !(leaf[0] && leaf[1]), row0 = !on_root || (gm & 0xf) != 0;
      const double g00 = gl(c0, c0), g03 = gl(c0, c3), g13 = gl(c1, c3), g23 = gl(c2, c3), g30 = gl(c3, c0),
                   g33 = gl(c3, c3);
      double gg = g33 * ct;
      gbg = g30;
      gct = g33 * g;
      gst = g13 * cp + g23 * sp;
      gcp = g13 * st;
      gsp = g23 * st;
      if constexpr (row0) {
        gg += g00;
        gbg += g03 * ct;
        gct += g03 * bg;
      }
      if constexpr (inner) {
        const double g01 = gl(c0, c1), g11 = gl(c1, c1), g12 = gl(c1, c2), g21 = gl(c2, c1), g22 = gl(c2, c2),
                     g31 = gl(c3, c1);
        gg -= g31 * st;
        gct += g11 * cp + g21 * sp;
        gst -= g31 * g;
        gcp += g11 * ct + g22;
        gsp += g21 * ct - g12;
        if constexpr (row0) { gbg -= g01 * st; gst -= g01 * bg; }
      }
      gbg += math::quot(gg * bg, g);   // gamma = sqrt(1 + bg^2)
      constexpr unsigned hm = handed_mask<SID, LM>(i);
      for_each([&](auto entry) {
        constexpr int q = entry.value;
        if constexpr (hm >> q & 1) Gc[q] = dot<(gm >> (q & 12)) & kL1Row[q & 3]>(G[q >> 2], L[q & 3]);
      }, std::make_integer_sequence<int, 16>{});
    }
    // phi = 2 pi x
    as_global(gx)[sn.xphi] = (gsp * cp - gcp * sp) * kTwoPi;
    // cos theta map of this branch (its own M through b0, b1)
    const double gfct = ce.f != 0 ? math::quot(W, ce.f) : 0.0;
    double gxc, gb0, gb1;
    ct_eval_adj(nc.ct_kind, xct, nc.b0, nc.b1, ce, gct, gst, gfct, gxc, gb0, gb1);
    as_global(gx)[sn.xphi + 1] = gxc;
    gpar[2 * i] += gb0 * nc.db_dm[0] + gb1 * nc.db_dm[1];
    // bg = p / m; pk = sl / (2 m); factor term f0 f1 sl / a; lambda = d^2 - 4 msq0 msq1, d = a - msq0 - msq1
    const double g_p0 = gbg * inv_m;
    const double g_mnode = -(g_p0 * p0 + g_pk * sl * inv_m * 0.5) * inv_m;
    const double glda = (g_pk * inv_m * 0.5 + W * inv_sl) * inv_sl * 0.5, gd = 2 * d * glda;
    g_msq[0] += -4 * msq[1] * glda - gd;
    g_msq[1] += -4 * msq[0] * glda - gd;
#pragma unroll
    for (int c = 0; c < 2; c++) {   // the msq maps of the internal daughters
      if (leaf[c]) continue;
      const double gfk = f[c] != 0 ? math::quot(W, f[c]) : 0.0;
      double gxk = 0, gM = 0, gW = 0;
      msq_eval_adj(nc.k[c], xk[c], s, r[c], g_msq[c], gfk, gxk, gM, gW);
      as_global(gx)[xi[c]] = gxk;
      gpar[2 * child[c]] += gM;
      gpar[2 * child[c] + 1] += gW;
    }
    // hand the adjoints of this branch's inputs to its parent: of p_decay, and of msq, also through
    // m = sqrt(msq)
    gc_msq = gd - W * inv_m * inv_m + 0.5 * g_mnode * inv_m;
    gc_p = g_p0;
    if constexpr (popped<SID>(i)) {   // in the forward sweep: kept for the parent
      constexpr unsigned hm = handed_mask<SID, LM>(i);
#pragma unroll
      for (int q = 0; q < 16; q++)
        if (hm >> q & 1) S.put(i, bits(hm & ((1u << q) - 1)), Gc[q]);
      S.put(i, bits(hm), gc_msq);
      S.put(i, bits(hm) + 1, gc_p);
    }
  };
  for_each_reversed(rev_branch, std::make_integer_sequence<int, N>{});
  }
  return true;
}

// The sums over the wavefront of v, step by step: the exchanges of all are in flight at once.
template <int N>
__device__ __forceinline__ void wave_sums(double (&v)[N]) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    double other[N];
#pragma unroll
    for (int k = 0; k < N; k++) other[k] = __shfl_xor(v[k], o, 64);
#pragma unroll
    for (int k = 0; k < N; k++) v[k] += other[k];
  }
}

// One 64-event unit: sub-tile `sub` of tile td; its partial parameter sums go to `part`.
template <int SID, int LM>
__device__ __forceinline__ void shape_unit(int sub, const TileDesc& td, const SegDesc& sd, const ChannelDesc& cd,
                                           const NodeCmd* __restrict__ prog, double* __restrict__ part, double* lds) {
  constexpr int kNp = 2 * kShapes[SID].n_nodes, kNx = kShapes[SID].n_x, kNout = kShapes[SID].n_out;
  const int lane = threadIdx.x, end = min(td.count, 64 * (sub + 1));
  double accv[kNp];   // (M, Gamma) of every branch
#pragma unroll
  for (int v = 0; v < kNp; v++) accv[v] = 0;
  if (const int local = 64 * sub + lane; local < end) {
    const int64_t e = td.e0 + local;
    const gdouble* xg = as_global(sd.x) + e * kNx;
    double xv[kNx];
#pragma unroll
    for (int k = 0; k < kNx; k++) xv[k] = xg[k];
    const double* gp = sd.g_p ? sd.g_p + e * (kNout * 4) : nullptr;
    const double gf = sd.g_f ? sd.g_f[e] : 0.0;
    double* p_out = sd.p ? sd.p + e * (kNout * 4) : nullptr;
    double F = 0, L = 0;
    const EvBeams eb = fixed_beams(cd);
    ShapeTape<SID, LM> S;
    S.base = lds + lane;
    const bool ok = shape_adjoint<SID, LM>(cd, eb, prog, xv, xg, gp, gf, p_out, &F, &L, sd.g_x + e * kNx, accv, S);
    if (sd.factor) sd.factor[e] = F;
    if (sd.volume) sd.volume[e] = eb.volume;
    if (sd.ok) sd.ok[e] = ok ? 1 : 0;
    if (sd.loss) sd.loss[e] = L;
  }
  wave_sums(accv);
#pragma unroll
  for (int v = 0; v < kNp; v++)
    if (lane == 0) part[v] = accv[v];
}

template <int LO, int HI, int LM>
__device__ __forceinline__ void unit_of_shape(int shape, int sub, const TileDesc& td, const SegDesc& sd,
                                              const ChannelDesc& cd, const NodeCmd* __restrict__ prog,
                                              double* __restrict__ part, double* lds) {
  if constexpr (HI - LO == 1) {
    shape_unit<LO, LM>(sub, td, sd, cd, prog, part, lds);
  } else {
    constexpr int MID = (LO + HI) / 2;
    if (shape < MID) unit_of_shape<LO, MID, LM>(shape, sub, td, sd, cd, prog, part, lds);
    else unit_of_shape<MID, HI, LM>(shape, sub, td, sd, cd, prog, part, lds);
  }
}

// Tiles of shapes [LO, HI): every workgroup takes the code specialised for its tile's shape.  One launch
// for all of them: a launch lasts at least one wave's lifetime.
template <int LO, int HI, int LM, int WPE>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WPE))) void shapes_kernel(
    const TileDesc* __restrict__ tiles, int t_begin, int n_units, int n_sub, const SegDesc* __restrict__ segs,
    const ChannelDesc* __restrict__ chans, const NodeCmd* __restrict__ nodes, double* __restrict__ gpart,
    int part_stride, AdjLayout) {
  __shared__ double lds[8 * kShapes[HI - 1].n_nodes * 64];
  // one workgroup per unit (the host launches n_units workgroups): no loop
  if (const int u = (int)blockIdx.x; u < n_units) {
    const int tl = u / n_sub, sub = u - tl * n_sub, t = t_begin + tl;
    const TileDesc td = tiles[t];
    const SegDesc sd = segs[td.seg];
    const ChannelDesc cd = chans[sd.channel];
    unit_of_shape<LO, HI, LM>(sd.shape, sub, td, sd, cd, nodes + sd.node0,
                              gpart + ((int64_t)t * n_sub + sub) * part_stride, lds);
  }
}

using Kernel = void (*)(const TileDesc*, int, int, int, const SegDesc*, const ChannelDesc*, const NodeCmd*, double*, int,
                        AdjLayout);

// The kernels of the shapes of five and of six final-state particles.
Kernel pick_5(int loss_mode);
Kernel pick_6_0();   // loss mode 0
Kernel pick_6_1();

}  // namespace adj

}  // namespace gphs
