// Inverse mapping kernels: the per-channel kernel, the shared-roots kernels of up to four final-state
// particles and of the generic walk, and the launch functions.  The device code is in phs_inverse.h.
#include "phs_inverse.h"

namespace gphs {

using namespace inv;

namespace {

// With RB (every deferred subtree is a daughter of the root, and no root has a friend) a bank
// entry is the root's cos theta, sin theta, cos phi, sin phi and the subtree's msq, m and
// p_decay: the root's G is its rotation applied to the identity (the root's bg is 0), so the
// pop re-forms it bit for bit from the four numbers.
constexpr int kInvRootBankWords = 7;

// Inverse of one event into channel `cd` (program `prog`): the randoms go to xo[0..n_x),
// returns the factor.
template <bool FR, bool PEV, bool RB>
__device__ __forceinline__ double inverse_event(const ChannelDesc& cd, const EvBeams& eb,
                                                const NodeCmd* __restrict__ prog, const double* __restrict__ pl,
                                                int S, double* bank, int B, gdouble* __restrict__ xo) {
  const double s = eb.s;
  double G[16] = {1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1};
  double cur_msq = s, cur_m = eb.sqrts, cur_p = 0, factor = 1;
  int depth = 0;
  for (int i = 0; i < cd.n_nodes; ++i) {
    const NodeCmd& nc = prog[i];
    double q0[4], q1[4];
    branch_sum(pl, S, cd.n_out, nc.k[0], q0);
    branch_sum(pl, S, cd.n_out, nc.k[1], q1);
    const double msq0 = q0[0] * q0[0] - q0[1] * q0[1] - q0[2] * q0[2] - q0[3] * q0[3];
    const double msq1 = q1[0] * q1[0] - q1[1] * q1[1] - q1[2] * q1[2] - q1[3] * q1[3];
    // x and factor of the internal daughters' msq maps
#pragma unroll
    for (int d = 0; d < 2; d++) {
      if (!nc.k[d].leaf) {
        double x, f;
        if constexpr (PEV) x_from_msq(child_at(nc.k[d], eb.sqrts, s, cd.m_tot), d == 0 ? msq0 : msq1, s, x, f);
        else x_from_msq(nc.k[d], d == 0 ? msq0 : msq1, s, x, f);
        xo[nc.k[d].xi] = x;
        factor *= f;
      }
    }
    // this branch's decay
    const Decay dk = decay(cur_msq, cur_m, cur_p, msq0, msq1);
    const double pk = dk.pk, bg = dk.bg;
    factor *= dk.lam;

    // angles of the first daughter in W = B_z(-bg) G
    const double g = math::sqrt_phys(1 + bg * bg);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const double r0 = G[j], r3 = G[12 + j];
      G[j] = g * r0 - bg * r3;
      G[12 + j] = -bg * r0 + g * r3;
    }
    double v0 = G[4] * q0[0] + G[5] * q0[1] + G[6] * q0[2] + G[7] * q0[3];
    double v1 = G[8] * q0[0] + G[9] * q0[1] + G[10] * q0[2] + G[11] * q0[3];
    double v2 = G[12] * q0[0] + G[13] * q0[1] + G[14] * q0[2] + G[15] * q0[3];
    if (FR && nc.friend_sign != 0) {
      // the beam k = (1, 0, 0, f) in the same frame fixes R (R e_z = n / |n|); v <- R^T v and
      // the rows of W likewise, so that G below is R_y(-theta) R_z(-phi) R^T W
      const double fs = (double)nc.friend_sign;
      const double n0 = G[4] + fs * G[7], n1 = G[8] + fs * G[11], n2 = G[12] + fs * G[15];
      const double nn = math::sqrt_phys(n0 * n0 + n1 * n1 + n2 * n2);
      const double a0 = n0 / nn, a1 = n1 / nn, c = n2 / nn;
      const double sa = math::sqrt_phys(a0 * a0 + a1 * a1);
      const double kx = sa > 0 ? -a1 / sa : 1.0, ky = sa > 0 ? a0 / sa : 0.0, h = 1 - c;
      const double r00 = c + h * kx * kx, r01 = h * kx * ky, r11 = c + h * ky * ky;
      // R^T rows: (r00, r01, -a0), (r01, r11, -a1), (a0, a1, c)
      const double u0 = r00 * v0 + r01 * v1 + -a0 * v2;
      const double u1 = r01 * v0 + r11 * v1 + -a1 * v2;
      const double u2 = a0 * v0 + a1 * v1 + c * v2;
      v0 = u0; v1 = u1; v2 = u2;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const double w1 = G[4 + j], w2 = G[8 + j], w3 = G[12 + j];
        G[4 + j] = r00 * w1 + r01 * w2 + -a0 * w3;
        G[8 + j] = r01 * w1 + r11 * w2 + -a1 * w3;
        G[12 + j] = a0 * w1 + a1 * w2 + c * w3;
      }
    }
    const Dir dr = direction(v0, v1, v2);
    const double ct = dr.ct, st = dr.st, cp = dr.cp, sp = dr.sp;
    xo[nc.x_phi] = dr.xphi;
    double xc, fct, m_max, cb0 = nc.b0, cb1 = nc.b1;
    if constexpr (PEV) node_at(nc, i == 0, eb, cd.m_tot, m_max, cb0, cb1);
    x_from_ct(nc.ct_kind, ct, cb0, cb1, xc, fct);
    xo[nc.x_phi + 1] = xc;
    factor *= fct;
    rotate_back(G, ct, st, cp, sp);

    // next branch: a daughter (G stays), or the deferred one from the save bank
    if (nc.push >= 0) {
      const double mp = nc.push == 0 ? msq0 : msq1;
      if constexpr (RB) {   // only the root pushes
        double* b = bank;
        b[0] = ct; b[B] = st; b[2 * B] = cp; b[3 * B] = sp;
        b[4 * B] = mp;
        b[5 * B] = math::sqrt_phys(mp);
        b[6 * B] = nc.push == 0 ? pk : -pk;
      } else {
        double* b = bank + kInvBankWords * depth * B;
#pragma unroll
        for (int j = 0; j < 16; j++) b[j * B] = G[j];
        b[16 * B] = mp;
        b[17 * B] = math::sqrt_phys(mp);
        b[18 * B] = nc.push == 0 ? pk : -pk;
      }
      depth++;
    }
    if (nc.desc >= 0) {
      cur_msq = nc.desc == 0 ? msq0 : msq1;
      cur_m = math::sqrt_phys(cur_msq);
      cur_p = nc.desc == 0 ? pk : -pk;
    } else if (depth > 0) {
      depth--;
      if constexpr (RB) {
        const double* b = bank;
#pragma unroll
        for (int j = 0; j < 16; j++) G[j] = (j % 5 == 0) ? 1.0 : 0.0;
        rotate_back(G, b[0], b[B], b[2 * B], b[3 * B]);
        cur_msq = b[4 * B];
        cur_m = b[5 * B];
        cur_p = b[6 * B];
      } else {
        const double* b = bank + kInvBankWords * depth * B;
#pragma unroll
        for (int j = 0; j < 16; j++) G[j] = b[j * B];
        cur_msq = b[16 * B];
        cur_m = b[17 * B];
        cur_p = b[18 * B];
      }
    }
  }
  return factor;
}

// LDS per workgroup: the momenta column (4 n_out rows of blockDim.x + 1 doubles), then the
// save banks (19 n_banks rows of blockDim.x doubles).
template <bool FR, bool PEV, bool RB>
__global__ __launch_bounds__(256) void inverse_kernel(const TileDesc* __restrict__ tiles, int n_tiles,
                                                      const SegDesc* __restrict__ segs,
                                                      const InvSeg* __restrict__ isegs,
                                                      const ChannelDesc* __restrict__ chans,
                                                      const NodeCmd* __restrict__ nodes, int n_ch, int n_out,
                                                      int n_x, int64_t n_rows, double* __restrict__ factors,
                                                      double* __restrict__ x_out) {
  const int B = (int)blockDim.x;
  const int S = B + 1;
  const int lane = (int)threadIdx.x;
  double* ps = inv_lds;
  double* bank = ps + 4 * n_out * S + lane;
  double* pl = ps + lane;
  for (int t = (int)blockIdx.x; t < n_tiles; t += (int)gridDim.x) {
    const TileDesc td = tiles[t];
    const SegDesc sd = segs[td.seg];
    const InvSeg is = isegs[td.seg];
    for (int base = 0; base < td.count; base += B) {
      const int cnt = min(B, td.count - base);
      const bool valid = lane < cnt;   // lanes past the end stage the last event and store nothing
      const int64_t e = td.e0 + base + (valid ? lane : cnt - 1);
      const int64_t row = is.row0 + e;
      EvBeams eb;
      if constexpr (PEV) eb = event_beams(chans[0], as_global(sd.e1)[e], as_global(sd.e2)[e]);
      else eb = fixed_beams(chans[0]);
      // momenta back in the centre-of-mass frame (inverse of phs.cu:1286-1301)
      const gdouble* pe = as_global((const double*)sd.p) + e * 4 * n_out;
      for (int j = 0; j < n_out; j++) {
        double q0 = pe[4 * j], q1 = pe[4 * j + 1], q2 = pe[4 * j + 2], q3 = pe[4 * j + 3];
        if (eb.bg_lab != 0) {
          const double a = eb.g_lab * q0 - eb.bg_lab * q3;
          const double b = -eb.bg_lab * q0 + eb.g_lab * q3;
          q0 = a; q3 = b;
        }
        pl[(4 * j) * S] = q0; pl[(4 * j + 1) * S] = q1; pl[(4 * j + 2) * S] = q2; pl[(4 * j + 3) * S] = q3;
      }
      for (int c = 0; c < n_ch; c++) {
        gdouble* xo = as_global(x_out) + ((int64_t)c * n_rows + row) * n_x;
        if (c == is.own) {
          if (valid) {
            const gdouble* xi = as_global(sd.x) + e * n_x;
            for (int k = 0; k < n_x; k++) xo[k] = xi[k];
            as_global(factors)[row * n_ch + c] = as_global((const double*)sd.factor)[e];
          }
          continue;
        }
        const ChannelDesc cd = chans[c];
        if (valid) as_global(factors)[row * n_ch + c] = inverse_event<FR, PEV, RB>(cd, eb, nodes + cd.node0, pl, S, bank, B, xo);
      }
    }
  }
}

}  // namespace

size_t inverse_lds_bytes(const InverseTables& it, int block) {
  if (it.shared_roots) return (size_t)(block / 64) * inverse_wave_words(it.n_out, it.n_x, it.generic ? it.rest_banks : 0) * sizeof(double);
  const size_t words = it.root_bank ? kInvRootBankWords : kInvBankWords;
  return ((size_t)4 * it.n_out * (block + 1) + words * it.n_banks * block) * sizeof(double);
}

namespace {

template <bool PEV>
SharedKernel pick_shared(const InverseTables& it) {
  if (!it.generic) {
    if (it.n_out == 2) return inverse_kernel_shared<PEV, 2, false, 3>;
    if (it.n_out == 3) return it.shared_branches ? inverse_kernel_shared<PEV, 3, true, 3> : inverse_kernel_shared<PEV, 3, false, 3>;
    if (it.n_out == 4) return it.shared_branches ? inverse_kernel_shared<PEV, 4, true, 3> : inverse_kernel_shared<PEV, 4, false, 3>;
    if (!PEV && it.n_out == 5) return shared_kernel_5();
    if (!PEV && it.n_out == 6) return shared_kernel_6();
  }
  return inverse_kernel_shared<PEV, 0, false, 0>;
}

}  // namespace

hipError_t launch_inverse(const InverseTables& it, const TileDesc* tiles, int n_tiles, int n_sub, const SegDesc* segs,
                          int block, int n_chunks, double* factors, double* x_out, int64_t n_rows,
                          hipStream_t stream) {
  if (n_tiles <= 0) return hipSuccess;
  if (block < 64 || block > 256 || block % 64 || n_sub < 1 || n_chunks < 1 || n_chunks > it.n_ch)
    return hipErrorInvalidValue;
  const size_t shmem = inverse_lds_bytes(it, block);
  if (shmem > forward_lds_limit()) return hipErrorInvalidValue;
  if (it.shared_roots) {
    const int64_t units = (int64_t)n_tiles * n_sub * n_chunks, waves = block / 64;
    if (units > 0x7fffffff) return hipErrorInvalidValue;
    auto k = it.per_event_beams ? pick_shared<true>(it) : pick_shared<false>(it);
    const int aligned = reinterpret_cast<uintptr_t>(x_out) % 16 == 0 ? 1 : 0;
    hipLaunchKernelGGL(k, dim3((unsigned)((units + waves - 1) / waves)), dim3(block), shmem, stream, tiles, (int)units,
                       n_sub, n_chunks, segs, it.isegs, it.steps, it.chans, it.nodes, it.maps, it.n_ch, it.n_out, it.n_x,
                       n_rows, it.generic ? it.rest_banks : 0, aligned, factors, x_out);
    return hipGetLastError();
  }
  using K = decltype(&inverse_kernel<false, false, false>);
  K k;
  if (it.root_bank)
    k = it.per_event_beams ? (it.has_friends ? inverse_kernel<true, true, true> : inverse_kernel<false, true, true>)
                           : (it.has_friends ? inverse_kernel<true, false, true> : inverse_kernel<false, false, true>);
  else
    k = it.per_event_beams ? (it.has_friends ? inverse_kernel<true, true, false> : inverse_kernel<false, true, false>)
                           : (it.has_friends ? inverse_kernel<true, false, false> : inverse_kernel<false, false, false>);
  hipLaunchKernelGGL(k, dim3(n_tiles), dim3(block), shmem, stream, tiles, n_tiles, segs, it.isegs, it.chans, it.nodes,
                     it.n_ch, it.n_out, it.n_x, n_rows, factors, x_out);
  return hipGetLastError();
}

}  // namespace gphs
