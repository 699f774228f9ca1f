// C ABI of the inverse mapping (include/gpu_phs.h): all-channel factors and randoms of the
// events of a plan (reference: the do_inverse_mapping branch of gen_phs_from_x_gpu,
// phs.cu:1491-1554).
#include <algorithm>
#include <cstring>
#include <string>
#include <utility>

#include "phs_state.h"

using namespace gphs;

namespace {

// The map constants of a branch as the specialised walks read them: p0, p1, q0, q1 and c are msq_min,
// msq_max - msq_min, -, -, f (linear); M^2, M Gamma, a0, a1 - a0, a2 (Breit-Wigner); msq_min, a0, msq_max,
// a1, a2 (the others), with the expressions of the maps themselves.
InvNode inv_node(const NodeCmd& nc) {
  InvNode r{};
  auto inverse = [](double v) { return v != 0 ? 1 / v : 0.0; };
  for (int d = 0; d < 2; d++) {
    const ChildCmd& c = nc.k[d];
    if (c.leaf) continue;
    InvMap& m = r.map[d];
    r.kind[d] = c.kind;
    if (c.kind == MK_LINEAR) m = InvMap{c.msq_min, c.msq_max - c.msq_min, 0, 0, 0, 0, c.f_lin};
    else if (c.kind == MK_BREIT_WIGNER) m = InvMap{c.m * c.m, c.m * c.w, 0, c.a0, c.a1 - c.a0, 0, c.a2};
    else m = InvMap{c.msq_min, c.a0, 0, c.msq_max, c.a1, 0, c.a2};
    m.inv0 = inverse(m.p1);
    m.inv1 = inverse(m.q1);
  }
  r.ct_kind = nc.ct_kind;
  r.b0 = nc.b0;
  r.b1 = nc.b1;
  r.inv_b0 = inverse(nc.b0);
  r.inv_2b1 = inverse(2 * nc.b1);
  return r;
}

// How a daughter's momentum is added up (a sum of two does not depend on their order).
std::string association(const NodeCmd* prog, const ChildCmd& k) {
  if (k.leaf) return std::to_string(k.out);
  if (k.sum_len <= 0) return "i" + std::to_string(k.leaves);   // in index order
  std::string a = association(prog, prog[k.node].k[0]), b = association(prog, prog[k.node].k[1]);
  if (b < a) std::swap(a, b);
  return "(" + a + " " + b + ")";
}

// Per branch of channel c in visit order, of the first n: everything its geometry depends on.
std::vector<std::string> branch_keys(const CompiledProcess& cp, int c, int n) {
  const NodeCmd* prog = &cp.nodes[cp.channels[c].node0];
  std::vector<std::string> keys;
  for (int i = 0; i < n; i++) {
    std::string up = i == 0 ? "" : keys[prog[i].parent] + "/" + std::to_string(prog[i].slot) + ":";
    keys.push_back(up + association(prog, prog[i].k[0]) + "," + association(prog, prog[i].k[1]));
  }
  return keys;
}

// Device tables of the inverse: per-segment (generating channel, first row), uploaded again when the rows
// change, then the process's channels and programs.
int inverse_prepare(PlanObj& pl, const int64_t* seg_row0, int64_t n_rows, hipStream_t stream) {
  if (pl.segs.empty()) return set_error(GPU_PHS_E_ARG, "inverse: the plan has no segments");
  const int proc = pl.chan_process.empty() ? -1 : pl.chan_process[0];
  for (int p : pl.chan_process)
    if (p != proc) return set_error(GPU_PHS_E_ARG, "inverse: all segments must belong to one process");
  ProcessObj* po = find_process(proc);
  if (!po) return set_error(GPU_PHS_E_HANDLE, "inverse: the plan's process was destroyed");
  const CompiledProcess& cp = po->cp;
  std::vector<InvSeg> is(pl.segs.size());
  for (size_t s = 0; s < pl.segs.size(); s++) {
    const int64_t r0 = seg_row0[s], n = pl.segs[s].n_events;
    if (r0 < 0 || r0 + n > n_rows) return set_error(GPU_PHS_E_ARG, "inverse: segment rows outside [0, n_rows)");
    is[s].own = pl.chan_channel[pl.segs[s].channel];
    is[s].pad = 0;
    is[s].row0 = r0;
  }
  const bool shared = !cp.has_friends && pl.specialize;
  if (pl.inv_dev && pl.inv_process == proc && pl.inv.per_event_beams == pl.dp.per_event_beams &&
      pl.inv.shared_roots == (shared ? 1 : 0) && is.size() == pl.inv_segs.size()) {
    // the process's tables are there; the rows may be others
    if (std::memcmp(is.data(), pl.inv_segs.data(), is.size() * sizeof(InvSeg)) == 0) return ok_status();
    hipError_t e = wait_for_queued(stream);
    if (e != hipSuccess) return hip_error(e, "hipStreamSynchronize(inverse rows)");
    e = hipMemcpy(pl.inv_dev, is.data(), is.size() * sizeof(InvSeg), hipMemcpyHostToDevice);
    if (e != hipSuccess) return hip_error(e, "hipMemcpy(inverse rows)");
    pl.inv_segs = std::move(is);
    return ok_status();
  }
  const int n_ch = (int)cp.channels.size();
  // the walk that reads a channel's structure from its program
  bool generic = cp.spec.n_out > (pl.dp.per_event_beams ? kInvShapeOutPev : kInvShapeOut);
  for (const ChannelDesc& c : cp.channels) generic = generic || c.shape < 0;
  // channel order: by what each branch, root first, computes from an event -- where it hangs, and both
  // daughters' final-state particles with the association their momenta are added in -- so that
  // channels sharing their first branches' evaluation are adjacent (the generic walk shares the root's
  // only); channel index within a group
  std::vector<std::vector<std::string>> keys(n_ch);
  for (int c = 0; shared && c < n_ch; c++) keys[c] = branch_keys(cp, c, generic ? 1 : cp.channels[c].n_nodes);
  std::vector<int> order(n_ch);
  for (int c = 0; c < n_ch; c++) order[c] = c;
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return keys[a] < keys[b]; });
  std::vector<InvStep> steps(n_ch);
  std::vector<std::string> last(kMaxOut);
  int branches = 0, evaluated = 0;   // below the roots
  for (int k = 0; k < n_ch; k++) {
    const int c = order[k];
    steps[k].channel = c;
    steps[k].node0 = cp.channels[c].node0;
    steps[k].shape = cp.channels[c].shape;
    steps[k].outs = 0;
    for (int i = 0; i < cp.channels[c].n_nodes && i < 8; i++)
      for (int d = 0; d < 2; d++) {
        const ChildCmd& k2 = cp.nodes[cp.channels[c].node0 + i].k[d];
        if (k2.leaf) steps[k].outs |= (uint64_t)k2.out << (4 * (2 * i + d));
      }
    steps[k].eval = 0;
    for (size_t i = 0; i < keys[c].size(); i++) {
      if (i > 0) branches++;
      if (keys[c][i] != last[i]) {
        steps[k].eval |= 1 << i;
        if (i > 0) evaluated++;
      }
      last[i] = keys[c][i];
    }
  }
  // save-bank levels of the subtrees deferred below the root (the root's own deferred daughter
  // is re-formed from the shared root)
  int rest_banks = 0;
  for (const ChannelDesc& c : cp.channels) {
    int depth = 0;
    for (int i = 1; i < c.n_nodes; i++) {
      const NodeCmd& nd = cp.nodes[c.node0 + i];
      if (nd.push >= 0) rest_banks = std::max(rest_banks, ++depth);
      if (nd.desc < 0 && depth > 0) depth--;
    }
  }
  auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
  const size_t o_chans = al(is.size() * sizeof(InvSeg));
  const size_t o_nodes = o_chans + al(cp.channels.size() * sizeof(ChannelDesc));
  const size_t o_steps = o_nodes + al(cp.nodes.size() * sizeof(NodeCmd));
  const size_t o_maps = o_steps + al(steps.size() * sizeof(InvStep));
  // (the walks specialised per tree shape read the maps' records; with per-event beams they read the programs)
  const size_t n_maps = generic || pl.dp.per_event_beams ? 0 : cp.nodes.size();
  const size_t total = o_maps + al(n_maps * sizeof(InvNode));
  if (total > pl.inv_bytes) {
    if (pl.inv_dev) (void)hipFree(pl.inv_dev);
    pl.inv_dev = nullptr;
    pl.inv_bytes = 0;
    hipError_t e = hipMalloc(&pl.inv_dev, total);
    if (e != hipSuccess) return hip_error(e, "hipMalloc(inverse tables)");
    pl.inv_bytes = total;
  }
  std::vector<char> host(total, 0);
  std::memcpy(host.data(), is.data(), is.size() * sizeof(InvSeg));
  std::memcpy(host.data() + o_chans, cp.channels.data(), cp.channels.size() * sizeof(ChannelDesc));
  std::memcpy(host.data() + o_nodes, cp.nodes.data(), cp.nodes.size() * sizeof(NodeCmd));
  std::memcpy(host.data() + o_steps, steps.data(), steps.size() * sizeof(InvStep));
  for (size_t i = 0; i < n_maps; i++) {
    const InvNode nd = inv_node(cp.nodes[i]);
    std::memcpy(host.data() + o_maps + i * sizeof(InvNode), &nd, sizeof nd);
  }
  hipError_t e = wait_for_queued(stream);
  if (e == hipSuccess) e = hipMemcpy(pl.inv_dev, host.data(), total, hipMemcpyHostToDevice);
  if (e != hipSuccess) return hip_error(e, "hipMemcpy(inverse tables)");
  char* base = (char*)pl.inv_dev;
  pl.inv.isegs = (const InvSeg*)base;
  pl.inv.chans = (const ChannelDesc*)(base + o_chans);
  pl.inv.nodes = (const NodeCmd*)(base + o_nodes);
  pl.inv.steps = (const InvStep*)(base + o_steps);
  pl.inv.maps = (const InvNode*)(base + o_maps);
  pl.inv.n_ch = n_ch;
  pl.inv.n_out = cp.spec.n_out;
  pl.inv.n_x = cp.spec.n_x();
  pl.inv.n_banks = cp.max_banks;
  int root_bank = cp.max_banks <= 1 ? 1 : 0;
  for (const ChannelDesc& c : cp.channels)
    for (int i = 0; i < c.n_nodes; i++) {
      const NodeCmd& nd = cp.nodes[c.node0 + i];
      if ((i > 0 && nd.push >= 0) || (i == 0 && nd.friend_sign != 0)) root_bank = 0;
    }
  pl.inv.root_bank = root_bank;
  pl.inv.has_friends = cp.has_friends ? 1 : 0;
  pl.inv.per_event_beams = pl.dp.per_event_beams;
  pl.inv.shared_roots = shared ? 1 : 0;
  pl.inv.rest_banks = rest_banks;
  // a repeated branch saves about a third of its channel's work, the tests for it cost a tenth of
  // every channel's: worth it where a quarter of the branches repeat
  pl.inv.shared_branches = shared && 4 * evaluated <= 3 * branches ? 1 : 0;
  pl.inv.generic = generic ? 1 : 0;
  if (generic || cp.spec.n_out > 4) pl.inv.shared_branches = 0;
  pl.inv_segs = std::move(is);
  pl.inv_process = proc;
  return ok_status();
}

// Ranges of channels that each 64-event unit is split over, one wave each: as many as give every
// SIMD its three waves (any split, also single channels), then as many as give a dozen rounds of
// waves, so that the last round's idle SIMDs cost little, but no fewer than min_channels channels
// each, since a range stages the momenta and evaluates its first root anew.  With the walks as they
// were when this was chosen (0.69 ms and 102 us since): 2e5 events x 120 channels (3190 units) 0.96 ms
// at 13 ranges, 1.08 at 4, 1.05 at 51; 1e6 events x 3 channels (15,627 units) 113 us unsplit, 138 at 3
// ranges.  Above four particles a channel is more work and a SIMD holds two waves, and three channels
// are enough: 1e5 events x 16 channels of 2->6 (1592 units) 154 us at 4 ranges, 145 at 5, 146 at 8, 157
// at 3.
int inverse_chunks(const InverseTables& it, int64_t units) {
  constexpr int64_t kFillWaves = 256 * 4 * 3, kManyWaves = 40000;
  const int64_t min_channels = it.n_out <= 4 ? 4 : 3;
  if (!it.shared_roots || units <= 0) return 1;
  const int64_t fill = std::min<int64_t>((kFillWaves + units - 1) / units, it.n_ch);
  const int64_t many = std::min<int64_t>((kManyWaves + units - 1) / units, it.n_ch / min_channels);
  return (int)std::max<int64_t>(1, std::max(fill, many));
}

}  // namespace

int gphs::plan_inverse(PlanObj& pl, const int64_t* seg_row0, int64_t n_rows, double* factors, double* x_out, int block,
                       hipStream_t stream) {
  if (!seg_row0 || n_rows <= 0 || !factors || !x_out)
    return set_error(GPU_PHS_E_ARG, "inverse: need seg_row0, n_rows > 0, factors and x_out");
  if (block != 0 && (block < 64 || block > 256 || block % 64))
    return set_error(GPU_PHS_E_ARG, "inverse: block must be 64, 128, 192 or 256");
  int rc = inverse_prepare(pl, seg_row0, n_rows, stream);
  if (rc) return rc;
  // the default workgroup: one wave with shared roots (its waves work alone), else 256 threads for
  // processes of a few channels, 128 for many, each where its LDS tables fit
  if (block == 0) {
    block = pl.inv.shared_roots ? 64 : pl.inv.n_ch <= 16 ? 256 : 128;
    while (block > 64 && inverse_lds_bytes(pl.inv, block) > forward_lds_limit()) block -= 64;
  }
  if (inverse_lds_bytes(pl.inv, block) > forward_lds_limit())
    return set_error(GPU_PHS_E_ARG, "inverse: the trees need more LDS than a workgroup of this size may use");
  // shared roots: a wave per 64-event unit, of every tile as many as the largest has or of those that have events
  const bool listed = pl.inv.shared_roots && pl.dp.units;
  hipError_t e = launch_inverse(pl.inv, listed ? pl.dp.units : pl.dp.tiles, listed ? (int)pl.units.size() : pl.dp.n_tiles,
                                listed ? 1 : std::max(1, (pl.tile_max + 63) / 64), pl.dp.segs, block,
                                inverse_chunks(pl.inv, pl.n_units), factors, x_out, n_rows, stream);
  if (e != hipSuccess) return hip_error(e, "inverse launch");
  return ok_status();
}

extern "C" {

int gpu_phs_plan_inverse(int plan, const int64_t* seg_row0, int64_t n_rows, double* factors, double* x_out,
                         int block, void* stream) {
  std::lock_guard<std::mutex> lk(api_mutex());
  PlanObj* pl = find_plan(plan);
  if (!pl) return set_error(GPU_PHS_E_HANDLE, "unknown plan");
  return plan_inverse(*pl, seg_row0, n_rows, factors, x_out, block, (hipStream_t)stream);
}

}  // extern "C"
