"""The work that is timed: what a program that uses this package has it do, through its public calls.

Every case is a dict of plain values:

  task       forward    momenta, factors, volumes and ok flags from randoms (``Plan.run``)
             inverse    the forward pass, then every channel's factor and randoms (``Plan.inverse``)
             adjoint    the built-in transverse-momentum loss and its gradients (``Plan.adjoint``)
             training   the forward pass, then the gradients for given cotangents
             adaptive   randoms drawn from the grids, the forward pass, the grids' update
             whizard    the host program's entry point: host arrays in, host arrays out
  process    one of PROCESSES, or "mix": the channels of four processes in one plan
  events     all events of a pass
  split      "even" or "ragged" shares of the events over the channels
  beams      "fixed", "boosted" (unequal fixed energies) or "event" (energies per event)
  submit     "direct" or "graph" (forward only)
  msq        the forward pass also writes every branch's msq

The inputs come from the seed alone; the shares of the channels from the case alone.
``exact`` restates the mapping in plain torch, in 64 bits.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import gpu_phs_amd as G
from gpu_phs_amd import workloads as W
from gpu_phs_amd.process import (MAP_COLLINEAR, MAP_INFRARED, MAP_NO, MAP_RADIATION, MAP_SCHANNEL, MAP_STEP_E,
                                 MAP_STEP_H, MAP_TCHANNEL, MAP_UCHANNEL)

DEV = "cuda:0"
F64 = torch.float64

PROCESSES = {
    "pair": W.process_c0,                       # 2->2, one channel
    "resonances": W.process_c1,                 # 2->4, three channels
    "jets": W.process_c2,                       # 2->4, 120 channels of random trees
    "sixbody": W.process_2to6,                  # 2->6, 16 channels
    "eightbody": lambda: W.process_large(8),    # 2->8, 12 channels: deep trees
    "friends": lambda: W.process_friends(4),    # 2->4 with beam-axis branches
    "friends6": lambda: W.process_friends(6),
    "threebody": lambda: W.process_shapes(3),   # every tree shape, every kind of map
    "fivebody": lambda: W.process_shapes(5, 1),
}


def _case(name, task, process, events, split="ragged", beams="fixed", submit="direct", msq=False):
    return dict(name=name, task=task, process=process, events=events, split=split, beams=beams, submit=submit,
                msq=msq)


def listed():
    return [
        # a host program that asks for a handful of points at a time: latency and launches
        _case("forward_small", "forward", "resonances", 999),
        # one integration batch of a multi-jet process: many channels, uneven shares
        _case("forward_jets", "forward", "jets", 1_000_003),
        # six heavy particles, a channel per topology
        _case("forward_sixbody", "forward", "sixbody", 500_009),
        # many processes and channels batched in one plan: the largest call
        _case("forward_mix", "forward", "mix", 20_000_000),
        # beam energies that vary from event to event (structure functions, beamstrahlung)
        _case("forward_event_beams", "forward", "resonances", 1_000_003, beams="event"),
        # the multi-channel weight: every event's factor in every channel, few channels
        _case("inverse_resonances", "inverse", "resonances", 1_000_003),
        # the same with many channels
        _case("inverse_jets", "inverse", "jets", 200_003),
        # the same with deep trees
        _case("inverse_sixbody", "inverse", "sixbody", 100_003),
        # gradients of the built-in loss in the randoms and the map parameters
        _case("adjoint_resonances", "adjoint", "resonances", 1_000_003),
        # a training step: forward, then the cotangents of the caller's own loss
        _case("training_sixbody", "training", "sixbody", 200_003),
        # one iteration of an adaptive integration
        _case("adaptive_resonances", "adaptive", "resonances", 4_000_037, split="even"),
        # the host program's batch call, copies included
        _case("whizard_resonances", "whizard", "resonances", 100_003),
    ]


# the processes a task is drawn with, and its range of events (the upper end at most the listed case's cost)
_RANGES = {
    "forward": {"pair": (100, 4_000_000), "resonances": (100, 4_000_000), "jets": (1_000, 4_000_000),
                "sixbody": (1_000, 2_000_000), "eightbody": (1_000, 500_000), "friends": (100, 2_000_000),
                "friends6": (100, 500_000), "threebody": (100, 2_000_000), "fivebody": (1_000, 2_000_000),
                "mix": (100_000, 10_000_000)},
    "inverse": {"pair": (100, 1_000_000), "resonances": (100, 1_000_000), "jets": (300, 200_000),
                "sixbody": (300, 100_000), "eightbody": (300, 50_000), "friends": (100, 500_000),
                "threebody": (100, 500_000), "fivebody": (300, 100_000)},
    "adjoint": {"pair": (100, 1_000_000), "resonances": (100, 1_000_000), "jets": (1_000, 500_000),
                "sixbody": (300, 200_000), "threebody": (100, 500_000), "fivebody": (300, 200_000)},
    "training": {"resonances": (100, 1_000_000), "jets": (1_000, 500_000), "sixbody": (300, 200_000),
                 "friends": (100, 200_000), "eightbody": (300, 50_000), "fivebody": (300, 200_000)},
    "adaptive": {"pair": (1_000, 2_000_000), "resonances": (1_000, 4_000_000), "jets": (10_000, 2_000_000),
                 "sixbody": (10_000, 1_000_000)},
    "whizard": {"pair": (100, 100_000), "resonances": (100, 100_000), "jets": (100, 5_000),
                "sixbody": (100, 10_000)},
}


def draw(rng):
    task = rng.choice(["forward", "forward", "forward", "inverse", "inverse", "adjoint", "training", "adaptive",
                       "whizard"])
    process = rng.choice(sorted(_RANGES[task]))
    lo, hi = _RANGES[task][process]
    case = _case("", task, process, int(math.exp(rng.uniform(math.log(lo), math.log(hi)))),
                 split=rng.choice(["even", "ragged"]))
    if process != "mix" and task != "adjoint":   # the built-in loss assumes symmetric beams
        case["beams"] = rng.choice(["fixed", "fixed", "boosted", "event"])
    if task == "forward":
        case["submit"] = rng.choice(["direct", "direct", "graph"])
        case["msq"] = process != "mix" and rng.random() < 0.2
    del case["name"]
    return case


# ---- the parts a program sets up once

def _segments(case):
    """(processes, [(process index, channel, events)]) of a case."""
    n = int(case["events"])
    if case["process"] == "mix":
        wl = W.workload("c3", n / 50_000_000)
        return wl.processes, [(s.process, s.channel, s.n_events) for s in wl.segments]
    proc = PROCESSES[case["process"]]()
    nc = proc.n_channels
    if case["split"] == "even":
        counts = [n // nc + (1 if c < n % nc else 0) for c in range(nc)]
    else:
        w = np.random.default_rng(n).dirichlet(np.full(nc, 0.5))
        counts = np.floor(w * n).astype(np.int64)
        counts[int(np.argmax(counts))] += n - int(counts.sum())
    return [proc], [(0, c, int(k)) for c, k in enumerate(counts) if k > 0]


def _fixed_energies(case, proc):
    half = proc.sqrts / 2
    return (1.25 * half, 0.8 * half) if case["beams"] == "boosted" else (half, half)


def _randoms(case, seed, procs, segs):
    """One buffer of randoms per process, the segments' events one after the other."""
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return [torch.rand((sum(n for q, _, n in segs if q == i), p.n_x), generator=g, device=DEV, dtype=F64)
            for i, p in enumerate(procs)], g


def _event_energies(case, proc, n, g):
    half = proc.sqrts / 2
    return [half * (0.7 + 0.3 * torch.rand(n, generator=g, device=DEV, dtype=F64)) for _ in range(2)]


def _inputs(case, seed):
    """What the seed fixes: the processes, the segments, the randoms, the beams, the cotangents, the grids' weights."""
    procs, segs = _segments(case)
    x, g = _randoms(case, seed, procs, segs)
    d = dict(procs=procs, segs=segs, x=x, seed=int(seed))
    if case["beams"] == "event":
        d["beams"] = _event_energies(case, procs[0], x[0].shape[0], g)
    if case["task"] == "training":
        n, n_out = x[0].shape[0], procs[0].n_out
        d["g_p"] = torch.randn((n, n_out, 4), generator=g, device=DEV, dtype=F64) / procs[0].sqrts
        d["g_f"] = torch.randn(n, generator=g, device=DEV, dtype=F64)
    if case["task"] == "adaptive":
        shape = (procs[0].n_channels, procs[0].n_x, G.Grid.BINS)
        d["weights"] = 0.5 + torch.rand(shape, generator=g, device=DEV, dtype=F64).cpu().numpy()
    return d


def _views(segs, i, t):
    """The segments' parts of a buffer that holds process i's events."""
    out, at = [], 0
    for q, _, n in segs:
        if q == i:
            out.append(t[at:at + n])
            at += n
    return out


def prepare(case, seed):
    st = _inputs(case, seed)
    if case["task"] == "whizard":
        return _prepare_whizard(case, st)
    procs, segs = st["procs"], st["segs"]
    handles = [G.ProcessHandle(p, *_fixed_energies(case, p)) for p in procs]
    out, parts = [], []
    for i, p in enumerate(procs):
        buf = G.EventBuffers.allocate(st["x"][i], p.n_out)
        out.append(buf)
        parts.append(zip(*(_views(segs, i, t) for t in (buf.x, buf.p, buf.factor, buf.volume, buf.ok))))
    plan = G.Plan([(handles[q], c, G.EventBuffers(*next(parts[q]))) for q, c, _ in segs])
    st.update(handles=handles, out=out, plan=plan, task=case["task"], graph=case["submit"] == "graph")
    n = st["x"][0].shape[0]
    if case["beams"] == "event":
        for k, (e1, e2) in enumerate(zip(*(_views(segs, 0, e) for e in st["beams"]))):
            plan.set_event_beams(k, e1, e2)
    if case["msq"]:
        st["msq"] = torch.zeros((n, 2 ** procs[0].n_out - 1), device=DEV, dtype=F64)
        for k, m in enumerate(_views(segs, 0, st["msq"])):
            plan.set_msq_output(k, m)
    if case["task"] == "inverse":
        st["factors"] = torch.empty((n, procs[0].n_channels), device=DEV, dtype=F64)
        st["x_out"] = torch.empty((procs[0].n_channels, n, procs[0].n_x), device=DEV, dtype=F64)
    if case["task"] in ("adjoint", "training"):
        st["g_x"] = torch.empty_like(st["x"][0])
        st["g_par"] = torch.empty(plan.n_params(), device=DEV, dtype=F64)
        st["g_x_parts"] = _views(segs, 0, st["g_x"])
    if case["task"] == "adjoint":
        st["loss"] = torch.empty(n, device=DEV, dtype=F64)
        st["loss_parts"] = _views(segs, 0, st["loss"])
    if case["task"] == "training":
        st["g_p_parts"], st["g_f_parts"] = _views(segs, 0, st["g_p"]), _views(segs, 0, st["g_f"])
    if case["task"] == "adaptive":
        st["grid"] = G.Grid(handles[0])
        st["grid"].set_weights(st["weights"])
    return st


def run(st):
    task = st["task"]
    if task == "whizard":
        return _run_whizard(st)
    plan = st["plan"]
    if task == "adjoint":
        plan.adjoint(st["g_x_parts"], loss=st["loss_parts"], loss_mode=1, write_forward=False, gparam=st["g_par"])
        return dict(g_x=st["g_x"], loss=st["loss"], g_par=st["g_par"])
    if task == "adaptive":
        st["grid"].generate(plan, st["seed"])
    if st["graph"]:
        plan.run_graph()
    else:
        plan.run()
    got = [dict(p=b.p, factor=b.factor, volume=b.volume, ok=b.ok) for b in st["out"]]
    if task == "forward":
        return dict(events=got, **({"msq": st["msq"]} if "msq" in st else {}))
    if task == "inverse":
        plan.inverse(factors=st["factors"], x_out=st["x_out"])
        return dict(events=got, factors=st["factors"], x_out=st["x_out"])
    if task == "training":
        plan.adjoint(st["g_x_parts"], g_p=st["g_p_parts"], g_f=st["g_f_parts"], write_forward=False,
                     gparam=st["g_par"])
        return dict(events=got, g_x=st["g_x"], g_par=st["g_par"])
    st["grid"].update(plan)
    return dict(events=got, x=st["x"][0], weights=st["grid"].weights())


# ---- the host program's interface: one process at a time, set up once

_whizard = {"process": None}


def _int(v):
    return ctypes.byref(ctypes.c_int(v))


def _at(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def _set_up_whizard(name, proc):
    if _whizard["process"] == name:
        return
    L, nc = G.lib(), proc.n_channels
    if _whizard["process"] is not None:
        L.c_whizard_finalize_gpu_phs()
    L.c_whizard_set_particle_structure(_int(nc), _int(nc), _int(1), _int(proc.n_x), _int(proc.n_in), _int(proc.n_out))
    L.c_whizard_set_flavors(_at(np.ascontiguousarray(proc.flv_masses)), _at(np.ascontiguousarray(proc.flv_widths)))
    L.c_whizard_init_mappings()
    L.c_whizard_init_tree_structures()
    friends = np.ascontiguousarray(proc.friends_or_zero(), np.int32)
    d1, d2, hc, ids, mm, mw, _ = proc.ctypes_args()
    for c in range(nc):
        L.c_whizard_fill_mapping(_int(c + 1), _at(ids[c]), _at(mm[c]), _at(mw[c]))
        L.c_whizard_fill_tree_structure(_int(c + 1), _at(d1[c]), _at(d2[c]), _at(hc[c]), _at(friends[c]))
    L.c_whizard_init_gpu_phs()
    if L.gpu_phs_last_error() != 0:
        raise RuntimeError(L.gpu_phs_last_error_message().decode())
    _whizard["process"] = name


def _whizard_energies(case, st):
    proc, n = st["procs"][0], st["x"][0].shape[0]
    if case["beams"] == "event":
        return [e.cpu().numpy() for e in st["beams"]]
    return [np.full(n, e) for e in _fixed_energies(case, proc)]


def _prepare_whizard(case, st):
    proc = st["procs"][0]
    _set_up_whizard(case["process"], proc)
    n, nc = st["x"][0].shape[0], proc.n_channels
    counts = np.zeros(nc, np.int64)
    for _, c, k in st["segs"]:
        counts[c] = k
    x = st["x"][0].cpu().numpy()
    e1, e2 = _whizard_energies(case, st)
    out = dict(p=np.zeros((n, proc.n_out, 4)), factors=np.zeros((n, nc)), volumes=np.zeros(n),
               oks=np.zeros(n, np.bool_), x_out=np.zeros((nc, n, proc.n_x)))
    limits = (ctypes.c_int * nc)(*np.cumsum(counts).tolist())
    batch = (_int(n), _int(nc), limits)
    call = (_at(e1), _at(e2), ctypes.byref(ctypes.c_bool(True)), _int(n), _int(nc), _int(proc.n_x), _at(x),
            _at(out["factors"]), _at(out["volumes"]), _at(out["oks"]), _at(out["p"]), _at(out["x_out"]))
    return dict(task="whizard", batch=batch, call=call, out=out, keep=(x, e1, e2))


def _run_whizard(st):
    L = G.lib()
    L.c_whizard_init_channel_ids(*st["batch"])
    L.c_whizard_gen_phs_from_x_gpu(*st["call"])
    if L.gpu_phs_last_error() != 0:
        raise RuntimeError(L.gpu_phs_last_error_message().decode())
    return st["out"]


# ---- what a pass cannot do without

def work(case):
    """Inputs read once, outputs written once.  Flops: per branch of a tree about 110 for the two maps and the decay
    and 90 for the boost, the same again for each inverse, three times as many for the gradients."""
    procs, segs = _segments(case)
    bytes_, flops = 0, 0
    for q, _, n in segs:
        p = procs[q]
        x, mom, branch = 8 * p.n_x, 32 * p.n_out, 200 * (p.n_out - 1)
        out = mom + 17
        per, ops = x + out, branch
        if case["beams"] == "event":
            per += 16
        if case["msq"]:
            per += 8 * (2 * p.n_out - 1)
        if case["task"] in ("inverse", "whizard"):
            per += 8 * p.n_channels * (1 + p.n_x)
            ops += branch * p.n_channels
        if case["task"] == "adjoint":
            per, ops = 2 * x + 8, 4 * branch
        if case["task"] == "training":
            per, ops = per + mom + 8 + x, 4 * branch
        if case["task"] == "whizard":
            per += 16
        bytes_ += n * per
        flops += n * ops
    return {"bytes": bytes_, "flops": flops}


# ---- the same results in plain torch

def _t(v):
    return torch.as_tensor(v, dtype=F64, device=DEV)


class _Tree:
    """One channel's tree, its masses and maps.  Branches go by their bincode."""

    def __init__(self, proc, c, M=None, Wd=None):
        self.proc, self.n_out, self.root = proc, proc.n_out, 2 ** proc.n_out - 1
        hc = proc.has_children[c]
        self.kids = {b: (int(proc.d1[c][b - 1]), int(proc.d2[c][b - 1])) for b in range(1, self.root + 1) if hc[b - 1]}
        self.kids = {b: k for b, k in self.kids.items() if b in self._below(self.root)}
        self.map = {b: int(proc.map_ids[c][b - 1]) for b in self.kids}
        M = _t(proc.map_masses[c].copy()) if M is None else M
        Wd = _t(proc.map_widths[c].copy()) if Wd is None else Wd
        self.M, self.W = {b: M[b - 1] for b in self.kids}, {b: Wd[b - 1] for b in self.kids}
        friends = proc.friends_or_zero()[c]
        self.friend = {b: {2 ** self.n_out: -1.0, 2 ** (self.n_out + 1): 1.0}.get(int(friends[b - 1]), 0.0)
                       for b in self.kids}
        self.m_min = {}
        self._masses(self.root)
        self.x_msq, self.x_phi = {}, {}
        self._post(self.root)
        self._pre(self.root)

    def _below(self, b):
        hc = self.kids
        return {b} | (self._below(hc[b][0]) | self._below(hc[b][1]) if b in hc else set())

    def _masses(self, b):
        if b in self.kids:
            self.m_min[b] = sum(self._masses(k) for k in self.kids[b])
        else:
            self.m_min[b] = float(self.proc.flv_masses[2 + b.bit_length() - 1])
        return self.m_min[b]

    def _post(self, b):
        for k in self.kids[b]:
            if k in self.kids:
                self._post(k)
        if b != self.root:
            self.x_msq[b] = len(self.x_msq)

    def _pre(self, b):
        self.x_phi[b] = self.n_out - 2 + 2 * len(self.x_phi)
        for k in self.kids[b]:
            if k in self.kids:
                self._pre(k)

    def visits(self, b=None):
        """The branches as the parameter gradients list them: the smaller daughter's subtree first."""
        b = self.root if b is None else b
        inner = sorted((k for k in self.kids[b] if k in self.kids), key=lambda k: bin(k).count("1"))
        return [b] + [v for k in inner for v in self.visits(k)]

    def limits(self, b, rs):
        lo = _t(self.m_min[b])
        return lo * lo, (rs - self.m_min[self.root] + lo) ** 2

    def msq_constants(self, b, rs):
        (lo, hi), s, m, w, kind = self.limits(b, rs), rs * rs, self.M[b], self.W[b], self.map[b]
        if kind == MAP_SCHANNEL:
            a0, a1 = torch.atan((lo - m * m) / (m * w)), torch.atan((hi - m * m) / (m * w))
            return a0, a1, (a1 - a0) * (m * w) / s
        if kind in (MAP_COLLINEAR, MAP_INFRARED, MAP_RADIATION):
            a0 = w * w if kind == MAP_RADIATION else m * m
            a1 = torch.log((hi - lo) / a0 + 1)
            return a0, a1, a1 / s
        if kind in (MAP_TCHANNEL, MAP_UCHANNEL):
            a0 = m * m
            a1 = 2 * torch.log((hi - lo) / (2 * a0) + 1)
            return a0, a1, a1 / s
        if kind == MAP_STEP_E:
            a2 = 2 * m * w / (hi - lo)
            a2 = torch.where(a2 < 0.01, torch.full_like(a2, 0.01), a2)
            a1 = torch.exp(-(m * m - lo) / (hi - lo) / a2)
            return 1 - a2 * torch.log((1 + a1 * torch.exp(1 / a2)) / (1 + a1)), a1, a2
        if kind == MAP_STEP_H:
            a2 = (m * m - lo) / (hi - lo)
            a1 = (2 * m * w / (hi - lo)) ** 2 / a2
            a1 = torch.where(a1 < 1e-6, torch.full_like(a1, 1e-6), a1)
            return (1 + torch.sqrt(1 + 4 * a1 / (1 - a2))) / 2, a1, a2
        return _t(0.0), hi - lo, (hi - lo) / s

    def msq_of(self, b, x, rs):
        (lo, hi), s, m, w, kind = self.limits(b, rs), rs * rs, self.M[b], self.W[b], self.map[b]
        a0, a1, a2 = self.msq_constants(b, rs)
        if kind == MAP_SCHANNEL:
            z = (1 - x) * a0 + x * a1
            t = torch.tan(z)
            inside = z.abs() < math.pi / 2
            return torch.where(inside, m * (m + w * t), 0 * t), torch.where(inside, a2 * (1 + t * t), 0 * t)
        if kind in (MAP_COLLINEAR, MAP_INFRARED, MAP_RADIATION):
            q = a0 * torch.exp(x * a1)
            return q - a0 + lo, a2 * q
        if kind in (MAP_TCHANNEL, MAP_UCHANNEL):
            low = x < 0.5
            q = a0 * torch.exp(torch.where(low, x, 1 - x) * a1)
            return torch.where(low, q - a0 + lo, -(q - a0) + hi), a2 * q
        if kind == MAP_STEP_E:
            q = torch.exp(-x * a0 / a2) * (1 + a1)
            z = -a2 * torch.log(q - a1)
            return z * hi + (1 - z) * lo, a0 / (1 - a1 / q) * (hi - lo) / s
        if kind == MAP_STEP_H:
            z = a1 / (a0 - x) - a1 / a0 + a2 * x
            return z * hi + (1 - z) * lo, (a1 / (a0 - x) ** 2 + a2) * (hi - lo) / s
        return (1 - x) * lo + x * hi, ((hi - lo) / s).expand_as(x)

    def x_of_msq(self, b, q, rs):
        (lo, hi), s, m, w, kind = self.limits(b, rs), rs * rs, self.M[b], self.W[b], self.map[b]
        a0, a1, a2 = self.msq_constants(b, rs)
        if kind == MAP_SCHANNEL:
            z = (q - m * m) / (m * w)
            return (torch.atan(z) - a0) / (a1 - a0), a2 * (1 + z * z)
        if kind in (MAP_COLLINEAR, MAP_INFRARED, MAP_RADIATION):
            z = q - lo + a0
            return torch.log(z / a0) / a1, a2 * z
        if kind in (MAP_TCHANNEL, MAP_UCHANNEL):
            low = q < (hi + lo) / 2
            z = torch.where(low, q - lo + a0, hi - q + a0)
            v = torch.log(z / a0) / a1
            return torch.where(low, v, 1 - v), a2 * z
        z = (q - lo) / (hi - lo)
        if kind == MAP_STEP_E:
            t = 1 + a1 * torch.exp(z / a2)
            return (z - a2 * torch.log(t / (1 + a1))) / a0, a0 * t * (hi - lo) / s
        if kind == MAP_STEP_H:
            t = a1 / (a0 * a2)
            u, v = a0 + z / a2, a0 - z / a2
            x = (u + t - torch.sqrt(v * v + 2 * t * u + t * t)) / 2
            return x, (a1 / (a0 - x) / (a0 - x) + a2) * (hi - lo) / s
        return z, ((hi - lo) / s).expand_as(z)

    def _peak(self, b, rs, s_friend):
        if self.map[b] not in (MAP_COLLINEAR, MAP_TCHANNEL, MAP_UCHANNEL):
            return None
        b0 = self.M[b] * self.M[b] / (s_friend if self.friend[b] else rs * rs)
        return b0, torch.log((b0 + 1) / b0)

    def cos_of(self, b, x, rs, s_friend):
        peak = self._peak(b, rs, s_friend)
        if peak is None:
            t = 2 * (1 - x)
            return 1 - t, torch.sqrt(t * (2 - t)), torch.ones_like(x)
        low = x < 0.5
        t = peak[0] * torch.exp(torch.where(low, 2 * x, 2 * (1 - x)) * peak[1])
        c = torch.where(low, t - peak[0] - 1, -(t - peak[0]) + 1)
        inside = c.abs() <= 1
        c = torch.where(inside, c, torch.ones_like(c))
        return c, torch.sqrt(1 - c * c), torch.where(inside, t * peak[1], 0 * t)

    def x_of_cos(self, b, c, rs, s_friend):
        peak = self._peak(b, rs, s_friend)
        if peak is None:
            return (c + 1) / 2, torch.ones_like(c)
        t = torch.where(c < 0, c, -c) + peak[0] + 1
        v = torch.log(t / peak[0]) / (2 * peak[1])
        return torch.where(c < 0, v, 1 - v), t * peak[1]

    def volume(self, b, rs):
        v = 1.0
        for k in self.kids[b]:
            v = v * (self.volume(k, rs) if k in self.kids else 1.0)
        return v / (4 * (2 * math.pi) ** 5) if b == self.root else v * rs * rs / (4 * (2 * math.pi) ** 2)


def _dot(a, b):
    r = a[0] * b[0]
    for u, v in zip(a[1:], b[1:]):
        r = r + u * v
    return r


def _mul(A, B):
    cols = list(zip(*B))
    return [[_dot(row, col) for col in cols] for row in A]


def _friend_rotation(n):
    """The rotation about e_z x n that takes e_z to n / |n|."""
    nn = torch.sqrt(_dot(n, n))
    a0, a1, c = (v / nn for v in n)
    sa = torch.sqrt(a0 * a0 + a1 * a1)
    one, zero = torch.ones_like(sa), torch.zeros_like(sa)
    kx, ky, h = torch.where(sa > 0, -a1 / sa, one), torch.where(sa > 0, a0 / sa, zero), 1 - c
    return [[c + h * kx * kx, h * kx * ky, a0], [h * kx * ky, c + h * ky * ky, a1], [-a0, -a1, c]]


def _beams(E1, E2):
    r = torch.sqrt(E1 * E2)
    bg = (E1 - E2) / (2 * r)
    return 2 * r, 4 * E1 * E2, bg, torch.sqrt(1 + bg * bg)


def _forward(tree, x, E1, E2):
    """(momenta [n][n_out][4], factor, volume, ok, {bincode: msq}) of randoms x [n][n_x]."""
    rs, s_friend, bg_lab, g_lab = _beams(E1, E2)
    zero = torch.zeros_like(x[:, 0])
    msq, f = {tree.root: rs * rs + zero}, zero + 1
    for b, k in tree.x_msq.items():
        msq[b], fm = tree.msq_of(b, x[:, k], rs)
        f = f * fm
    for j in range(tree.n_out):
        msq[1 << j] = zero + tree.m_min[1 << j] ** 2
    p_decay, ok = {tree.root: zero}, torch.ones_like(zero, dtype=torch.bool)
    for b, (k1, k2) in tree.kids.items():
        q, q1, q2 = msq[b], msq[k1], msq[k2]
        m = rs + zero if b == tree.root else torch.sqrt(q)
        top = rs if b == tree.root else rs - tree.m_min[tree.root] + tree.m_min[b]
        lam = (q - q1 - q2) ** 2 - 4 * q1 * q2
        ok = ok & (lam > 0) & (m > torch.sqrt(q1) + torch.sqrt(q2)) & (m <= top)
        sl = torch.sqrt(lam)
        p_decay[k1], p_decay[k2], f = sl / (2 * m), -sl / (2 * m), f * (sl / q)
    p = [None] * tree.n_out
    one = zero + 1

    def walk(b, L0, f):
        pd = p_decay[b]
        if b not in tree.kids:
            E = torch.sqrt(msq[b] + pd * pd)
            q = [L0[i][0] * E + L0[i][3] * pd for i in range(4)]
            q[0], q[3] = g_lab * q[0] + bg_lab * q[3], bg_lab * q[0] + g_lab * q[3]
            p[b.bit_length() - 1] = torch.stack(q, 1)
            return f
        m = rs + zero if b == tree.root else torch.sqrt(msq[b])
        bg = torch.where(m > 0, pd / m, zero) if b != tree.root else zero
        g = torch.sqrt(1 + bg * bg)
        phi = 2 * math.pi * x[:, tree.x_phi[b]]
        cp, sp = torch.cos(phi), torch.sin(phi)
        ct, st, fc = tree.cos_of(b, x[:, tree.x_phi[b] + 1], rs, s_friend)
        Q = [[ct * cp, -sp, st * cp], [ct * sp, cp, st * sp], [-st, zero, ct]]
        if tree.friend[b]:
            fs = tree.friend[b]
            u = [L0[0][0] - fs * L0[3][0]] + [-L0[0][j] + fs * L0[3][j] for j in (1, 2, 3)]
            Q = _mul(_friend_rotation([u[1], u[2], -bg * u[0] + g * u[3]]), Q)
        L1 = [[g] + [bg * v for v in Q[2]], [zero] + Q[0], [zero] + Q[1], [bg] + [g * v for v in Q[2]]]
        L = _mul(L0, L1)
        f = f * fc
        for k in tree.kids[b]:
            f = walk(k, L, f)
        return f

    f = walk(tree.root, [[one if i == j else zero for j in range(4)] for i in range(4)], f)
    return torch.stack(p, 1), f, tree.volume(tree.root, rs) + zero, ok, msq


def _inverse(tree, p, E1, E2):
    """(factor [n], randoms [n][n_x]) under which the tree gives the momenta p [n][n_out][4]."""
    rs, s_friend, bg_lab, g_lab = _beams(E1, E2)
    mom = {}
    for j in range(tree.n_out):
        q = [p[:, j, i] for i in range(4)]
        mom[1 << j] = [g_lab * q[0] - bg_lab * q[3], q[1], q[2], -bg_lab * q[0] + g_lab * q[3]]
    zero = torch.zeros_like(p[:, 0, 0])
    one = zero + 1
    x = [zero] * tree.proc.n_x

    def add(b):
        if b in tree.kids:
            k1, k2 = tree.kids[b]
            mom[b] = [u + v for u, v in zip(add(k1), add(k2))]
        return mom[b]

    add(tree.root)
    msq = {b: q[0] * q[0] - q[1] * q[1] - q[2] * q[2] - q[3] * q[3] for b, q in mom.items()}
    msq[tree.root] = rs * rs + zero

    def walk(b, G0, pd, f):
        k1, k2 = tree.kids[b]
        for k in (k1, k2):
            if k in tree.kids:
                x[tree.x_msq[k]], fm = tree.x_of_msq(k, msq[k], rs)
                f = f * fm
        lam = (msq[b] - msq[k1] - msq[k2]) ** 2 - 4 * msq[k1] * msq[k2]
        sl = torch.where(lam > 0, torch.sqrt(lam), zero)
        m = rs + zero if b == tree.root else torch.sqrt(msq[b])
        f = f * torch.where(lam > 0, sl / msq[b], zero)
        bg = torch.where(m > 0, pd / m, zero)
        g = torch.sqrt(1 + bg * bg)
        Gb = [[g * u - bg * v for u, v in zip(G0[0], G0[3])], G0[1], G0[2],
              [-bg * u + g * v for u, v in zip(G0[0], G0[3])]]
        if tree.friend[b]:
            R = _friend_rotation([Gb[i][0] + tree.friend[b] * Gb[i][3] for i in (1, 2, 3)])
            Gb = [Gb[0]] + _mul(list(zip(*R)), Gb[1:])
        v = [_dot(Gb[i], mom[k1]) for i in (1, 2, 3)]
        rho, vv = torch.sqrt(v[0] * v[0] + v[1] * v[1]), torch.sqrt(_dot(v, v))
        phi = torch.atan2(v[1], v[0])
        x[tree.x_phi[b]] = torch.where(phi < 0, phi + 2 * math.pi, phi) / (2 * math.pi)
        cp, sp = torch.where(rho > 0, v[0] / rho, one), torch.where(rho > 0, v[1] / rho, zero)
        ct, st = v[2] / vv, rho / vv
        x[tree.x_phi[b] + 1], fc = tree.x_of_cos(b, ct, rs, s_friend)
        f = f * fc
        R = [[ct * cp, ct * sp, -st], [-sp, cp, zero], [st * cp, st * sp, ct]]
        Gk = [Gb[0]] + _mul(R, Gb[1:])
        for k, pk in ((k1, sl / (2 * m)), (k2, -sl / (2 * m))):
            if k in tree.kids:
                f = walk(k, Gk, pk, f)
        return f

    f = walk(tree.root, [[one if i == j else zero for j in range(4)] for i in range(4)], zero, one)
    return f, torch.stack(x, 1)


def _segment_events(case, d):
    """(process index, channel, rows, E1, E2) of every segment."""
    at = [0] * len(d["procs"])
    for q, c, n in d["segs"]:
        rows = slice(at[q], at[q] + n)
        at[q] += n
        if case["beams"] == "event":
            yield q, c, rows, d["beams"][0][rows], d["beams"][1][rows]
        else:
            yield q, c, rows, *(_t(e) for e in _fixed_energies(case, d["procs"][q]))


def _exact_forward(case, d):
    events, msq = [], None
    for p, x in zip(d["procs"], d["x"]):
        n = x.shape[0]
        events.append(dict(p=torch.empty((n, p.n_out, 4), device=DEV, dtype=F64),
                           factor=torch.empty(n, device=DEV, dtype=F64), volume=torch.empty(n, device=DEV, dtype=F64),
                           ok=torch.empty(n, device=DEV, dtype=torch.uint8)))
    if case["msq"]:
        msq = torch.zeros((d["x"][0].shape[0], 2 ** d["procs"][0].n_out - 1), device=DEV, dtype=F64)
    for q, c, rows, E1, E2 in _segment_events(case, d):
        o = events[q]
        o["p"][rows], o["factor"][rows], o["volume"][rows], ok, m = _forward(_Tree(d["procs"][q], c), d["x"][q][rows], E1, E2)
        o["ok"][rows] = ok.to(torch.uint8)
        if msq is not None:
            for b, v in m.items():
                msq[rows, b - 1] = v
    return events, msq


def _exact_inverse(case, d, events):
    proc, n = d["procs"][0], d["x"][0].shape[0]
    factors = torch.empty((n, proc.n_channels), device=DEV, dtype=F64)
    x_out = torch.empty((proc.n_channels, n, proc.n_x), device=DEV, dtype=F64)
    if case["beams"] == "event":
        E1, E2 = d["beams"]
    else:
        E1, E2 = (_t(e) for e in _fixed_energies(case, proc))
    for c in range(proc.n_channels):
        factors[:, c], x_out[c] = _inverse(_Tree(proc, c), events[0]["p"], E1, E2)
    for _, c, rows, _, _ in _segment_events(case, d):
        factors[rows, c], x_out[c, rows] = events[0]["factor"][rows], d["x"][0][rows]
    return factors, x_out


def _exact_gradients(case, d, events):
    """Gradients by torch's own differentiation, of the accepted events only (the others have none)."""
    proc = d["procs"][0]
    g_x, loss, g_par = torch.zeros_like(d["x"][0]), torch.zeros(d["x"][0].shape[0], device=DEV, dtype=F64), []
    for _, c, rows, E1, E2 in _segment_events(case, d):
        ok = events[0]["ok"][rows].bool()
        x = d["x"][0][rows][ok].clone().requires_grad_(True)
        M = _t(proc.map_masses[c].copy()).requires_grad_(True)
        Wd = _t(proc.map_widths[c].copy()).requires_grad_(True)
        if case["beams"] == "event":
            E1, E2 = E1[ok], E2[ok]
        with torch.enable_grad():
            tree = _Tree(proc, c, M, Wd)
            p, f, _, _, _ = _forward(tree, x, E1, E2)
            if case["task"] == "adjoint":
                each = f * (p[:, :, 1] ** 2 + p[:, :, 2] ** 2).sum(1) / (proc.sqrts * proc.sqrts)
            else:
                each = (p * d["g_p"][rows][ok]).sum((1, 2)) + f * d["g_f"][rows][ok]
            grads = torch.autograd.grad(each.sum(), (x, M, Wd), allow_unused=True)
        part = torch.zeros_like(g_x[rows])
        part[ok] = grads[0]
        g_x[rows] = part
        loss[rows] = torch.zeros_like(loss[rows]).masked_scatter(ok, each.detach())
        gM, gW = (torch.zeros_like(M) if g is None else g for g in grads[1:])
        for b in tree.visits():
            g_par += [gM[b - 1], gW[b - 1]]
    return g_x, loss, torch.stack(g_par).detach()


def _philox(seed, segment, events, n_x):
    """Uniforms [events][n_x] of Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC 2011): counter (event, segment, block),
    key the seed, two 32-bit outputs per number."""
    low = 0xFFFFFFFF
    e = torch.arange(events, device=DEV, dtype=torch.int64)
    out = []
    for j in range((n_x + 1) // 2):
        c = [e & low, e >> 32, torch.full_like(e, segment), torch.full_like(e, j)]
        k0, k1 = seed & low, (seed >> 32) & low
        for _ in range(10):
            p0, p1 = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57
            c = [((p1 >> 32) & low) ^ c[1] ^ k0, p1 & low, ((p0 >> 32) & low) ^ c[3] ^ k1, p0 & low]
            k0, k1 = (k0 + 0x9E3779B9) & low, (k1 + 0xBB67AE85) & low
        for a, b in ((c[0], c[1]), (c[2], c[3])):
            out.append(((a << 21) | (b >> 11)).to(F64) * 2.0 ** -53)
    return torch.stack(out[:n_x], 1)


def _exact_adaptive(case, d):
    w, nb = d["weights"], G.Grid.BINS
    F = np.zeros(w.shape[:2] + (nb + 1,))
    for b in range(nb):
        F[..., b + 1] = F[..., b] + w[..., b] / w.sum(-1)
    F[..., nb] = 1
    F = _t(F)
    for k, (_, c, rows, _, _) in enumerate(_segment_events(case, d)):
        u = _philox(d["seed"], k, rows.stop - rows.start, d["procs"][0].n_x)
        for i in range(u.shape[1]):
            b = torch.searchsorted(F[c, i, 1:nb].contiguous(), u[:, i].contiguous(), right=True)
            d["x"][0][rows, i] = b.to(F64) / nb + (u[:, i] - F[c, i][b]) / ((F[c, i][b + 1] - F[c, i][b]) * nb)
    events, _ = _exact_forward(case, d)
    weights = w.copy()
    for _, c, rows, _, _ in _segment_events(case, d):
        ok = events[0]["ok"][rows].bool()
        n_ok = int(ok.sum())
        if n_ok:
            bins = (d["x"][0][rows][ok] * nb).long().clamp(0, nb - 1)
            for i in range(bins.shape[1]):
                weights[c, i] = torch.bincount(bins[:, i], minlength=nb).cpu().numpy() / n_ok
    return dict(events=events, x=d["x"][0], weights=weights)


@torch.no_grad()
def exact(case, seed):
    d = _inputs(case, seed)
    if case["task"] == "adaptive":
        return _exact_adaptive(case, d)
    events, msq = _exact_forward(case, d)
    if case["task"] == "forward":
        return dict(events=events, **({"msq": msq} if msq is not None else {}))
    if case["task"] in ("inverse", "whizard"):
        factors, x_out = _exact_inverse(case, d, events)
        if case["task"] == "inverse":
            return dict(events=events, factors=factors, x_out=x_out)
        e = events[0]
        return dict(p=e["p"], factors=factors, volumes=e["volume"], oks=e["ok"], x_out=x_out)
    g_x, loss, g_par = _exact_gradients(case, d, events)
    if case["task"] == "adjoint":
        return dict(g_x=g_x, loss=loss, g_par=g_par)
    return dict(events=events, g_x=g_x, g_par=g_par)
