"""Adaptive grids on the GPU against the oracle's restatement: the randoms drawn from the grid
(Philox4x32-10 and the inverse distribution function) bit for bit, the weight update exactly,
and a short adaptation loop."""
import numpy as np
import pytest

import oracle
from gpu_phs_amd import workloads as W

pytestmark = pytest.mark.gpu


def _plan(proc, counts, **cfg):
    import torch
    import gpu_phs_amd as G
    ph = G.ProcessHandle(proc)
    segs, bufs = [], []
    for c, n in enumerate(counts):
        if n == 0:
            continue
        x = torch.zeros((n, proc.n_x), dtype=torch.float64, device="cuda")
        b = G.EventBuffers.allocate(x, proc.n_out)
        segs.append((ph, c, b))
        bufs.append(b)
    return ph, G.Plan(segs, **cfg), bufs, [c for c, n in enumerate(counts) if n]


@pytest.mark.parametrize("cfg", [dict(), dict(block=64, ept=3)])
def test_generate_matches_oracle(cfg):
    import torch
    import gpu_phs_amd as G
    proc = W.process_c1()
    ph, plan, bufs, chans = _plan(proc, [3001, 0, 777], **cfg)
    grid = G.Grid(ph)
    rng = np.random.default_rng(9)
    w = rng.random(grid.shape) + 0.01
    w[0, 2, 4] = 0.0
    grid.set_weights(w)
    seed = 0x1234_5678_9ABC
    grid.generate(plan, seed)
    torch.cuda.synchronize()
    F = oracle.grid_cdf(w)
    for s, (b, c) in enumerate(zip(bufs, chans)):
        got = b.x.cpu().numpy()
        want = oracle.grid_sample(F[c], oracle.grid_uniforms(seed, s, got.shape[0], proc.n_x))
        assert np.array_equal(got, want)


def test_update_matches_oracle_and_adapts():
    import torch
    import gpu_phs_amd as G
    proc = W.process_c1()
    counts = [20000, 15000, 5000]
    ph, plan, bufs, chans = _plan(proc, counts)
    grid = G.Grid(ph)
    w = grid.weights()
    assert np.allclose(w, 0.1)
    for it in range(3):
        grid.generate(plan, 1000 + it)
        plan.run()
        grid.update(plan)
        torch.cuda.synchronize()
        x = np.concatenate([b.x.cpu().numpy() for b in bufs])
        ok = np.concatenate([b.ok.cpu().numpy().astype(bool) for b in bufs])
        ch = np.repeat(chans, [b.x.shape[0] for b in bufs])
        want = oracle.grid_update(w, x, ok, ch)
        w = grid.weights()
        assert np.array_equal(w, want)
    # the weights now follow where accepted events lie: every dimension sums to one
    assert np.allclose(w.sum(axis=2), 1.0)


@pytest.mark.parametrize("n_out,counts,cfg", [
    (4, [1], dict()),                                   # one event
    (2, [128 * 256], dict()),                           # as many tiles as the kernel for few takes
    (2, [128 * 256 + 1], dict()),                       # one more
    (2, [1025 * 256 + 7], dict()),                      # one tile more than the workgroups of the histogram
    (3, [1000, 255, 0, 64, 1, 4097], dict(block=64)),   # odd n_x: threads without an element; many short segments
    (6, [300, 70001, 2], dict(block=64, ept=4)),        # several tiles per run, runs that end inside a range
    (4, [400_000, 1, 300_000], dict()),                 # more elements per thread than a private count holds
])
def test_update_counts_every_accepted_event(n_out, counts, cfg):
    """The histogram at its edges: the counts are whole numbers, so the weights are exact."""
    import torch
    import gpu_phs_amd as G
    proc = W.process_shapes(n_out, 3)
    counts = (counts + [0] * proc.n_channels)[:proc.n_channels]
    ph, plan, bufs, chans = _plan(proc, counts, **cfg)
    gen = torch.Generator(device="cuda").manual_seed(5)
    for b in bufs:
        b.x.copy_(torch.rand(b.x.shape, generator=gen, device="cuda", dtype=torch.float64) ** 2)
        b.ok.copy_(torch.rand(b.ok.shape, generator=gen, device="cuda") < 0.7)
    bufs[0].x.view(-1)[0], bufs[0].x.view(-1)[1] = 1.0, 0.0   # the ends of the range
    grid = G.Grid(ph)
    w = grid.weights()
    grid.update(plan)
    x = np.concatenate([b.x.cpu().numpy() for b in bufs])
    ok = np.concatenate([b.ok.cpu().numpy().astype(bool) for b in bufs])
    ch = np.repeat(chans, [b.x.shape[0] for b in bufs])
    assert np.array_equal(grid.weights(), oracle.grid_update(w, x, ok, ch))


@pytest.mark.parametrize("n_out,counts,cfg", [
    (2, [1], dict()),
    (3, [65, 0, 4097, 1], dict(block=64)),          # odd rows: 8-byte words; several runs per workgroup
    (4, [4097 * 256 + 63], dict()),                 # more tiles than workgroups
    (6, [64, 63, 300_001], dict(block=128, ept=2)),
])
def test_generate_edges_match_oracle(n_out, counts, cfg):
    """Draws at the edges of the kernel's tables: bins without weight at both ends and in a row, weights over
    many orders of magnitude (several bounds inside one cell of the first-bin table), one full bin."""
    import torch
    import gpu_phs_amd as G
    proc = W.process_shapes(n_out, 3)
    counts = (counts + [0] * proc.n_channels)[:proc.n_channels]
    ph, plan, bufs, chans = _plan(proc, counts, **cfg)
    grid = G.Grid(ph)
    rng = np.random.default_rng(n_out)
    w = 10.0 ** rng.uniform(-6, 0, grid.shape)
    w[:, 0, 0] = w[:, 0, 9] = 0.0
    w[:, 1, 3:7] = 0.0
    w[0, 1, :9] = 0.0
    grid.set_weights(w)
    seed = 0xFEDC_BA98_7654_3210
    grid.generate(plan, seed)
    torch.cuda.synchronize()
    F = oracle.grid_cdf(w)
    for s, (b, c) in enumerate(zip(bufs, chans)):
        got = b.x.cpu().numpy()
        assert np.array_equal(got, oracle.grid_sample(F[c], oracle.grid_uniforms(seed, s, got.shape[0], proc.n_x)))


@pytest.mark.parametrize("n_out,counts,cfg,bin_", [
    # 140 tiles, a workgroup each: 64 elements a thread, all in one bin, one more than its private count holds
    (4, [140 * 4096], dict(block=256, ept=16), 3),
    (4, [140 * 4096], dict(block=256, ept=16), 9),
    # 1025 tiles on 1024 workgroups: one of two tiles
    (4, [1024 * 512 + 1], dict(block=256, ept=2), None),
    # 11 randoms: 6 of 512 threads without an element; 400 tiles of 42 segments on 128 workgroups, whose ranges
    # hold the ends of several segments and channels
    (5, [65 + 613 * k % 997 for k in range(42)], dict(block=64, ept=1), None),
    # one to ten tiles of 1024 events and a last one that is a pass of 64 events, or a batch of 8, or next to it
    (4, [1024 * (12 - k) + n for k, n in enumerate([64, 65, 63, 511, 512, 513, 575, 576, 577, 1, 128])] + [12 * 1024] * 4,
     dict(block=256, ept=4), None),
])
def test_update_counts_on_many_tiles(n_out, counts, cfg, bin_):
    """The histogram of more than 128 tiles where its loops begin and end: threads that hand over their counts in
    the middle of a range, threads without an element, ranges across segments, whole batches and what is left."""
    import torch
    import gpu_phs_amd as G
    proc = W.process_shapes(n_out, 3)
    counts = (counts + [0] * proc.n_channels)[:proc.n_channels]
    ph, plan, bufs, chans = _plan(proc, counts, **cfg)
    assert plan.info()["n_tiles"] > 128
    gen = torch.Generator(device="cuda").manual_seed(6)
    for b in bufs:
        if bin_ is None:
            b.x.copy_(torch.rand(b.x.shape, generator=gen, device="cuda", dtype=torch.float64) ** 2)
            b.ok.copy_(torch.rand(b.ok.shape, generator=gen, device="cuda") < 0.7)
        else:
            b.x.fill_((bin_ + 0.5) / 10)
            b.ok.fill_(1)
    grid = G.Grid(ph)
    w = grid.weights()
    grid.update(plan)
    x = np.concatenate([b.x.cpu().numpy() for b in bufs])
    ok = np.concatenate([b.ok.cpu().numpy().astype(bool) for b in bufs])
    ch = np.repeat(chans, [b.x.shape[0] for b in bufs])
    assert np.array_equal(grid.weights(), oracle.grid_update(w, x, ok, ch))


@pytest.mark.parametrize("n_out,segments,cfg,accept", [
    # a channel of one more tile than the kernel of a tile per workgroup takes, and one of as many
    (2, [(0, 193 * 256)], dict(), 0.7),
    (2, [(0, 192 * 256)], dict(), 0.7),
    # as many events as it takes, and one more
    (4, [(k, 34_952) for k in range(14)] + [(14, 34_960)], dict(), 0.7),
    (4, [(k, 34_952) for k in range(14)] + [(14, 34_961)], dict(), 0.7),
    # 5 randoms: 2 of 512 threads without an element; ranges across many segments of two channels in turn
    (3, [(k % 2, (65, 64, 1, 130, 63)[k % 5]) for k in range(500)], dict(block=64, ept=1), 0.7),
    # tiles of 1024 events, the last of a segment a pass of 64 events, or a batch of 8, or next to it
    (4, [(0, 200 * 1024)] + [(1 + k, 1024 * (k % 3) + n) for k, n in enumerate([64, 65, 63, 511, 512, 513, 575, 576, 577, 1, 128])],
     dict(block=256, ept=4), 0.7),
    # whole waves without an accepted event, and none at all
    (4, [(0, 300 * 256), (1, 300 * 256)], dict(), 0.002),
    (4, [(0, 300 * 256), (1, 5)], dict(), 0.0),
])
def test_update_counts_by_either_kernel(n_out, segments, cfg, accept):
    """The histogram on both sides of the rule that picks its kernel, and where the one for many tiles begins and ends
    a pass, a batch or a segment; randoms of rejected events, NaN here, do not matter."""
    import torch
    import gpu_phs_amd as G
    proc = W.process_shapes(n_out, 3)
    ph = G.ProcessHandle(proc)
    gen = torch.Generator(device="cuda").manual_seed(7)
    segs = []
    for c, n in segments:
        b = G.EventBuffers.allocate(torch.rand((n, proc.n_x), generator=gen, device="cuda", dtype=torch.float64) ** 2, n_out)
        b.ok.copy_(torch.rand(n, generator=gen, device="cuda") < accept)
        b.x[b.ok == 0] = float("nan")
        segs.append((ph, c, b))
    plan = G.Plan(segs, **cfg)
    grid = G.Grid(ph)
    w = grid.weights()
    grid.update(plan)
    x = np.concatenate([b.x.cpu().numpy() for _, _, b in segs])
    ok = np.concatenate([b.ok.cpu().numpy().astype(bool) for _, _, b in segs])
    ch = np.concatenate([np.full(b.ok.shape[0], c) for _, c, b in segs])
    assert np.array_equal(grid.weights(), oracle.grid_update(w, np.nan_to_num(x), ok, ch))


@pytest.mark.parametrize("n_out", [7, 8, 12])
def test_grids_of_large_trees(n_out):
    """Trees above six particles: the draw's tables in LDS grow with the randoms (2,640 bytes each, 84 KB for
    twelve particles), as does the histogram's."""
    import torch
    import gpu_phs_amd as G
    proc = W.process_large(n_out)
    counts = [700, 33_000][:proc.n_channels]
    ph, plan, bufs, chans = _plan(proc, counts)
    grid = G.Grid(ph)
    w = np.random.default_rng(n_out).random(grid.shape) + 0.01
    grid.set_weights(w)
    grid.generate(plan, 77)
    torch.cuda.synchronize()
    F = oracle.grid_cdf(w)
    for s, (b, c) in enumerate(zip(bufs, chans)):
        got = b.x.cpu().numpy()
        assert np.array_equal(got, oracle.grid_sample(F[c], oracle.grid_uniforms(77, s, got.shape[0], proc.n_x)))
    plan.run()
    grid.update(plan)
    x = np.concatenate([b.x.cpu().numpy() for b in bufs])
    ok = np.concatenate([b.ok.cpu().numpy().astype(bool) for b in bufs])
    ch = np.repeat(chans, [b.x.shape[0] for b in bufs])
    assert np.array_equal(grid.weights(), oracle.grid_update(w, x, ok, ch))
