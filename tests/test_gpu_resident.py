"""Whole-run kernels of small Ising programs (k_resident.hip): every chain's
sweeps in one launch, from the oracle's states bit for bit.

The cases lie where the kernels' layout turns: sites per block around a
wave and around 16-site keystream blocks, blocks with more keystream blocks
than a workgroup has lanes (several parts per sweep), slot counts of 0, odd,
4 | 5 (register and streaming kernels) and above 16 (several entries per
slice), more blocks than waves, clamped blocks, 1, 64 and 65 chains, runs
longer than a phase, and observations that cut a run into segments."""
import numpy as np
import pytest

import pyoracle as orc
import thrml_hip as th
from conftest import log_case

pytestmark = pytest.mark.gpu


def _random_graph(rng, n, degree):
    m = int(n * degree / 2)
    e = rng.integers(0, n, (4 * m + 8, 2))
    e = np.sort(e[e[:, 0] != e[:, 1]], axis=1)
    return np.unique(e, axis=0)[:m].astype(np.uint32) if m else np.zeros((0, 2), np.uint32)


def _torus(L):
    n, edges, up, lo = th.make_nearest_neighbor_lattice(L, True)
    return n, edges, [up, lo], []


def _sparse(n, degree, hub=0, seed=1):
    rng = np.random.default_rng(seed)
    e = _random_graph(rng, n, degree)
    if hub:
        e = np.concatenate([e, np.stack([np.zeros(hub), 1 + np.arange(hub)], axis=1).astype(np.uint32)])
        e = np.unique(np.sort(e, axis=1), axis=0).astype(np.uint32)
    return n, e, th.coloring_to_blocks(th.greedy_coloring(n, e)), []


def _ring(n, blocks):
    """A cycle coloured with `blocks` colours (n a multiple of blocks)."""
    u = np.arange(n, dtype=np.uint32)
    e = np.stack([u, (u + 1) % n], axis=1).astype(np.uint32)
    return n, e, [th.Block(u[b::blocks]) for b in range(blocks)], []


def _bipartite_clamped(n, degree):
    """Three bands, the middle one clamped: sites with clamped tails only."""
    rng = np.random.default_rng(3)
    a, b, c = np.arange(n), n + np.arange(n), 2 * n + np.arange(n)
    e = np.concatenate([np.stack([rng.choice(a, n * degree), rng.choice(b, n * degree)], 1),
                        np.stack([rng.choice(b, n * degree), rng.choice(c, n * degree)], 1)])
    e = np.unique(e, axis=0).astype(np.uint32)
    return 3 * n, e, [th.Block(a), th.Block(c)], [th.Block(b)]


def _regular(n, degree):
    """Two bands of n sites with `degree` neighbours each in the other."""
    i = np.arange(n)
    e = np.concatenate([np.stack([i, n + (i + 37 * k) % n], axis=1) for k in range(degree)])
    return 2 * n, e.astype(np.uint32), [th.Block(i), th.Block(n + i)], []


# name, graph, chains, sweeps, kernel (test_host_dispatch.py holds the launches to it)
CASES = [
    ("one wave", _torus(10), 1, 40, "reg_kernel<2>"),
    ("one wave, 65 chains", _torus(4), 65, 300, "reg_kernel<2>"),
    ("register kernel, 2 entries", _torus(32), 64, 37, "reg_kernel<2>"),
    ("register kernel, 4 entries", _torus(64), 3, 19, "reg_kernel<4>"),
    ("register kernel, 6 entries", _torus(74), 2, 9, "reg_kernel<10>"),
    ("register kernel, 8 entries", _torus(80), 2, 60, "reg_kernel<10>"),
    ("register kernel, 10 entries", _torus(96), 2, 60, "reg_kernel<10>"),
    ("streaming kernel, 4 slots, several parts", _torus(140), 200, 5, "stream_kernel<2>"),
    ("no edges", _sparse(77, 0), 5, 21, "reg_kernel<2>"),
    ("odd slot counts", _sparse(501, 3.0), 7, 33, "stream_kernel<5>"),
    ("several entries per slice", _sparse(700, 14.0, hub=90), 9, 12, "stream_kernel<8>"),
    ("wide slices", _sparse(1030, 22.0), 2, 9, "stream_kernel<8>"),
    ("eight slots", _regular(130, 8), 3, 14, "stream_kernel<4>"),
    ("twelve slots", _regular(1100, 12), 2, 14, "stream_kernel<6>"),
    ("fourteen slots", _regular(640, 14), 65, 14, "stream_kernel<7>"),
    ("several parts, ragged", _sparse(17011, 5.0), 130, 4, "stream_kernel<3>"),
    ("more blocks than waves", _ring(600, 30), 4, 17, "stream_kernel<2>"),
    ("uneven blocks", _ring(1023, 3), 2, 70, "reg_kernel<4>"),
    ("clamped block between", _bipartite_clamped(300, 3), 6, 25, "stream_kernel<3>"),
]


def case_program(device, graph):
    n, edges, free, clamped = graph
    rng = np.random.default_rng(5)
    ebm = th.IsingEBM(n, edges, rng.normal(0, 0.4, n), rng.normal(0.1, 0.5, len(edges)), 0.9)
    return ebm, th.IsingSamplingProgram(ebm, free, clamped, device)


def observed_schedule(prog):
    """Segments long enough for whole runs, which a lattice's own moment counters
    compete with."""
    return (3, 3, 20) if prog.kind == "lattice" else (3, 3, 4)


@pytest.mark.parametrize("name,graph,chains,sweeps", [c[:4] for c in CASES],
                         ids=[c[0].replace(" ", "-") for c in CASES])
def test_whole_run_matches_oracle(device, name, graph, chains, sweeps):
    log_case(f"resident run: {name}")
    n, edges, free, clamped = graph
    ebm, prog = case_program(device, graph)
    o = orc.Ising(n, ebm.edges, ebm.biases, ebm.weights, ebm.beta, [b.nodes for b in free],
                  [b.nodes for b in clamped])
    init = np.random.default_rng(6).integers(0, 2, (chains, prog.n_total)).astype(np.uint8)
    st = prog.new_state(chains)
    st.set_global(init)
    th.run_blocks(th.RngKey(77), prog, st, (), sweeps)
    want, _ = o.run_blocks(77, init, sweeps)
    assert np.array_equal(st.get_global(), want)
    # again from where it stands, observed: segments of a few sweeps
    pairs = ebm.edges if len(edges) else np.zeros((0, 2), np.uint32)
    nodes = np.arange(n)
    sched = observed_schedule(prog)
    ns, es = th.estimate_moments(th.RngKey(78), nodes, pairs, prog, th.SamplingSchedule(*sched), st,
                                 return_sums=True)
    wn, we, want, _ = o.estimate_moments(78, sched, want, nodes, pairs)
    assert np.array_equal(ns, wn) and np.array_equal(es, we)
    assert np.array_equal(st.get_global(), want)


def test_overflowing_lattice_sums(device):
    """Infinite weights: opposite infinities sum to NaN, which the lattice
    kernel's threshold table decides up; such a program keeps that rule."""
    log_case("lattice with infinite weights")
    n, edges, up, lo = th.make_nearest_neighbor_lattice(32, True)
    rng = np.random.default_rng(9)
    w = rng.normal(0.2, 0.4, len(edges)).astype(np.float32)
    w[::7] = np.inf
    big = th.IsingSamplingProgram(th.IsingEBM(n, edges, np.zeros(n), w, 1.0), [up, lo], [], device)
    init = rng.integers(0, 2, (4, n)).astype(np.uint8)
    st = big.new_state(4)
    st.set_global(init)
    th.run_blocks(th.RngKey(1), big, st, (), 1)
    got = st.get_global()
    # one block after the other by hand: a site whose sum is NaN is up
    state = {int(v): init[:, i] for i, v in enumerate(np.concatenate([up.nodes, lo.nodes]))}
    nan_sites = 0
    for blk, base in ((up, 0), (lo, len(up))):
        for i, node in enumerate(blk.nodes):
            slots = np.concatenate([np.where(edges[:, 0] == node)[0], np.where(edges[:, 1] == node)[0]])
            tails = np.where(edges[slots, 0] == node, edges[slots, 1], edges[slots, 0])
            s = np.array([2.0 * state[int(t)] - 1.0 for t in tails])
            with np.errstate(invalid="ignore"):
                g = (w[slots][:, None] * s).sum(0)
            nan_sites += int(np.isnan(g).sum())
            assert (got[np.isnan(g), base + i] == 1).all()
        for i, node in enumerate(blk.nodes):
            state[int(node)] = got[:, base + i]
    assert nan_sites > 10
