"""Which kernels a call launches, and which sizes it refuses, against a stand-in of
the HIP runtime (hostrun.py): no GPU is used and no kernel runs."""
import numpy as np
import pytest

import hostrun
import test_gpu_dense as dense
import test_gpu_discrete as discrete
import test_gpu_potts as potts
import test_gpu_resident as resident
import test_gpu_wide_q as wide_q
import thrml_hip as th
from thrml_hip import workloads as wl


def _spin_factor_run(sites, chains):
    """The spin kernel's launches of one sweep over one block, or the error."""
    dev = th.Device(0)
    prog = th.FactorSamplingProgram(np.zeros(sites, np.uint8), 2, [th.SpinEBMFactor([np.arange(sites)], np.zeros(sites))],
                                    [np.arange(sites)], [], dev)
    st = prog.new_state(chains)
    hostrun.clear_launches()
    try:
        th.run_blocks(th.RngKey(1), prog, st, (), 1)
    except th.ThrmlError as e:
        return str(e)
    return hostrun.launches().get("discrete_spin_kernel<unsigned_char>", 0)


@pytest.mark.parametrize("sites,chains,runs", [(16148, 531900, True), (16145, 531900, True), (16149, 531900, False),
                                               (1, 699000, True), (13, 660000, True)])
def test_spin_factor_block_limit(sites, chains, runs):
    """(sites / 4) x chains below 2^31, whatever the sites are modulo 16."""
    assert ((sites + 3) // 4 * chains < 1 << 31) == runs
    got = hostrun.call(_spin_factor_run, sites, chains)
    assert got == 1 if runs else "must stay below 2^31" in got


def _potts_run(q, sites, chains):
    dev = th.Device(0)
    prog = th.CategoricalProgram(sites, q, np.zeros((0, 2)), np.zeros((0, q, q)), np.zeros((sites, q)),
                                 [np.arange(sites)], dev)
    st = prog.new_state(chains)
    hostrun.clear_launches()
    th.run_blocks(th.RngKey(1), prog, st, (), 1)
    return {k: n for k, n in hostrun.launches().items() if k.startswith("potts")}


@pytest.mark.parametrize("sites,chains,lanes", [(3906, 549791, 1), (3906, 549759, 2)])
def test_wide_categorical_block_limit(sites, chains, lanes):
    """Up to 2^31 - 1 (site, chain) items run; two lanes each, where that is the
    faster, while whole workgroups of them stay below 2^32 threads."""
    assert sites * chains in ((1 << 31) - 2, (1 << 31) - 2 - 32 * 3906)
    assert hostrun.call(_potts_run, 32, sites, chains) == {f"potts_wide_kernel<unsigned_char,{lanes}>": 1}


def _ising_kernels(prog, C, sched, cus=256):
    """The sweep kernels that a run with moments launches."""
    st = prog.new_state(C)
    m = th.MomentAccumulatorObserver(prog, th.ising_moment_spec([0], np.zeros((0, 2))))
    hostrun.clear_launches()
    m.sample_with_observation(th.RngKey(1), th.SamplingSchedule(*sched), st)
    return sorted(k for k in hostrun.launches() if "half" in k or k.startswith("resident") and "commit" not in k)


def _one_block_of_many(clamped, C):
    """512 free sites with 60 neighbours each among `clamped` clamped ones."""
    rng = np.random.default_rng(0)
    e = np.stack([np.repeat(np.arange(512), 60), 512 + rng.integers(0, clamped, 512 * 60)], axis=1)
    e = np.unique(e, axis=0).astype(np.uint32)
    n = 512 + clamped
    prog = th.IsingSamplingProgram(th.IsingEBM(n, e, np.zeros(n), np.zeros(len(e))), [np.arange(512)],
                                   [np.arange(512, n)], th.Device(0))
    return _ising_kernels(prog, C, (10, 30, 10))


@pytest.mark.parametrize("clamped,C,resident", [(20000, 256, True), (20000, 260, True), (54000, 256, True),
                                                (54000, 260, False)])
def test_resident_workgroups_that_lds_keeps_apart(clamped, C, resident):
    """Chains beyond one per compute unit cost a second turn where two
    workgroups' states and keystreams (n + 64 bytes per thread) do not fit one unit's LDS."""
    k = hostrun.call(_one_block_of_many, clamped, C)
    assert {x.startswith("resident") for x in k} == {resident}, k


def _lattice_on(cus, C):
    hostrun.fake.fake_set_cus(cus)
    n, edges, up, lo = th.make_nearest_neighbor_lattice(64, True)
    prog = th.IsingSamplingProgram(th.IsingEBM(n, edges, np.zeros(n), np.zeros(len(edges)), 1.0), [up, lo], [],
                                   th.Device(0))
    return _ising_kernels(prog, C, (500, 1, 1))


@pytest.mark.parametrize("cus,C,resident", [(256, 256, True), (32, 32, True), (32, 256, False)])
def test_resident_turns_count_the_compute_units(cus, C, resident):
    k = hostrun.call(_lattice_on, cus, C)
    assert {x.startswith("resident") for x in k} == {resident}, k


def _few_sites(free, clamped, C, sched):
    rng = np.random.default_rng(0)
    e = np.stack([np.repeat(np.arange(free), 6), free + rng.integers(0, clamped, free * 6)], axis=1)
    e = np.unique(e, axis=0).astype(np.uint32)
    n = free + clamped
    prog = th.IsingSamplingProgram(th.IsingEBM(n, e, np.zeros(n), np.zeros(len(e))), [np.arange(free)],
                                   [np.arange(free, n)], th.Device(0))
    return _ising_kernels(prog, C, sched)


def _random_graph(n, C, sched):
    e = th.erdos_renyi(n, 6.0 / (n - 1), 3)
    prog = th.IsingSamplingProgram(th.IsingEBM(n, e, np.zeros(n), np.zeros(len(e))),
                                   th.coloring_to_blocks(th.greedy_coloring(n, e)), [], th.Device(0))
    return _ising_kernels(prog, C, sched)


@pytest.mark.parametrize("f,args,resident", [
    # measured, us per segment:                     whole, block by block
    (_few_sites, (64, 1000, 32, (5, 10, 5)), True),        # 17, 27
    (_few_sites, (64, 60000, 32, (10, 10, 10)), False),    # 360, 51
    (_few_sites, (64, 60000, 32, (200, 3, 200)), True),    # 442, 980
    (_few_sites, (512, 60000, 256, (5, 10, 5)), False),    # 62, 29
    (_few_sites, (2048, 1000, 32, (10, 10, 10)), True),    # 27, 52
    (_random_graph, (60000, 200, (1, 10, 1)), False),      # 96, 85
    (_random_graph, (20000, 200, (4, 10, 4)), True),       # 101, 211
])
def test_a_segment_costs_its_way_into_and_out_of_lds(f, args, resident):
    """Every run between observations moves the whole state, clamped positions
    too, with the lanes of its largest block."""
    k = hostrun.call(f, *args)
    assert {x.startswith("resident") for x in k} == {resident}, k


def _wide_kernels(prog, C, sweeps=1):
    """The wide categorical kernels of a run, as (kernel and element, lanes)."""
    st = prog.new_state(C)
    hostrun.clear_launches()
    th.run_blocks(th.RngKey(1), prog, st, (), sweeps)
    return {tuple(k.rstrip(">").rsplit(",", 1)) for k in hostrun.launches() if "wide_kernel" in k}


def _lanes_of(i):
    q, n, C, m = wide_q.LANES[i][:4]
    prog, fp, _, _ = wide_q.lanes_programs(th.Device(0), q, n, C, m)
    return _wide_kernels(prog, C), _wide_kernels(fp, C)


@pytest.mark.parametrize("i", range(len(wide_q.LANES)))
def test_lanes_of_the_parity_cases(i):
    q, want = wide_q.LANES[i][0], wide_q.LANES[i][5:]
    t = "unsigned_char" if q <= 256 else "unsigned_short"
    for kernel, got, lanes in zip(("potts", "discrete"), hostrun.call(_lanes_of, i), want):
        assert got == {(f"{kernel}_wide_kernel<{t}", str(p)) for p in lanes}


def test_parity_cases_reach_every_lane_count():
    for wide, every in ((False, {1, 2, 4, 8, 16}), (True, {1, 2, 4, 8, 16, 64})):
        for kind in (5, 6):
            assert set().union(*(c[kind] for c in wide_q.LANES if (c[0] > 256) == wide)) == every


def _bias_only_lanes(q):
    prog, _ = potts.bias_only_program(th.Device(0), q)
    return {C: {int(lanes) for _, lanes in _wide_kernels(prog, C)} for C in potts.BIAS_ONLY_LANES[q]}


@pytest.mark.parametrize("q", potts.BIAS_ONLY_LANES)
def test_lanes_either_side_of_a_change(q):
    assert hostrun.call(_bias_only_lanes, q) == {C: {p} for C, p in potts.BIAS_ONLY_LANES[q].items()}


def _factor_lanes():
    kinds, q, factors, free = discrete.wide_factor_model()
    fs = [th.DiscreteEBMFactor(s, c, w) for s, c, w in factors]
    prog = th.FactorSamplingProgram(kinds, q, fs, free, [], th.Device(0))
    return {C: {int(lanes) for _, lanes in _wide_kernels(prog, C)} for C in discrete.FACTOR_LANES}


def test_factor_lanes_either_side_of_a_change():
    assert hostrun.call(_factor_lanes) == {C: {p} for C, p in discrete.FACTOR_LANES.items()}


def _resident_case(i):
    """The sweep kernels of a whole-run parity case: its run, its observed run."""
    _, graph, C, sweeps, _ = resident.CASES[i]
    ebm, prog = resident.case_program(th.Device(0), graph)
    st = prog.new_state(C)
    sched = resident.observed_schedule(prog)
    seen = []
    for run in (lambda: th.run_blocks(th.RngKey(1), prog, st, (), sweeps),
                lambda: th.estimate_moments(th.RngKey(1), [0], ebm.edges, prog, th.SamplingSchedule(*sched), st)):
        hostrun.clear_launches()
        run()
        seen.append({k: n for k, n in hostrun.launches().items() if "half" in k or "_kernel<" in k and "resident" in k})
    return seen, sched[1]


@pytest.mark.parametrize("i", range(len(resident.CASES)), ids=[c[0].replace(" ", "-") for c in resident.CASES])
def test_kernels_of_the_whole_run_cases(i):
    """One launch for the run, one per observation for the observed one."""
    kernel = "resident_" + resident.CASES[i][4]
    seen, n_obs = hostrun.call(_resident_case, i)
    assert seen == [{kernel: 1}, {kernel: n_obs}]


def test_whole_run_cases_reach_every_kernel():
    assert {c[4] for c in resident.CASES} == {f"reg_kernel<{e}>" for e in (2, 4, 10)} | {
        f"stream_kernel<{p}>" for p in range(2, 9)}


def _dense_kernels(V, H, C):
    prog = th.RbmProgram(np.zeros((V, H)), np.zeros(V), np.zeros(H), 1.0, th.Device(0))
    st = prog.new_state(C)
    seen = []
    for blk in (0, 1):
        hostrun.clear_launches()
        prog.half_sweep(st, blk, np.zeros((C, 8), np.uint32))
        seen += [k for k in hostrun.launches() if k.startswith("dense")]
    return seen


@pytest.mark.parametrize("V,H,C", dense.SMALL_TILES)
def test_dense_tiles_of_the_parity_cases(V, H, C):
    assert hostrun.call(_dense_kernels, V, H, C) == ["dense_small_kernel"] * 2
    assert hostrun.call(_dense_kernels, V, H, dense.LARGE_TILES_C) == ["dense_half_kernel<false>"] * 2


def _moment_kernels(C):
    """Of two observations of a graph too large for whole runs, the first before any
    sweep."""
    ebm, blocks = wl.er_ising(70_001, 3.0, 0.2, 0.0, 0.3)
    prog = th.IsingSamplingProgram(ebm, blocks, [], th.Device(0))
    st = prog.new_state(C)
    hostrun.clear_launches()
    th.estimate_moments(th.RngKey(1), [0], ebm.edges, prog, th.SamplingSchedule(0, 2, 1), st)
    return {k: n for k, n in hostrun.launches().items() if k.startswith("moments")}


@pytest.mark.parametrize("C,kernels", [(32, {"moments_kernel<unsigned_int>": 1, "moments_kernel<unsigned_long>": 1}),
                                       (33, {"moments_kernel<unsigned_long>": 2})])
def test_moment_sums_read_the_low_halves(C, kernels):
    assert hostrun.call(_moment_kernels, C) == kernels


def _export_kernels(n):
    prog = th.IsingSamplingProgram(th.IsingEBM(n, np.zeros((0, 2)), np.zeros(n), []), [np.arange(n)], [], th.Device(0))
    st = prog.new_state(100)
    seen = []
    for dt in (np.uint8, np.float32):
        hostrun.clear_launches()
        st.get_block(0, dt)
        seen += hostrun.launches()
    return seen


@pytest.mark.parametrize("n,u8,f32", [(8, "_narrow", "_narrow"), (9, "_narrow", ""), (16, "_narrow", ""), (17, "", "")])
def test_export_of_few_positions(n, u8, f32):
    assert hostrun.call(_export_kernels, n) == [f"unpack{u8}_kernel<unsigned_char>", f"unpack{f32}_kernel<float>"]
