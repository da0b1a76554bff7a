"""Device memory and waits of the library's host code, against a stand-in of the
HIP runtime (hostrun.py): no GPU is used and no kernel runs."""
import ctypes
import os
import threading

import numpy as np
import pytest

import hostrun
import thrml_hip as th
from thrml_hip import _lib

def _lattice(dev, L=64):
    n, edges, up, lo = th.make_nearest_neighbor_lattice(L, True)
    return th.IsingSamplingProgram(th.IsingEBM(n, edges, np.zeros(n), np.zeros(len(edges)), 1.0), [up, lo], [],
                                   dev)


def _rbm(dev):
    rng = np.random.default_rng(0)
    return th.RbmProgram(rng.normal(0, 1, (64, 96)), np.zeros(64), np.zeros(96), 1.0, dev)


def _low_memory(what):
    """`what` on a device whose memory holds it only without the blocks that the
    context keeps for its next objects."""
    fake = hostrun.fake
    dev = th.Device(0)
    prog = _rbm(dev) if what == "dense half-sweep" else _lattice(dev)
    st = prog.new_state(4096)
    for s in [_lattice(dev).new_state(1 << 15) for _ in range(2)]:
        s.close()  # 16 MiB of words each, kept
    fake.fake_set_capacity(fake.fake_live_bytes())
    if what == "stream keys":
        th.run_blocks(th.RngKey(1), prog, st, (), 3)
    elif what == "state transfer":
        st.set_global(np.zeros((4096, prog.n_total), np.uint8))
    elif what == "large state transfer":
        big = prog.new_state(1 << 14)
        fake.fake_set_capacity(fake.fake_live_bytes() + (112 << 20))
        big.get_block(0, np.float32)  # 128 MiB
    elif what == "dense half-sweep":
        prog.half_sweep(st, 0, np.zeros((4096, 8), np.uint32))
    elif what == "program":
        _lattice(dev, 96)
    assert fake.hipGetLastError() == 0  # a later launch's check does not find the refused attempt
    dev.close()


@pytest.mark.parametrize("what", ["stream keys", "state transfer", "large state transfer", "dense half-sweep",
                                  "program"])
def test_kept_blocks_make_room(what):
    """An allocation that the device refuses is tried again without the blocks
    that the context keeps, whoever makes it."""
    hostrun.call(_low_memory, what)


def _read_during_a_run():
    """Whether a state can be read by a second thread while sample_states is
    between two of its launches."""
    dev = th.Device(0)
    prog = _csr(dev)
    st, other = prog.new_state(4), prog.new_state(4)
    reads = []

    @ctypes.CFUNCTYPE(None)
    def launched():
        hostrun.fake.fake_on_launch(None)
        t = threading.Thread(target=lambda: reads.append(other.get_block(0)))
        t.start()
        t.join(timeout=10)
        reads.append("run goes on")

    hostrun.fake.fake_on_launch(launched)
    th.sample_states(th.RngKey(1), prog, th.SamplingSchedule(1, 3, 1), st)
    return [r if isinstance(r, str) else "read" for r in reads]


def test_transfers_do_not_wait_for_a_run():
    assert hostrun.call(_read_during_a_run) == ["read", "run goes on"]


def _transfer_memory():
    """Device memory after transfers of several sizes, whole states and blocks."""
    dev = th.Device(0)
    prog = _lattice(dev)
    st = prog.new_state(1 << 13)
    small = prog.new_state(3)
    st.get_block(0)  # 16 MiB
    fake = hostrun.fake
    before, n = fake.fake_live_bytes(), fake.fake_mallocs()
    st.get_global()
    grown = fake.fake_live_bytes() - before
    for _ in range(3):
        st.get_block(0)
        st.get_global()
        small.set_global(small.get_global())
    st.get_block(0, np.float32)
    st.get_block(0)
    return grown, fake.fake_mallocs() - n, fake.fake_live_bytes() - before


def test_one_block_serves_transfers_of_every_size():
    """The block grows to the largest transfer of up to 64 MiB and serves the
    smaller ones."""
    grown, mallocs, end = hostrun.call(_transfer_memory)
    assert grown == 16 << 20          # 32 MiB in place of 16
    assert end == 48 << 20            # 64 MiB in place of 16
    assert mallocs == 2


def _moment_memory(L):
    """Bytes of a spec of all nodes and edges of a torus, allocated at its creation, by
    a run into device memory and by a run into host memory, and the
    allocations that a second spec and run make."""
    dev = th.Device(0)
    prog = _lattice(dev, L)
    st = prog.new_state(2)
    n, edges, _, _ = th.make_nearest_neighbor_lattice(L, True)
    fake = hostrun.fake
    sched = th.SamplingSchedule(1, 1, 1)
    th.run_blocks(th.RngKey(1), prog, st, (), 1)

    def spec():
        return th.MomentAccumulatorObserver(prog, th.ising_moment_spec(np.arange(n), edges))

    steps = [fake.fake_live_bytes()]
    m = spec()
    steps.append(fake.fake_live_bytes())
    sums = np.zeros(n + len(edges), np.int64)
    _lib.check(_lib.load().thrml_moments_run(prog._h, 1, sched._c(), st._h, m._h, sums.ctypes.data,
                                             sums.ctypes.data, 1))
    steps.append(fake.fake_live_bytes())
    m.sample_with_observation(th.RngKey(1), sched, st)
    steps.append(fake.fake_live_bytes())
    m.close()
    before = fake.fake_mallocs()
    m = spec()
    m.sample_with_observation(th.RngKey(1), sched, st)
    return np.diff(steps).tolist(), fake.fake_mallocs() - before


def test_moment_specs_hold_host_sums_for_host_outputs_only():
    n, e = 1024 * 1024, 2 * 1024 * 1024
    steps, again = hostrun.call(_moment_memory, 1024)
    # 12 bytes per counter and 4 per table entry; 8 per sum on the host, unless a
    # kept block holds them
    assert steps[:2] == [16 * (n + e), 0] and steps[2] in (0, 8 * (n + e))
    assert again == 0  # below the pool's largest block


def _stream_changes():
    lib = ctypes.CDLL(os.path.join(os.path.dirname(hostrun.FAKE), "libpooltest.so"))
    lib.pool_kept_across_stream_change.restype = ctypes.c_uint64
    return lib.pool_kept_across_stream_change(ctypes.c_uint64(20000))


def test_memory_of_the_old_stream_is_not_kept():
    """A buffer whose last use lies on the old stream is never handed to an object
    on the new one, also when it is let go of while the stream changes."""
    assert hostrun.call(_stream_changes) == 0


def _graph():
    e = np.unique(np.sort(np.random.default_rng(1).integers(0, 90, (300, 2)), axis=1), axis=0)
    e = e[e[:, 0] != e[:, 1]].astype(np.uint32)
    return 90, e, th.coloring_to_blocks(th.greedy_coloring(90, e))


def _csr(dev):
    n, e, blocks = _graph()
    return th.IsingSamplingProgram(th.IsingEBM(n, e, np.zeros(n), np.zeros(len(e))), blocks, [], dev)


def _potts(dev):
    n, e, blocks = _graph()
    return th.CategoricalProgram(n, 5, e, np.zeros((len(e), 5, 5)), np.zeros((n, 5)), blocks, dev)


def _factors(dev):
    n, e, blocks = _graph()
    f = th.SpinEBMFactor([e[:, 0], e[:, 1]], np.zeros((len(e), 1, 1)))
    return th.FactorSamplingProgram(np.zeros(n, np.uint8), 2, [f], blocks, [], dev)


def _nothing(dev):
    return dev


def _energy(prog):
    st = prog.new_state(3)
    return lambda: th.energy(prog, st)


# name: (what stands before, the call on it)
CALLS = {
    "lattice program": (_nothing, _lattice),
    "irregular program": (_nothing, _csr),
    "categorical program": (_nothing, _potts),
    "factor program": (_nothing, _factors),
    "dense program": (_nothing, _rbm),
    "moments": (_csr, lambda p: th.MomentAccumulatorObserver(p, th.ising_moment_spec(np.arange(90), _graph()[1]))),
    "observer": (_csr, lambda p: th.MomentAccumulatorObserver(p, [[[0], [1, 2, 3]]])),
    "hinton_init": (lambda dev: (lambda p: (p, p.new_state(4)))(_rbm(dev)),
                    lambda s: th.hinton_init(th.RngKey(1), s[0], state=s[1])),
    "spin energies": (lambda dev: _energy(_csr(dev)), lambda f: f()),
    "categorical energies": (lambda dev: _energy(_potts(dev)), lambda f: f()),
    "factor energies": (lambda dev: _energy(_factors(dev)), lambda f: f()),
    "dense energies": (lambda dev: _energy(_rbm(dev)), lambda f: f()),
}


def _each_allocation_fails(name):
    before, do = CALLS[name]
    fake = hostrun.fake
    _lattice(th.Device(0))  # the device's one-time checks
    fails = 0
    for nth in range(1, 40):
        dev = th.Device(0)
        what = before(dev)
        fake.fake_fail_malloc(nth)
        try:
            do(what)
            done = True
        except th.ThrmlError as e:
            assert "device allocation of" in str(e)
            done = False
        assert fake.fake_pending_host() == 0, f"allocation {nth} refused: copies of freed memory are queued"
        fake.fake_fail_malloc(0)
        assert fake.hipGetLastError() == 0
        if done:
            return fails
        do(what)  # and it works once there is memory
        fails += 1
    raise AssertionError("no end to the allocations")


@pytest.mark.parametrize("name", CALLS)
def test_no_copy_outlives_its_memory(name):
    """Whichever allocation fails, the copies that a call has queued from or to
    its own or the caller's memory have ended when it returns."""
    assert hostrun.call(_each_allocation_fails, name) >= 1
