"""Device memory and waits of the library's host code, against a stand-in of the
HIP runtime (hostrun.py): no GPU is used and no kernel runs."""
import numpy as np
import pytest

import hostrun
import thrml_hip as th

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
