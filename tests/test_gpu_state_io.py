"""Whole-state transfers (thrml_state_set_global / get_global) and the tiled
import and export kernels: rows around 4 positions per lane, 64 per tile and
256 per wave, chains around 16, 64 and 65 per wave or tile, u8 and f32, every
program kind, against the values written and the per-block reads; a rejected
value anywhere leaves the state as it was and names its block; objects made
from memory that earlier ones let go of start clean."""
import numpy as np
import pytest

import pyoracle as orc
import thrml_hip as th
from conftest import log_case

pytestmark = pytest.mark.gpu


def _ising(n, device):
    e = np.stack([np.arange(n - 1), np.arange(1, n)], axis=1)
    blocks = [np.arange(0, n, 2), np.arange(1, n, 2)]
    return th.IsingSamplingProgram(th.IsingEBM(n, e, np.zeros(n), np.zeros(n - 1)), blocks, [], device)


@pytest.mark.parametrize("n", [2, 3, 5, 63, 66, 129, 255, 258, 515])
@pytest.mark.parametrize("C", [1, 15, 17, 64, 65])
def test_spin_state_round_trip(device, n, C):
    log_case(f"spin state io n={n} C={C}")
    prog = _ising(n, device)
    rng = np.random.default_rng(n * C)
    x = rng.integers(0, 2, (C, n)).astype(np.uint8)
    st = prog.new_state(C)
    assert not st.get_global().any()  # a new state is all down, whatever its memory held
    st.set_global(x)
    assert np.array_equal(st.get_global(), x)
    parts = [st.get_block(b) for b in range(2)]
    assert np.array_equal(np.concatenate(parts, axis=1), x)
    assert np.array_equal(st.get_block(1, np.float32), parts[1].astype(np.float32))
    y = 1 - x
    st.set_block(1, y[:, len(prog.free_blocks[0]):].astype(np.float32))
    x[:, len(prog.free_blocks[0]):] = y[:, len(prog.free_blocks[0]):]
    assert np.array_equal(st.get_global(), x)
    st.set_global(y.astype(np.float32))
    assert np.array_equal(st.get_global(), y)
    for c, i, bad in ((0, 0, 2), (C - 1, n - 1, 255), (C // 2, n // 2, 128)):
        z = x.copy()
        z[c, i] = bad
        b = 0 if i < len(prog.free_blocks[0]) else 1
        with pytest.raises(th.ThrmlError, match=f"block {b} holds a value other than 0 and 1"):
            st.set_global(z)
        with pytest.raises(th.ThrmlError, match=f"block {b} "):
            st.set_global(np.where(z > 1, 0.5, z).astype(np.float32))
        assert np.array_equal(st.get_global(), y)
    s = th.sample_states(th.RngKey(1), prog, th.SamplingSchedule(1, 3, 1), st)
    assert np.array_equal(s[-1], st.get_global())
    st.close()
    prog.close()


@pytest.mark.parametrize("C", [1, 63, 65, 4100])
def test_narrow_spin_blocks(device, C):
    """Blocks around the widths that the export by rows of chains takes."""
    sizes = [1, 2, 8, 9, 16, 17]
    n = sum(sizes)
    cuts = np.cumsum(sizes)[:-1]
    log_case(f"narrow spin blocks C={C}")
    prog = th.IsingSamplingProgram(th.IsingEBM(n, np.zeros((0, 2)), np.zeros(n), []), np.split(np.arange(n), cuts), [],
                                   device)
    x = np.random.default_rng(C).integers(0, 2, (C, n)).astype(np.uint8)
    st = prog.new_state(C)
    st.set_global(x)
    for b, want in enumerate(np.split(x, cuts, axis=1)):
        assert np.array_equal(st.get_block(b), want)
        assert np.array_equal(st.get_block(b, np.float32), want.astype(np.float32))
    st.close()


@pytest.mark.parametrize("q,n,C", [(2, 7, 1), (3, 64, 64), (129, 65, 66), (256, 130, 3), (300, 67, 65)])
def test_categorical_state_round_trip(device, q, n, C):
    log_case(f"categorical state io q={q} n={n} C={C}")
    rng = np.random.default_rng(q)
    blocks = [np.arange(0, n // 2), np.arange(n // 2, n)]
    prog = th.CategoricalProgram(n, q, np.zeros((0, 2)), np.zeros((0, q, q)), rng.normal(0, 1, (n, q)), blocks,
                                 device)
    dt = np.uint16 if q > 256 else np.uint8
    x = rng.integers(0, q, (C, n)).astype(dt)
    st = prog.new_state(C)
    st.set_global(x)
    assert np.array_equal(st.get_global(), x)
    assert np.array_equal(np.concatenate([st.get_block(b) for b in range(2)], axis=1), x)
    if q < 256:
        z = x.copy()
        z[C - 1, n - 1] = q
        with pytest.raises(th.ThrmlError, match=f"block 1 holds a value outside 0..{q - 1}"):
            st.set_global(z)
        assert np.array_equal(st.get_global(), x)
    s = th.sample_states(th.RngKey(1), prog, th.SamplingSchedule(0, 4, 1), st)
    assert np.array_equal(s[0], x) and np.array_equal(s[-1], st.get_global())


def test_mixed_state_checks_each_block(device):
    """A mixed program's spin and categorical blocks take different values."""
    log_case("mixed state io")
    n, q, C = 70, 5, 9
    fs = [th.SpinEBMFactor([np.arange(n)], np.zeros((n, 1, 1))),
          th.CategoricalEBMFactor([np.arange(n, 2 * n)], np.zeros((n, q, 1)))]
    kinds = np.r_[np.zeros(n), np.ones(n)].astype(np.uint8)
    prog = th.FactorSamplingProgram(kinds, q, fs, [np.arange(n, 2 * n), np.arange(n)], [], device)
    rng = np.random.default_rng(2)
    x = np.concatenate([rng.integers(0, q, (C, n)), rng.integers(0, 2, (C, n))], axis=1).astype(np.uint8)
    st = prog.new_state(C)
    st.set_global(x)
    assert np.array_equal(st.get_global(), x)
    z = x.copy()
    z[3, n + 1] = 2  # a category, but not a spin
    with pytest.raises(th.ThrmlError, match="block 1 holds a value other than 0 and 1"):
        st.set_global(z)
    assert np.array_equal(st.get_global(), x)


def test_observations_in_several_transfers(device):
    """More observations than one transfer holds (64 MiB: 29 of 33 here), every one
    of them against the oracle."""
    log_case("observations in several transfers")
    n, C = 2048, 1100  # 2.25 MB per observation
    prog = _ising(n, device)
    st = th.hinton_init(th.RngKey(3), prog, C)
    init = st.get_global()
    out = th.sample_states(th.RngKey(4), prog, th.SamplingSchedule(0, 33, 1), st)
    assert out.shape == (33, C, n) and 29 * C * n < 64 << 20 < 30 * C * n
    e = np.stack([np.arange(n - 1), np.arange(1, n)], axis=1)
    o = orc.Ising(n, e, np.zeros(n), np.zeros(n - 1), 1.0, [np.arange(0, n, 2), np.arange(1, n, 2)])
    want = o.sample_states(4, (0, 33, 1), init)
    for i in range(33):
        assert np.array_equal(out[i], want[i]), f"observation {i} differs"
    assert np.array_equal(st.get_global(), want[-1])


def test_memory_is_kept_within_one_stream(device):
    """A context moved to another stream, objects made and let go of on both."""
    import torch

    log_case("memory kept across a stream change")
    dev = th.Device(0)
    rng = np.random.default_rng(0)
    x = rng.integers(0, 2, (50, 400)).astype(np.uint8)
    want = None
    for rep in range(6):
        if rep == 2:
            side = torch.cuda.Stream()
            dev.set_stream(side.cuda_stream)
        if rep == 4:
            dev.set_stream(torch.cuda.current_stream().cuda_stream)
        prog = _ising(400, dev)
        st = prog.new_state(50)
        st.set_global(x)
        th.run_blocks(th.RngKey(5), prog, st, (), 20)
        got = st.get_global()
        want = got if want is None else want
        assert np.array_equal(got, want)
        st.close()
        prog.close()
    dev.close()
