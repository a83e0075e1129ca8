"""States read back in the caller's agent order (put in order on the device)
against the storage-order download and the permutation: sizes around the
16-agent groups of the kernel, ghost slots after the agents, a new order set
over an old one, and the host's refusals."""
import numpy as np
import pytest

from sagesim_amd import Engine, Replica, graphs, sir_model
from sagesim_amd._lib import NativeError

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ghosts", [0, 1, 37])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 4095, 4097, 50_001])
def test_ordered_states(n, ghosts):
    print("[case] order", n, ghosts, flush=True)
    rng = np.random.default_rng(n)
    degs = rng.integers(0, min(6, n + ghosts) + 1, n)
    rp = np.concatenate([[0], np.cumsum(degs)])
    g = graphs.CSRGraph(rp, rng.integers(0, n + ghosts, rp[-1]).astype(np.int32), n_cols=n + ghosts)
    st = rng.integers(0, 3, n + ghosts).astype(np.int8)
    with Engine(0) as eng:
        rep = Replica(eng, g, st, sir_model(0.3, 0.2), n)
        assert np.array_equal(rep.states(), st)
        for ticks in (1, 2):                        # either state buffer
            eng.simulate(ticks)
            raw = eng.state(rep.rep, n + ghosts)
            want = np.concatenate([raw[:n][rep.inv], raw[n:]])
            assert np.array_equal(rep.states(), want)
        other = rng.permutation(n).astype(np.int32)
        eng.set_order(rep.rep, other)
        raw = eng.state(rep.rep, n + ghosts)
        assert np.array_equal(eng.state_ordered(rep.rep, n + ghosts), np.concatenate([raw[:n][other], raw[n:]]))


def test_order_refusals():
    print("[case] order refusals", flush=True)
    g = graphs.from_edges(100, np.arange(99), np.arange(1, 100))
    with Engine(0) as eng:
        rep = Replica(eng, g, np.zeros(100, np.int8), sir_model(0.3, 0.2), 1)
        with pytest.raises(NativeError):
            eng.state_ordered(rep.rep, 100)         # no order yet
        with pytest.raises(NativeError):
            eng.set_order(rep.rep, np.arange(99))   # not every agent
        for bad in (-1, 100):
            slots = np.arange(100)
            slots[50] = bad
            with pytest.raises(NativeError):
                eng.set_order(rep.rep, slots)
            with pytest.raises(NativeError):
                eng.state_ordered(rep.rep, 100)
        assert np.array_equal(rep.states(), np.zeros(100, np.int8))
