"""Engine.set_order and Replica.states() on one replica: each keeps the order it
was given, whoever came first and whatever was refused in between."""
import numpy as np
import pytest

from sagesim_amd import Engine, Replica, graphs, sir_model
from sagesim_amd._lib import NativeError

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ghosts", [0, 3])
@pytest.mark.parametrize("first", ["states", "set_order"])
def test_states_beside_another_order(first, ghosts):
    print("[case] order owner", first, ghosts, flush=True)
    n = 700
    rng = np.random.default_rng(n)
    rp = np.concatenate([[0], np.cumsum(rng.integers(0, 7, n))])
    g = graphs.CSRGraph(rp, rng.integers(0, n + ghosts, rp[-1]).astype(np.int32), n_cols=n + ghosts)
    st = rng.integers(0, 3, n + ghosts).astype(np.int8)
    with Engine(0) as eng:
        rep = Replica(eng, g, st, sir_model(0.3, 0.2), 1)
        assert not np.array_equal(rep.inv, np.arange(n))
        other = rng.permutation(n).astype(np.int32)
        raw = eng.state(rep.rep, n + ghosts)
        want = np.concatenate([raw[:n][other], raw[n:]])
        if first == "states":
            assert np.array_equal(rep.states(), st)
        eng.set_order(rep.rep, other)
        for _ in range(2):
            assert np.array_equal(rep.states(), st)
            assert np.array_equal(eng.state_ordered(rep.rep, n + ghosts), want)
        with pytest.raises(NativeError):
            eng.set_order(rep.rep, np.full(n, n, np.int32))
        assert np.array_equal(rep.states(), st)
        second = Replica(eng, g, st, sir_model(0.3, 0.2), 1)
        rep.remove()
        assert np.array_equal(second.states(), st)
        third = Replica(eng, g, st, sir_model(0.3, 0.2), 1)      # in the first one's place
        assert third.rep == rep.rep
        assert np.array_equal(third.states(), st)
