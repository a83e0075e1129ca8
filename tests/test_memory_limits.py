"""What a device without memory to spare still does: states() without the order
table it keeps on the device, a footprint that counts the table, and calls after
one that ran out of memory."""
import numpy as np
import pytest

from sagesim_amd import Engine, Replica, graphs, sir_model
from sagesim_amd._lib import SS_ERR_OOM, NativeError, step_lib
from sagesim_amd.serving import footprint


class _Full:
    """An engine whose device has no memory for an order."""

    def __init__(self, code):
        self.code = code

    def add_replica(self, rp, ci, ids, state, *a, **kw):
        self.kept = np.array(state)
        return 0

    def order_of(self, rep):
        return None

    def set_order(self, rep, slots):
        raise NativeError(self.code, "hipMalloc: out of memory")

    def state(self, rep, n_total):
        assert n_total == self.kept.size
        return self.kept.copy()


@pytest.mark.parametrize("ghosts", [0, 5])
def test_states_without_memory_for_the_order(ghosts):
    rng = np.random.default_rng(1)
    n = 400
    degs = rng.integers(0, 9, n)
    rp = np.concatenate([[0], np.cumsum(degs)])
    g = graphs.CSRGraph(rp, rng.integers(0, n + ghosts, rp[-1]).astype(np.int32), n_cols=n + ghosts)
    st = rng.integers(0, 3, n + ghosts).astype(np.int8)
    rep = Replica(_Full(SS_ERR_OOM), g, st, sir_model(0.3, 0.2), 1)
    assert not np.array_equal(rep.engine.kept, st)
    for _ in range(2):
        assert np.array_equal(rep.states(), st)
    with pytest.raises(NativeError):
        Replica(_Full(-2), g, st, sir_model(0.3, 0.2), 1).states()


def test_footprint_counts_the_order():
    """An agent more costs its row bound (8), key and degree byte (5), three states
    and its order (4) at least, groups of 64 agents at a time."""
    L = step_lib()
    a, b = (L.ss_replica_footprint(n, 0, 10_000, 0, 50) for n in (64_000, 128_000))
    assert b - a >= 64_000 * (8 + 5 + 3 + 4 + 4)           # and the push counts (4)


@pytest.mark.gpu
@pytest.mark.parametrize("n,ghosts", [(1, 0), (1000, 0), (4097, 33), (50_000, 0)])
def test_replica_bytes_within_footprint(n, ghosts):
    print("[case] footprint", n, ghosts, flush=True)
    rng = np.random.default_rng(n)
    degs = rng.integers(0, min(9, n + ghosts), n)
    rp = np.concatenate([[0], np.cumsum(degs)])
    g = graphs.CSRGraph(rp, rng.integers(0, n + ghosts, rp[-1]).astype(np.int32), n_cols=n + ghosts)
    with Engine(0) as eng:
        rep = Replica(eng, g, np.zeros(n + ghosts, np.int8), sir_model(0.3, 0.2), 1)
        eng.simulate(2)
        rep.states()
        assert eng.replica_bytes(rep.rep) <= footprint(g)


@pytest.mark.gpu
def test_calls_after_running_out_of_memory():
    print("[case] out of memory", flush=True)
    g = graphs.barabasi_albert(2000, 3, 1)
    st = (np.arange(g.n) % 50 == 0).astype(np.int8)
    with Engine(0) as eng:
        rep = Replica(eng, g, st, sir_model(0.3, 0.2), 1)
        eng.simulate(5)
        want = rep.states()
        rep.reset()
        for _ in range(2):
            with pytest.raises(NativeError) as ex:
                eng.copy_probe(1 << 50)                     # a petabyte
            assert ex.value.code == SS_ERR_OOM
            assert np.array_equal(rep.states(), st)
        eng.simulate(5)
        assert np.array_equal(rep.states(), want)


@pytest.mark.gpu
def test_kept_workspace_makes_room():
    """The workspace that a map build leaves with the context goes before an
    allocation fails, and comes back with the next build."""
    print("[case] kept workspace", flush=True)
    n = 200_000
    g = graphs.CSRGraph(np.zeros(n + 1, np.int64), np.zeros(0, np.int32))
    ids = np.arange(n, dtype=np.int64) * 7
    with Engine(0) as eng:
        rep = Replica(eng, g, np.zeros(n, np.int8), sir_model(0.3, 0.2), 1)
        eng.simulate(1)
        rep.states()
        for _ in range(2):
            eng.map_build(rep.rep, ids, np.arange(n))
            full = eng.info()["ctx_bytes"]
            with pytest.raises(NativeError):
                eng.copy_probe(1 << 50)
            assert eng.info()["ctx_bytes"] <= full - 20 * n            # ids, slots and claims
            slots, missing = eng.map_lookup(rep.rep, ids)
            assert missing == 0 and np.array_equal(slots, np.arange(n))
            assert np.array_equal(rep.states(), np.zeros(n, np.int8))
