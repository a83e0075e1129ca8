"""Models built and counters read while another engine's work is queued on the
device: results do not depend on when that work ends."""
import numpy as np
import pytest

from oracle import oracle as O
from sagesim_amd import Breed, Engine, Model, NetworkSpace, Replica, graphs, sir_model
from sagesim_amd.steps import reference_sir_step

pytestmark = pytest.mark.gpu


@pytest.fixture
def busy():
    """An engine with a large network, and a call that queues ticks of it."""
    g = graphs.barabasi_albert(200_000, 5, 3)
    st = (np.random.default_rng(3).random(g.n) < 0.01).astype(np.int8)
    with Engine(0) as eng:
        rep = Replica(eng, g, st, sir_model(0.02, 0.001), 3)

        def queue():
            rep.reset()
            eng.simulate(300)
        yield queue
        eng.sync()


@pytest.mark.parametrize("n", [300, 20_000])
def test_model_set_up_beside_queued_ticks(n, busy):
    print("[case] model beside queued ticks", n, flush=True)
    g = graphs.watts_strogatz(n, 8, 0.1, 7)
    init = np.where(np.random.default_rng(n).random(n) < 0.1, 2, 1).astype(np.float32)
    want = O.ref_sir_run(g.row_ptr, g.col_idx, np.arange(n, dtype=np.float32), init, 9, 10, 0.2, 0.1)
    for _ in range(3):
        b = Breed("SIR")
        b.register_property("state", 1)
        b.register_step_func(reference_sir_step())
        m = Model(NetworkSpace())
        m.register_breed(b)
        m.register_global_property("p_infection", 0.2)
        m.register_global_property("p_recovery", 0.1)
        m.set_seed(9)
        for s in init:
            m.create_agent_of_breed(b, state=float(s))
        m.get_space().connect_agents_bulk(np.repeat(np.arange(n), np.diff(g.row_ptr)), g.col_idx, directed=True)
        busy()
        m.setup()
        busy()
        m.simulate(10)
        assert np.array_equal(m.get_breed_data("SIR", "state"), want)
        m.reset()


def test_counters_cleared_beside_queued_ticks(busy):
    print("[case] counters beside queued ticks", flush=True)
    g = graphs.barabasi_albert(3000, 5, 1)
    st = (np.random.default_rng(1).random(g.n) < 0.02).astype(np.int8)
    want = None
    for _ in range(5):
        busy()
        with Engine(0) as eng:
            eng.set_counting(True)
            rep = Replica(eng, g, st, sir_model(0.05, 0.1), 1)
            for _ in range(3):
                rep.reset()
                eng.simulate(20)
                got = eng.read_counters()
                busy()
                want = got if want is None else want
                assert np.array_equal(got, want)
