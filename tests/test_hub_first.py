"""Compiled step functions on networks whose hubs were created first, longest
first: the agents' order is then the order they have, and the hubs' rows are
staged all the same.  On the host, what setup tells the library; on the GPU, the
oracle's restatement of the reference's SIR step."""
import types

import numpy as np
import pytest

from oracle import oracle as O
from sagesim_amd import Breed, Model, NetworkSpace, graphs
from sagesim_amd import model as model_mod
from sagesim_amd.steps import reference_sir_step


def _hub_first(hubs, n):
    """Agents 0, 1, ... with that many neighbours each over a ring of the rest."""
    ring = np.arange(len(hubs), n)
    u, v = [ring], [np.roll(ring, -1)]
    for h, d in enumerate(hubs):
        u.append(np.full(d, h))
        v.append(ring[np.arange(d)])
    return graphs.from_edges(n, np.concatenate(u), np.concatenate(v))


def _model(g, init):
    b = Breed("SIR")
    b.register_property("state", 1)
    b.register_step_func(reference_sir_step())
    m = Model(NetworkSpace(), use_fused=False)
    m.register_breed(b)
    m.register_global_property("p_infection", 0.05)
    m.register_global_property("p_recovery", 0.1)
    m.set_seed(9)
    for s in init:
        m.create_agent_of_breed(b, state=float(s))
    m.get_space().connect_agents_bulk(np.repeat(np.arange(g.n), np.diff(g.row_ptr)), g.col_idx, directed=True)
    return m


CASES = [([299], 300), ([256], 3000), ([2999], 3000), ([900, 500], 3000), ([10_240, 700, 256], 12_000)]


@pytest.mark.parametrize("hubs,n", CASES)
def test_order_is_set_before_long_rows(hubs, n, monkeypatch):
    g = _hub_first(hubs, n)
    order, staged = model_mod._agent_order(np.diff(g.row_ptr))
    assert staged == len(hubs) and np.array_equal(order, np.arange(n))
    calls = []

    class Lib:
        def __getattr__(self, name):
            return lambda *a: calls.append(name) or 0

    monkeypatch.setattr(model_mod, "step_lib", lambda: Lib())
    m = _model(g, np.ones(n))
    m._engine = types.SimpleNamespace(_h=None)
    m.setup()
    assert "ss_prog_set_order" in calls
    assert calls.index("ss_prog_set_schedule") < calls.index("ss_prog_set_order") < calls.index("ss_prog_set_long")


@pytest.mark.gpu
@pytest.mark.parametrize("hubs,n", CASES)
def test_hub_first_model(hubs, n):
    print("[case] hub first", hubs, n, flush=True)
    g = _hub_first(hubs, n)
    init = np.where(np.random.default_rng(n).random(n) < 0.05, 2, 1).astype(np.float32)
    init[:len(hubs)] = 1
    m = _model(g, init)
    m.setup()
    m.simulate(12)
    want = O.ref_sir_run(g.row_ptr, g.col_idx, np.arange(n, dtype=np.float32), init, 9, 12, 0.05, 0.1)
    assert np.array_equal(m.get_breed_data("SIR", "state"), want)
