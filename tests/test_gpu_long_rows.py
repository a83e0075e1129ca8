"""Compiled step functions on networks with long rows, whose agents get a block
each with the row in LDS: rows around the staging limits (256 and 10,240
entries), a breed range that does not start at 0, and steps that use the row in
every form a plain row allows (by `auto`, through the runtime's type names, by
get_neighbor, through another agent's row, by assigning rows to each other,
which cannot be staged) against the oracle's restatement of the reference's SIR
step."""
import numpy as np
import pytest

from oracle import oracle as O
from sagesim_amd import Breed, Model, NetworkSpace, StepFunction, graphs
from sagesim_amd import model as model_mod

pytestmark = pytest.mark.gpu

_HEAD = """
__device__ void step(auto tick, {index}, auto p_infection, auto p_recovery, auto agent_ids, auto breeds,
                     {locations}, auto state) {{
    const int mine = (int)state[agent_index];
    const double rand = rand_uniform_philox(tick, agent_index, 1);
    {row}
    if (mine == 2 && rand < p_recovery) state[agent_index] = 3;
    else if (mine == 1)
        for (int i = 0; i < {n}; ++i)
            if ((int)state[{at}] == 2 && rand < p_infection) state[agent_index] = 2;
}}
"""
_AUTO = dict(index="auto agent_index", locations="auto locations", row="auto nb = locations[agent_index];",
             n="len(nb)", at="nb[i]")
FORMS = {
    "auto": _AUTO,
    "typed": dict(_AUTO, index="AgentIndex agent_index", locations="const Locations &locations",
                  row="NeighborRow nb = locations[agent_index];"),
    "typed row": dict(_AUTO, row="const NeighborRow nb = locations[agent_index];"),
    "helpers": dict(_AUTO, row="", n="get_num_neighbors(agent_index, locations)",
                    at="get_neighbor(agent_index, i, locations)"),
    "offsets": dict(_AUTO, row="", n="get_num_neighbors(agent_index, neighbor_offsets)",
                    at="get_neighbor(agent_index, i, neighbor_offsets, neighbor_values)"),
    "plain index": dict(_AUTO, row="const long long me = agent_index; auto nb = locations[me];"),
    "assigned": dict(_AUTO, row="auto nb = locations[agent_index]; if (len(nb) < 0) nb = locations[0ll];"),
    "chosen": dict(_AUTO, row="auto nb = len(locations[agent_index]) >= 0 ? locations[agent_index] : locations[0ll];"),
}


def _network():
    """Hubs of 255, 256, 257, 1000, 10240 and 10241 neighbours over a ring of 12,000."""
    n, degs = 12_000, [255, 256, 257, 1000, 10_240, 10_241]
    ring = np.arange(len(degs), n)
    u, v = [ring], [np.roll(ring, -1)]
    for h, d in enumerate(degs):
        u.append(np.full(d, h))
        v.append(ring[(np.arange(d) * 7 + h) % ring.size if d < 1500 else np.arange(d)])
    return graphs.from_edges(n, np.concatenate(u), np.concatenate(v)), degs


def _run(form, ticks, other_first=False):
    g, degs = _network()
    assert np.diff(g.row_ptr)[:len(degs)].tolist() == degs
    rng = np.random.default_rng(3)
    init = np.where(rng.random(g.n) < 0.1, 2, 1).astype(np.float32)
    init[:len(degs)] = 1
    b, other = Breed("SIR"), Breed("Other")
    for x in (other, b) if other_first else (b, other):
        x.register_property("state", 1)
    b.register_step_func(StepFunction("step", _HEAD.format(**FORMS[form])), priority=0)
    m = Model(NetworkSpace())
    for x in (other, b) if other_first else (b, other):
        m.register_breed(x)
    m.register_global_property("p_infection", 0.2)
    m.register_global_property("p_recovery", 0.1)
    m.set_seed(77)
    for s in init:
        m.create_agent_of_breed(b, state=float(s))
    n_other = 70 if other_first else 0
    for _ in range(n_other):
        m.create_agent_of_breed(other, state=3.0)
    m.get_space().connect_agents_bulk(np.repeat(np.arange(g.n), np.diff(g.row_ptr)), g.col_idx, directed=True)
    m.setup()
    m.simulate(ticks)
    got = m.get_breed_data("SIR", "state")
    want = O.ref_sir_run(g.row_ptr, g.col_idx, np.arange(g.n, dtype=np.float32), init, 77, ticks, 0.2, 0.1)
    assert np.array_equal(got, want), np.nonzero(got != want)[0][:5]
    assert (want[:len(degs)] != 1).any()


@pytest.mark.parametrize("form", list(FORMS))
def test_forms(form):
    print("[case] long rows:", form, flush=True)
    _run(form, 15)


def test_other_breed_first():
    print("[case] long rows after another breed", flush=True)
    _run("auto", 15, other_first=True)


def test_agent_order():
    """The order is a permutation whose front holds the staged rows, longest first."""
    rng = np.random.default_rng(1)
    for n in (1, 63, 64, 65, 1000, 50_000):
        for deg in (rng.integers(0, 10, n), (rng.pareto(1.0, n) * 4).astype(np.int64), np.full(n, 300)):
            order, staged = model_mod._agent_order(deg)
            assert np.array_equal(np.sort(order), np.arange(n))
            front = deg[order[:staged]]
            assert np.all(np.diff(front) <= 0)
            assert np.all((front >= model_mod._STAGED_ROW_MIN) & (front <= model_mod._STAGED_ROW_MAX))
            assert model_mod._agent_order(deg, stage=False)[1] == 0
