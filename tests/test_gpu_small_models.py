"""Small models, whose whole ticks run on one block, against the same models on
a launch per priority group (and the reference's SIR step against the oracle):
one agent, sizes around a wavefront and around the limits, two breeds at three
priorities with scalar, 2-D and in-place properties and breed-local arrays, one
tick a call and many, and a network past the limit on its entries."""
import numpy as np
import pytest

from oracle import oracle as O
from sagesim_amd import Breed, Model, NetworkSpace, StepFunction, graphs
from sagesim_amd import model as model_mod
from sagesim_amd.steps import reference_sir_step

pytestmark = pytest.mark.gpu

_STEPS = r"""
__device__ void walk(auto tick, auto agent_index, auto p, auto agent_ids, auto breeds, auto locations, auto state,
                     auto energy, auto row, auto seen, auto mem, auto mem_idx) {
    auto nb = locations[agent_index];
    float sum = 0.0f;
    for (int j = 0; j < len(nb); ++j) sum += energy[nb[j]] * row[nb[j]][tick % 3];
    energy[agent_index] = 0.5f * energy[agent_index] + 0.125f * sum;
    if (rand_uniform_philox(tick, agent_index, 2) < p) state[agent_index] = (int)state[agent_index] == 1 ? 0 : 1;
    mem[mem_idx[agent_index]][1] = mem[mem_idx[agent_index]][1] + 1.0f;
    row[agent_index][(tick + 1) % 3] = sum;
}
__device__ void tally(auto tick, auto agent_index, auto p, auto agent_ids, auto breeds, auto locations, auto state,
                      auto energy, auto row, auto seen, auto mem, auto mem_idx) {
    auto nb = locations[agent_index];
    int k = 0;
    for (int j = 0; j < len(nb); ++j) k += (int)state[nb[j]] == 1;
    seen[agent_index] = seen[agent_index] + (float)k;
}
__device__ void look(auto tick, auto agent_index, auto p, auto agent_ids, auto breeds, auto locations, auto state,
                     auto energy, auto row, auto seen, auto mem, auto mem_idx) {
    auto nb = locations[agent_index];
    for (int j = 0; j < len(nb); ++j)
        if ((float)seen[nb[j]] > 2.0f) mem[mem_idx[agent_index]][0] = (float)seen[nb[j]];
}
"""


def _breeds(n, calls, loop, monkeypatch):
    monkeypatch.setattr(model_mod, "_LOOP_AGENTS", 1 << 20 if loop else 0)
    rng = np.random.default_rng(n)
    walker, sensor = Breed("Walker"), Breed("Sensor")
    for b in (walker, sensor):
        b.register_property("state", 0)
        b.register_property("energy", 1.0)
        b.register_property("row", [1.0, 0.5, 0.25], max_dims=[3])
        b.register_property("seen", 0.0)
    walker.register_step_func(StepFunction("walk", _STEPS), priority=0)
    sensor.register_step_func(StepFunction("tally", _STEPS), priority=1, no_double_buffer=["seen"])
    walker.register_step_func(StepFunction("look", _STEPS), priority=2)
    m = Model(NetworkSpace())
    m.register_breed(walker)
    m.register_breed(sensor)
    m.register_breed_local_array("mem", walker, (2,))
    m.register_global_property("p", 0.3)
    m.set_seed(5)
    for i in range(n):
        m.create_agent_of_breed(sensor if i % 3 == 2 else walker, energy=float(np.float32(rng.random())), seen=0.0)
    g = graphs.erdos_renyi(n, min(1.0, 6.0 / n), 3) if n > 1 else graphs.CSRGraph(np.zeros(2, np.int64), np.zeros(0, np.int32))
    m.get_space().connect_agents_bulk(np.repeat(np.arange(g.n), np.diff(g.row_ptr)), g.col_idx, directed=True)
    m.setup()
    for c in calls:
        m.simulate(c)
    out = [m.get_breed_data(b, p) for b in ("Walker", "Sensor") for p in ("state", "energy", "row", "seen")]
    return out + [m.get_breed_local_array("mem")]


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 600, 1025, 2047, 2048])
def test_one_block_equals_launches(n, monkeypatch):
    print("[case] small model", n, flush=True)
    for calls in ([1, 1, 3], [12]):
        for a, b in zip(_breeds(n, calls, True, monkeypatch), _breeds(n, calls, False, monkeypatch)):
            assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("n,k", [(64, 6), (1000, 20), (1200, 20), (2048, 10), (2049, 10), (2048, 12)])
def test_sir_around_the_limits(n, k):
    print("[case] sir", n, k, flush=True)
    g = graphs.watts_strogatz(n, k, 0.1, 7)
    rng = np.random.default_rng(n)
    init = np.where(rng.random(n) < 0.1, 2, 1).astype(np.float32)
    b = Breed("SIR")
    b.register_property("state", 1)
    b.register_step_func(reference_sir_step())
    m = Model(NetworkSpace())
    m.register_breed(b)
    m.register_global_property("p_infection", 0.05)
    m.register_global_property("p_recovery", 0.1)
    m.set_seed(9)
    for s in init:
        m.create_agent_of_breed(b, state=float(s))
    m.get_space().connect_agents_bulk(np.repeat(np.arange(n), np.diff(g.row_ptr)), g.col_idx, directed=True)
    m.setup()
    for t0, t in ((0, 1), (1, 9), (10, 15)):
        m.simulate(t)
        want = O.ref_sir_run(g.row_ptr, g.col_idx, np.arange(n, dtype=np.float32), init, 9, t0 + t, 0.05, 0.1)
        assert np.array_equal(m.get_breed_data("SIR", "state"), want)
