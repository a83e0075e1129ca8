"""Wide light tiles (16 agents per lane) against the narrow ones, which take
another path through loads, queues and masks: the same states after every few
ticks, pulled, pushed and with neighbour counts, at sizes on either side of a
lane's, a chunk's and a tile's agents, and with state bytes that are no codes
(such agents stay as they are).  Whole numbers: equal exactly.
"""
import numpy as np
import pytest

from sagesim_amd import Engine, graphs, seir_model, sir_model
from sagesim_amd.engine import Replica

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("odd_codes", [False, True])
@pytest.mark.parametrize("kind", ["sir", "seir", "sirs"])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 65, 1023, 1025, 4096, 16_411, 300_007])
def test_wide_and_narrow_tiles_agree(n, kind, odd_codes):
    rng = np.random.default_rng(n)
    g = graphs.watts_strogatz(n, 6, 0.3, 5) if n > 20 else graphs.from_edges(n, np.arange(n - 1), np.arange(1, n))
    state = (rng.random(n) < 0.02).astype(np.int8)
    state[0] = 1
    if odd_codes:
        state[rng.integers(0, n, 1 + n // 50)] = rng.choice(np.array([-1, 4, 7, 100, -128], np.int8), 1 + n // 50)
    model = seir_model(0.2, 0.3, 0.1) if kind == "seir" else sir_model(0.15, 0.08)
    if kind == "sirs":                                  # immunity wanes: every count is pushed
        model.trans_p[2], model.trans_next[2] = 0.05, 0
    out = []
    for apl in (16, 4):
        with Engine() as eng:
            print("wide", n, kind, odd_codes, apl, flush=True)
            eng.set_tiling(agents_per_lane=apl)
            rep = Replica(eng, g, state, model, 77)
            got = []
            for ticks in (1, 2, 7, 20, 60):
                eng.simulate(ticks)
                got.append(rep.states())
            out.append(np.stack(got))
    assert np.array_equal(out[0], out[1])
