"""The start of a tick (reset, new states, another tick number): states, bitmaps,
statistics and pushed counts made in two launches.  A replica that was run and
started again gives what a fresh one gives, whether ticks push or only pull, with
an infectious hub whose degree does not fit a byte.  Whole numbers: equal exactly.
"""
import numpy as np
import pytest

from sagesim_amd import Engine, graphs, sir_model
from sagesim_amd.engine import Replica

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tick0", [0, 1, 5])
@pytest.mark.parametrize("n", [1, 17, 64, 1000, 4097, 70_001])
def test_started_again_equals_fresh(n, tick0):
    rng = np.random.default_rng(n + tick0)
    u = np.concatenate([np.zeros(min(n - 1, 700), np.int64), rng.integers(0, n, 3 * n)])
    v = np.concatenate([np.arange(1, min(n - 1, 700) + 1), rng.integers(0, n, 3 * n)])
    g = graphs.from_edges(n, u, v)
    a = (rng.random(n) < 0.01).astype(np.int8)
    b = (rng.random(n) < 0.2).astype(np.int8)
    a[0] = b[0] = 1                                     # the hub
    say = print

    def run(eng, rep):
        eng.simulate(9)
        return rep.states()

    out = []
    for ratio in (0.25, 1e6, 0.0):
        say("begin", n, tick0, ratio, flush=True)
        with Engine() as eng:
            eng.set_push(ratio)
            one = Replica(eng, g, a, sir_model(0.2, 0.1), 3, tick0=tick0)
            first = run(eng, one)
            one.reset()
            assert np.array_equal(one.states(), a)
            again = run(eng, one)
            one.set_states(b)
            assert np.array_equal(one.states(), b)
            after = run(eng, one)
            eng.set_tick(one.rep, tick0 + 4)            # same states, another tick and maybe parity
            moved_from = one.states()
            moved = run(eng, one)
            assert np.array_equal(moved_from, after)
            assert np.array_equal(first, again)
        with Engine() as eng:
            eng.set_push(ratio)
            fresh = Replica(eng, g, b, sir_model(0.2, 0.1), 3, tick0=tick0 + 9)
            assert np.array_equal(run(eng, fresh), after)
        with Engine() as eng:
            eng.set_push(ratio)
            fresh = Replica(eng, g, after, sir_model(0.2, 0.1), 3, tick0=tick0 + 4)
            assert np.array_equal(run(eng, fresh), moved)
        out.append(np.stack([first, after, moved]))
    assert np.array_equal(out[0], out[2])
    assert np.array_equal(out[1], out[2])
