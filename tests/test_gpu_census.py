"""Census of a replica (agents per state, sum of the susceptible degrees)
against numpy over the downloaded states: sizes around the kernel's 16-agent
groups and its blocks of 4096, rows of 254 to 1000 entries (the one-byte
degree copy holds 255 for the long ones), ghost slots that do not count, and a
census queued right after every call of a run on several engines."""
import numpy as np
import pytest

from sagesim_amd import Engine, Replica, graphs, seir_model, sir_model

pytestmark = pytest.mark.gpu


def _check(eng, rep, s_code=0):
    st = eng.state(rep.rep, rep.n_total)[:rep.n]
    got = eng.census(rep.rep)
    assert got[:4].tolist() == np.bincount(st, minlength=4)[:4].tolist()
    assert got[4] == np.diff(rep.graph.row_ptr)[st == s_code].sum()


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 4095, 4096, 4097, 70_001])
def test_census_sizes(n):
    print("[case] census n", n, flush=True)
    rng = np.random.default_rng(n)
    g = graphs.from_edges(n, rng.integers(0, n, 3 * n), rng.integers(0, n, 3 * n))
    with Engine(0) as eng:
        rep = Replica(eng, g, rng.integers(0, 4, n).astype(np.int8), seir_model(0.1, 0.2, 0.1), n)
        _check(eng, rep)
        eng.simulate(3)
        _check(eng, rep)


def test_census_long_rows_and_ghosts():
    print("[case] census long rows, ghosts", flush=True)
    rng = np.random.default_rng(5)
    degs = np.array([1000, 256, 255, 254, 300] + [7] * 60 + [0] * 10, np.int64)
    rp = np.concatenate([[0], np.cumsum(degs)])
    n, ghosts = degs.size, 1100
    ci = np.concatenate([rng.permutation(n + ghosts)[:d] for d in degs]).astype(np.int32)
    g = graphs.CSRGraph(rp, ci, n_cols=n + ghosts)
    with Engine(0) as eng:
        rep = Replica(eng, g, rng.integers(0, 3, n + ghosts).astype(np.int8), sir_model(0.1, 0.1), 3, sort=False)
        _check(eng, rep)


def test_census_after_every_call_on_several_engines():
    print("[case] census in a run", flush=True)
    n = 20_000
    g = graphs.watts_strogatz(n, 10, 0.1, 4)
    st = np.zeros(n, np.int8)
    st[::50] = 2
    runs = []
    for seed in range(4):
        eng = Engine(0)
        runs.append((eng, Replica(eng, g, st, seir_model(0.05, 0.2, 0.1), seed)))
    for _ in range(10):
        for eng, rep in runs:
            eng.simulate(5)
            _check(eng, rep)
    for eng, _ in runs:
        eng.close()
