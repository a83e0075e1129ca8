"""Row scans and pushes of the tick kernel at the lengths where they can go
wrong, tick by tick against the oracle: chunks whose rows all have one length
(the scan then computes a row's start), lengths around the eight entries of a
scan round, around the 32 and 256 entries where a row is pushed by more lanes,
and at 255, where the one-byte degree copy ends; graphs whose last row ends at
the last entry, with and without the last-infector history, all pull, all push
and the default rule; and one length broken by a single longer row."""
import numpy as np
import pytest

from oracle import oracle as O
from sagesim_amd import Engine, Replica, graphs, sir_model

pytestmark = pytest.mark.gpu


def _circulant(n, d):
    """Every agent linked to the d / 2 on either side (and, for odd d and even n, to the one opposite)."""
    u = np.arange(n)
    offs = list(range(1, d // 2 + 1)) + ([n // 2] if d % 2 else [])
    return graphs.from_edges(n, np.tile(u, len(offs)), np.concatenate([(u + o) % n for o in offs]))


def _check(g, beta, ticks, history, rule, heavy=512, sort=True):
    rng = np.random.default_rng(g.n)
    st = (rng.random(g.n) < 0.15).astype(np.int8)
    hist = np.full((g.n, 32), -1, np.int32) if history else None
    hist_want = None if hist is None else hist.copy()
    _, trace = O.sir_run(O.sir_model(beta, 0.2, 9), g.row_ptr, g.col_idx, np.arange(g.n), st, ticks,
                         history=hist_want, trace=True)
    with Engine(0) as e:
        e.set_push(rule)
        e.set_tiling(heavy, 16, 0, True)
        r = Replica(e, g, st, sir_model(beta, 0.2), 9, history=hist, sort=sort)
        for t in range(ticks):
            e.simulate(1)
            got = r.states()
            bad = np.nonzero(got != trace[t])[0]
            assert bad.size == 0, (t, bad[:5])
        if history:
            assert np.array_equal(r.history(), hist_want)


@pytest.mark.parametrize("rule", [0.0, 0.25, 1.0e6])
@pytest.mark.parametrize("d", [1, 3, 4, 5, 8, 9, 16, 17, 32, 33, 254, 255, 256, 258])
def test_rows_of_one_length(d, rule):
    n = 1300 if d > 100 else 5002                  # not whole chunks; even for the opposite neighbour
    print("[case] rows of", d, "rule", rule, flush=True)
    _check(_circulant(n, d), min(0.9, 1.0 / d), 12, d in (5, 9, 255), rule)


def test_one_longer_row():
    print("[case] one longer row", flush=True)
    n = 4096
    u = np.arange(n)
    g = graphs.from_edges(n, np.concatenate([u, [17, 17, 17]]), np.concatenate([(u + 1) % n, [900, 2000, 4000]]))
    for sort in (True, False):
        _check(g, 0.5, 12, False, 0.0, sort=sort)


@pytest.mark.parametrize("beta", [0.02, 0.2])
@pytest.mark.parametrize("d", [10, 12, 15, 24, 63, 64, 65, 71, 72, 73, 80])
def test_scans_that_give_up(d, beta):
    """Rows whose scan ends when what is left cannot infect: lengths around
    whole rounds of eight and around the 64 thresholds held in LDS, few and many
    hits needed, every tick pulled."""
    print("[case] scans that give up", d, beta, flush=True)
    for history in (False, True):
        _check(_circulant(3002, d), beta, 8, history, 0.0)
