"""Copies of ordinary memory through page-locked chunks: states up, down and
down in another order, at sizes on either side of one chunk (1 MiB), of several,
and of where more threads take part (4 MiB); and from and to page-locked arrays.
"""
import numpy as np
import pytest

from sagesim_amd import Engine, sir_model

pytestmark = pytest.mark.gpu

MB = 1 << 20


@pytest.mark.parametrize("n", [1, 15, 17, MB - 1, MB, MB + 1, 2 * MB + 5, 4 * MB - 1, 4 * MB + 1, 9 * MB + 7])
def test_states_round_trip(n):
    print("staging", n, flush=True)
    rng = np.random.default_rng(n)
    first, second = rng.integers(0, 3, (2, n), dtype=np.int8)
    slot = rng.permutation(n).astype(np.int32)
    with Engine() as eng:
        rep = eng.add_replica(np.zeros(n + 1, np.int64), np.zeros(0, np.int32), np.arange(n), first,
                              sir_model(0.5, 0.0), 1)
        eng.set_order(rep, slot)
        for want in (first, second):
            if want is second:
                eng.set_state(rep, second)
            for _ in range(2):                                  # into fresh and into used memory
                assert np.array_equal(eng.state(rep, n), want)
                assert np.array_equal(eng.state_ordered(rep, n), want[slot])
        locked = eng.pinned_empty((n,), np.int8)
        locked[...] = first
        eng.set_state(rep, locked)
        locked[...] = 3                                         # the call is done with it
        assert np.array_equal(eng.state(rep, n), first)


def test_two_contexts_at_once():
    """Each context has chunks and threads of its own."""
    import threading
    n = 6 * MB + 3
    bad = []

    def go(seed):
        rng = np.random.default_rng(seed)
        st = rng.integers(0, 3, n, dtype=np.int8)
        with Engine() as eng:
            rep = eng.add_replica(np.zeros(n + 1, np.int64), np.zeros(0, np.int32), np.arange(n), st,
                                  sir_model(0.5, 0.0), 1)
            for k in range(5):
                st = np.roll(st, 1)
                eng.set_state(rep, st)
                if not np.array_equal(eng.state(rep, n), st):
                    bad.append((seed, k))

    ts = [threading.Thread(target=go, args=(s,)) for s in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


@pytest.mark.parametrize("n", [16 * MB - 1, 16 * MB, 21 * MB + 3])
def test_uploads_over_two_streams(n):
    """Around the 16 MiB from where every other chunk goes over the second
    stream: after work that still reads the states, before work that does."""
    print("two streams", n, flush=True)
    rng = np.random.default_rng(n)
    with Engine() as eng:
        rep = eng.add_replica(np.zeros(n + 1, np.int64), np.zeros(0, np.int32), np.arange(n),
                              rng.integers(0, 3, n, dtype=np.int8), sir_model(0.5, 1.0), 1)
        for _ in range(3):
            st = rng.integers(0, 3, n, dtype=np.int8)
            eng.simulate(2)
            eng.set_state(rep, st)
            assert eng.census(rep)[:3].tolist() == np.bincount(st, minlength=3).tolist()
            eng.simulate(1)                                     # every infectious agent recovers
            st[st == 1] = 2
            assert np.array_equal(eng.state(rep, n), st)
