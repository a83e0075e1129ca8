"""What the device finds out about a network when a replica is made: the hashes
of its entries and key ids as a checkpoint carries them, against the same sums in
numpy and plain integers, and the first row or entry that is wrong.  Whole
numbers: equal exactly.
"""
import numpy as np
import pytest

from sagesim_amd import Engine, sir_model
from sagesim_amd._lib import NativeError

pytestmark = pytest.mark.gpu


def mix64(x):
    x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return x ^ (x >> np.uint64(31))


def csr_hash(deg, col):
    row = np.repeat(np.arange(deg.shape[0], dtype=np.uint64), deg)
    with np.errstate(over="ignore"):
        fwd = (row << np.uint64(32)) | col.astype(np.uint64)
        a = mix64(fwd ^ np.uint64(0x9E3779B97F4A7C15))
        b = mix64(fwd * np.uint64(0xD6E8FEB86659FD93) + np.uint64(0x2545F4914F6CDD1D))
        return int(a.sum(dtype=np.uint64)), int(b.sum(dtype=np.uint64))


def key_hash(ids):
    h = 1469598103934665603
    for i in ids.tolist():
        h = ((h ^ (i & (2 ** 64 - 1))) * 1099511628211) % 2 ** 64
    return h


def degrees(kind, n, rng):
    if kind == "short":
        return rng.integers(0, 6, n)
    if kind == "hub":                                   # one row for many threads, then ones
        return np.concatenate([[5000], np.ones(n - 1, np.int64)])
    if kind == "holes":                                 # runs of empty rows inside a thread's entries
        return np.where(np.arange(n) % 37 == 5, 7, 0)
    return np.full(n, 16)                               # "even": rows as long as a thread's share


@pytest.mark.parametrize("kind", ["short", "hub", "holes", "even"])
@pytest.mark.parametrize("n,ghosts", [(1, 0), (63, 1), (64, 0), (257, 100), (4099, 64), (110_001, 0)])
def test_hashes_of_a_network(kind, n, ghosts):
    rng = np.random.default_rng(n + ghosts)
    deg = degrees(kind, n, rng).astype(np.int64)
    rp = np.concatenate([[0], np.cumsum(deg)])
    col = rng.integers(0, n + ghosts, rp[-1]).astype(np.int32)
    ids = rng.integers(0, 2 ** 40 if n == 257 else 2 ** 31, n)
    st = rng.integers(0, 3, n + ghosts).astype(np.int8)
    print("create", kind, n, ghosts, col.shape[0], flush=True)
    with Engine() as eng:
        rep = eng.add_replica(rp, col, ids, st, sir_model(0.3, 0.1), 5, n_ghost=ghosts)
        words = eng.replica_save(rep)[:64].view(np.uint64).tolist()
        assert np.array_equal(eng.state(rep, n + ghosts), st)
    assert words[2:5] == [n, ghosts, col.shape[0]]
    assert tuple(words[5:7]) == csr_hash(deg, col)
    assert words[7] == key_hash(ids)


@pytest.mark.parametrize("n", [2, 65, 5000])
def test_the_first_wrong_row_or_entry_is_named(n):
    rng = np.random.default_rng(n)
    rp = np.arange(n + 1, dtype=np.int64) * 3
    col = rng.integers(0, n, 3 * n).astype(np.int32)
    ids, st = np.arange(n), np.zeros(n, np.int8)
    with Engine() as eng:
        for at in sorted({0, 1, n // 2, n - 2}):
            bad = rp.copy()
            bad[at + 1:n] += 4                          # row at reaches past where its successors ...
            bad[n - 1] = bad[n] + 1                     # ... and the last row begins past its end
            first = int(np.flatnonzero(np.diff(bad) < 0)[0])
            with pytest.raises(NativeError, match=f"row_ptr decreases at row {first}$"):
                eng.add_replica(bad, col, ids, st, sir_model(0.3, 0.1), 1)
        for at in sorted({0, 15, 16, 3 * n - 1} & set(range(3 * n))):
            for v in (-1, n):
                bad = col.copy()
                bad[at] = v
                bad[-1] = n + 7 if at < 3 * n - 1 else v
                with pytest.raises(NativeError, match=rf"col_idx\[{at}\] = {v} outside"):
                    eng.add_replica(rp, bad, ids, st, sir_model(0.3, 0.1), 1)
        assert eng.replica_save(eng.add_replica(rp, col, ids, st, sir_model(0.3, 0.1), 1)).shape[0] > 0
