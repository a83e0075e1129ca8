"""One-tick calls of a live exchange: the halo read from page-locked memory by
a kernel, and the boundary states packed into it, against the same run in one
call from ordinary memory.  Both are copies of whole numbers: equal exactly.
"""
import numpy as np
import pytest

from sagesim_amd import Engine, pack_2bit, sir_model, workloads
from sagesim_amd._lib import NativeError
from sagesim_amd.engine import Replica

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


@pytest.mark.parametrize("drop", [0, 1, 2, 3])
@pytest.mark.parametrize("offset", [0, 1, 4])
def test_ticks_one_by_one_from_page_locked_memory(offset, drop):
    """Halo lengths and starts of every width the copy has, bytes and 2-bit."""
    pw = workloads.sbm_partition(n_blocks=4, block_size=1500, deg_in=8, deg_out=1, n_parts=2, part=1, ticks=6, seed=31)
    g = pw.graph
    ids = pw.halo_ids[:pw.halo_ids.shape[0] - drop]
    vals = np.ascontiguousarray(pw.halo_vals(0, pw.ticks)[:, :ids.shape[0]])
    slots = np.arange(g.n, g.n_cols, dtype=np.int32)
    out = []
    with Engine() as eng:
        for mode in ("one call", "bytes", "2bit", "mixed"):
            say("exchange", offset, drop, mode, g.n, ids.shape[0])
            rep = Replica(eng, g, pw.state, sir_model(pw.beta, pw.gamma), pw.seed, rng_key_id=pw.local_ids,
                          history=pw.history)
            eng.map_build(rep.rep, pw.ghost_ids, slots, 0.5)
            eng.halo_bind(rep.rep, ids)
            if mode == "one call":
                eng.simulate_halo(rep.rep, pw.ticks, vals)
            for t in range(pw.ticks) if mode != "one call" else ():
                packed = mode == "2bit"
                row = pack_2bit(vals[t]) if packed else vals[t]
                if mode == "mixed" and t % 2:                   # staged through the ring, into the same buffers
                    eng.simulate_halo(rep.rep, 1, row)
                    continue
                whole = eng.pinned_empty((offset + row.shape[0],), row.dtype)
                buf = whole[offset:]
                buf[...] = row
                (eng.simulate_halo_2bit if packed else eng.simulate_halo)(rep.rep, 1, buf)
                buf[...] = 0xFF if packed else 3                # the call is done with the buffer
            out.append((rep.states(), rep.history()))
            rep.remove()
    for st, hist in out[1:]:
        assert np.array_equal(st, out[0][0])
        assert np.array_equal(hist, out[0][1])


@pytest.mark.parametrize("n", [1, 3, 4, 5, 255, 1024, 1027, 200_001, 300_000])
def test_pack_either_side_of_the_staging_size(n):
    """Packs through page-locked memory and, above its size, through the
    device's workspace."""
    g = workloads.sbm_partition(n_blocks=4, block_size=1500, deg_in=8, deg_out=1, n_parts=2, part=0, ticks=1,
                                seed=3).graph
    rng = np.random.default_rng(n)
    state = rng.integers(0, 3, g.n_cols).astype(np.int8)
    with Engine() as eng:
        rep = Replica(eng, g, state, sir_model(0.3, 0.1), 9)
        say("pack", n)
        eng.simulate(2)
        st = rep.states()
        agents = rng.integers(0, g.n, n)
        slots = rep.inv[agents].astype(np.int32)
        assert np.array_equal(eng.halo_pack(rep.rep, slots), st[agents])
        assert np.array_equal(eng.halo_pack_2bit(rep.rep, slots), pack_2bit(st[agents]))


@pytest.mark.parametrize("n", [1, 4, 5, 1027, 300_000])
def test_pack_of_a_slot_outside(n):
    """A slot outside the replica, anywhere in the list, is an error, and the
    next pack is not."""
    g = workloads.sbm_partition(n_blocks=4, block_size=1500, deg_in=8, deg_out=1, n_parts=2, part=0, ticks=1,
                                seed=3).graph
    state = np.random.default_rng(n).integers(0, 3, g.n_cols).astype(np.int8)
    with Engine() as eng:
        rep = Replica(eng, g, state, sir_model(0.3, 0.1), 9)
        agents = np.random.default_rng(n + 1).integers(0, g.n, n)
        slots = rep.inv[agents].astype(np.int32)
        for at in sorted({0, n // 2, n - 1}):
            for wrong in (-1, rep.n_total, 2**31 - 1, -(2**31)):
                say("pack outside", n, at, wrong)
                bad = slots.copy()
                bad[at] = wrong
                for pack in (eng.halo_pack, eng.halo_pack_2bit):
                    with pytest.raises(NativeError, match="slot %d outside the replica" % wrong):
                        pack(rep.rep, bad)
        assert np.array_equal(eng.halo_pack(rep.rep, slots), state[agents])
        assert np.array_equal(eng.halo_pack_2bit(rep.rep, slots), pack_2bit(state[agents]))
