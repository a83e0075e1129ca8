"""The kernel that runs whole ticks of a small program, through the C ABI: a
schedule or an array that came after it is not overlooked."""
import ctypes

import numpy as np
import pytest

from sagesim_amd import Breed, Engine, Model, NetworkSpace, StepFunction
from sagesim_amd import model as model_mod
from sagesim_amd._lib import ptr
from sagesim_amd.model import _Program

pytestmark = pytest.mark.gpu

_SOURCE = r"""
#include "sagesim_rt.h"
static __device__ void bump(const SSProgArgs *A, int id, long long i) {
    if (A->prop_r[id]) ss_st((float *)A->prop_w[id] + i, ss_ld((const float *)A->prop_r[id] + i) + 1.0f);
}
extern "C" __global__ void step(const SSProgArgs *A, long long tick, long long start, long long count,
                                const int *order) {
    const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= count) return;
    bump(A, 0, start + k);
    bump(A, 1, start + k);
}
extern "C" __global__ void ticks(const SSProgArgs *A, long long tick, long long ticks) {
    for (long long t = tick; t < tick + ticks; ++t) {
        for (int k = threadIdx.x; k < 100; k += blockDim.x) bump(A, 0, k);
        __syncthreads();
        ss_write_back(A->prop_w[0], A->prop_r[0], 400, threadIdx.x, blockDim.x);
        __syncthreads();
    }
}
"""


class _Small:
    """100 agents, one float each, a step that adds 1 to every array it finds."""

    def __init__(self, eng):
        self.prog = _Program(eng, 100)
        self.L, self.h, self.ck = self.prog._L, self.prog._h, self.prog.ck
        self.add()
        self.ck(self.L.ss_prog_compile(self.h, _SOURCE.encode(), b"step\nticks", None, 0))
        self.schedule(0, 100)
        self.ck(self.L.ss_prog_set_loop(self.h, 1, 128))

    def add(self):
        aid = ctypes.c_int32()
        self.ck(self.L.ss_prog_add_prop(self.h, 4, 1, 1, ptr(np.zeros(100, np.float32)), ctypes.byref(aid)))

    def schedule(self, start, count):
        self.ck(self.L.ss_prog_set_schedule(self.h, 1, ptr(np.zeros(1, np.int32)), ptr(np.array([start], np.int64)),
                                            ptr(np.array([count], np.int64))))

    def run(self, ticks, arrays):
        self.ck(self.L.ss_prog_simulate(self.h, 0, ticks))
        out = np.empty((arrays, 100), np.float32)
        for i in range(arrays):
            self.ck(self.L.ss_prog_prop_download(self.h, i, ptr(out[i])))
        return out


def test_loop_then_schedule():
    print("[case] loop, then another schedule", flush=True)
    with Engine(0) as eng:
        p = _Small(eng)
        assert np.array_equal(p.run(3, 1), np.full((1, 100), 3))
        p.schedule(10, 20)
        want = np.full((1, 100), 3)
        want[0, 10:30] = 5
        assert np.array_equal(p.run(2, 1), want)
        p.prog.close()


def test_loop_then_array():
    print("[case] loop, then another array", flush=True)
    with Engine(0) as eng:
        p = _Small(eng)
        p.run(3, 1)
        p.add()
        assert np.array_equal(p.run(2, 2), np.array([[5.0], [2.0]]).repeat(100, 1))
        p.prog.close()


_WALK = """
__device__ void walk(auto tick, auto agent_index, auto n_agents, auto agent_ids, auto breeds, auto locations,
                     auto state) {
    float sum = 0.0f;
    for (int j = 0; j < (int)n_agents; ++j)
        sum += state[j] * (float)rand_uniform_philox(tick, agent_index, j);
    state[agent_index] = 0.5f * state[agent_index] + sum / (float)n_agents;
}
"""


def _walkers(n, limit, monkeypatch):
    """n agents whose step walks all of them."""
    monkeypatch.setattr(model_mod, "_LOOP_AGENTS", limit)
    b = Breed("Walker")
    b.register_property("state", 1.0)
    b.register_step_func(StepFunction("walk", _WALK), priority=0)
    m = Model(NetworkSpace())
    m.register_breed(b)
    m.register_global_property("n_agents", n)
    m.set_seed(3)
    for i in range(n):
        m.create_agent_of_breed(b, state=float(i % 7))
    m.get_space().connect_agents_bulk(np.arange(n - 1), np.arange(1, n))
    m.setup()
    return m


def _loop_of(m):
    k = ctypes.c_int32(-2)
    m._prog.ck(m._prog._L.ss_prog_loop(m._prog._h, ctypes.byref(k)))
    return k.value


@pytest.mark.parametrize("calls", [[100], [1] * 8, [3, 30, 2]])
@pytest.mark.parametrize("n", [1, 300, 2000])
def test_heavy_step(n, calls, monkeypatch):
    """A step that keeps one block busy for a millisecond a tick goes back to the
    schedule after a few ticks, with the same results."""
    print("[case] heavy step", n, calls, flush=True)
    one, many = _walkers(n, 2048, monkeypatch), _walkers(n, 0, monkeypatch)
    assert _loop_of(one) >= 0 and _loop_of(many) == -1
    for c in calls:
        one.simulate(c)
        many.simulate(c)
        assert np.array_equal(one.get_breed_data("Walker", "state"), many.get_breed_data("Walker", "state"))
    if n == 2000:
        assert _loop_of(one) == -1
