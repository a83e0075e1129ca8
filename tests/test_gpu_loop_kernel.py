"""The kernel that runs whole ticks of a small program, through the C ABI: a
schedule or an array that came after it is not overlooked."""
import ctypes

import numpy as np
import pytest

from sagesim_amd import Engine
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
