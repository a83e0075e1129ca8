"""Programs (compiled step functions) and their context going in either order,
as a garbage collector may have them: a program destroyed after its engine was
closed, calls on it in between, and models dropped in reference cycles."""
import gc

import numpy as np
import pytest

from sagesim_amd import Breed, Model, NetworkSpace
from sagesim_amd._lib import NativeError
from sagesim_amd.steps import reference_sir_step

pytestmark = pytest.mark.gpu


def _model(n=200):
    b = Breed("SIR")
    b.register_property("state", 1)
    b.register_step_func(reference_sir_step())
    m = Model(NetworkSpace())
    m.register_breed(b)
    m.register_global_property("p_infection", 0.3)
    m.register_global_property("p_recovery", 0.1)
    m.set_seed(1)
    for i in range(n):
        m.create_agent_of_breed(b, state=1 + i % 2)
    m.get_space().connect_agents_bulk(np.arange(n - 1), np.arange(1, n))
    m.setup()
    return m


def test_engine_closed_before_its_program():
    print("[case] engine first", flush=True)
    m = _model()
    m.simulate(3)
    want = m.get_breed_data("SIR", "state")
    m._engine.close()
    m._cache = {}
    with pytest.raises(NativeError, match="context"):
        m.simulate(1)
    with pytest.raises(NativeError, match="context"):
        m.get_breed_data("SIR", "state")
    m._prog.close()
    again = _model()                    # a new context beside the closed one
    again.simulate(3)
    assert np.array_equal(again.get_breed_data("SIR", "state"), want)
    again._prog.close()                 # program first
    again._engine.close()


def test_models_dropped_in_cycles():
    print("[case] cycles", flush=True)
    want = None
    for _ in range(4):
        models = [_model() for _ in range(3)]
        for m in models:
            m.simulate(3)
        got = [m.get_breed_data("SIR", "state") for m in models]
        want = got[0] if want is None else want
        assert all(np.array_equal(g, want) for g in got)
        del m, models
        gc.collect()
