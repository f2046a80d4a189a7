"""What a compiled function keeps: as many plans as its cache holds, and nothing
of the calls whose plans were dropped."""

import gc
import weakref

import numpy as np

import openpacho as p
from openpacho.backends import NumpyBackend


def test_dropped_plans_leave_nothing_behind():
    compiled = p.compile(lambda x, scale: x * scale, cache_size=2)
    backend = NumpyBackend()
    seen = weakref.ref(backend)
    compiled(p.ones((3,), backend=backend), 2.0)
    for n in (4, 5):  # the plan of the first call goes
        compiled(p.ones((n,)), 2.0)
    assert set(compiled._quick.values()) == set(compiled._plans)
    del backend
    gc.collect()
    assert seen() is None
    for _ in range(3):  # and comes back as any other
        for n in (3, 4, 5):
            np.testing.assert_array_equal(p.asnumpy(compiled(p.ones((n,)), 0.5)), np.full(n, 0.5))
            assert set(compiled._quick.values()) <= set(compiled._plans)
    compiled.clear_cache()
    assert not compiled._quick and not compiled._plans
