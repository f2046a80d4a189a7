"""Work that would take 2^32 threads or more in one launch, which drops the
workgroups past them without an error: several launches, or workgroups that loop."""

import numpy as np
import pytest

import openpacho as p
from openpacho import _hip_map_reduce

pytestmark = pytest.mark.gpu
GROUPS = 1 << 24  # of 256 threads


def _all(array, value):
    return float(p.asnumpy(array.min())) == float(p.asnumpy(array.max())) == value


def test_compiled_reductions_of_many_small_matrices(hip):
    x = p.ones((GROUPS + 2, 2, 2), dtype=np.float32, backend=hip)
    assert _all(p.compile(lambda x: (x * 2).sum(axis=1))(x), 4)
    assert _all(p.compile(lambda x: (x * 2).sum(axis=(1, 2)))(x), 8)
    y = x.reshape(2, GROUPS + 2, 2)
    assert _all(p.compile(lambda y: (y + 1).sum(axis=(0, 2)))(y), 8)


@pytest.mark.parametrize("shape,axis", [((300, 70, 33), 1), ((40, 5, 7), 1), ((300, 2000), 0), ((7, 31, 300), (0, 2))])
def test_workgroups_that_loop_give_the_same_values(hip, monkeypatch, shape, axis):
    host = np.random.default_rng(2).integers(-5, 6, shape).astype(np.float64)
    x = p.asarray(host, backend=hip)
    function = lambda x: ((x * 2).sum(axis=axis), (x - 1).max(axis=axis))  # noqa: E731
    monkeypatch.setattr(_hip_map_reduce, "MOST_WORKGROUPS", 3)
    for got, want in zip(p.compile(function)(x), function(host)):
        np.testing.assert_array_equal(p.asnumpy(got), want)


def test_batches_of_many_small_products(hip):
    a = p.ones((GROUPS + 1, 1, 1), dtype=np.float32, backend=hip)
    assert _all(a @ (a * 3), 3)


def test_many_short_rows_times_a_vector(hip):
    rows = 4 * GROUPS + 5
    a = p.ones((rows, 2), dtype=np.float32, backend=hip)
    assert _all(a @ p.full((2,), 1.5, dtype=np.float32, backend=hip), 3)


def test_a_launch_of_too_many_threads_is_refused(hip):
    # As every other launch of the library: an error instead of a part of the work.
    a = p.ones((GROUPS + 1, 1, 1), dtype=np.int32, backend=hip)
    with pytest.raises(ValueError, match="too many tiles"):
        a @ a
