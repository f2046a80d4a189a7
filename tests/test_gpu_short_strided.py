"""Reductions over a short strided axis at the edges of the one-launch rule:
512 rows, the last one over it, arrays around 8 MiB. Elements are small
integers, so every order of a sum gives the same value; norms within the bound
of their summation."""

import numpy as np
import pytest

import openpacho as p

pytestmark = pytest.mark.gpu

SHAPES = [(rows, cols) for rows in (17, 33, 511, 512, 513) for cols in (2, 31, 32, 257, 1024, 1025)]
SHAPES += [(480, 4369), (480, 4370), (3, 300, 70), (2, 512, 1025)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32])
def test_short_strided_axes(hip, shape, dtype):
    host = np.random.default_rng(len(shape) + shape[-1]).integers(-9, 10, shape).astype(dtype)
    x, axis = p.asarray(host, backend=hip), len(shape) - 2
    for function in (np.sum, np.min, np.max):
        np.testing.assert_array_equal(p.asnumpy(function(x, axis=axis)), function(host, axis=axis))
    if dtype == np.int32:
        return
    want = np.sqrt((host.astype(np.float64) ** 2).sum(axis=axis))
    # A sum of n squares in any order: n / 2 units of u for its root at most.
    np.testing.assert_allclose(p.asnumpy(p.linalg.norm(x, axis=axis)), want, rtol=shape[axis] * np.finfo(dtype).eps)


def test_short_strided_axes_keep_nan_and_infinities(hip):
    host = np.ones((480, 70), np.float32)
    host[3, 1], host[479, 2], host[100, 3] = np.nan, np.inf, -np.inf
    x = p.asarray(host, backend=hip)
    for function in (np.sum, np.min, np.max):
        np.testing.assert_array_equal(p.asnumpy(function(x, axis=0)), function(host, axis=0))
    np.testing.assert_allclose(p.asnumpy(p.linalg.norm(x, axis=0)), np.linalg.norm(host, axis=0), rtol=1e-6)
