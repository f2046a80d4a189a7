"""Direct products at the edges of their tiles: extents around 16, 32 and 64 (a
tile that undercuts an extent, tiles moved back inside one), K below, at and
around one slice and one slice per wave, K split over workgroups, batches with
broadcasting, every layout, operands at element alignment. Against float64, and
bit for bit between layouts and between calls. Memory next to the operands is
NaN, which a read that reaches an output would carry there."""

import numpy as np
import pytest

import openpacho as p
from openpacho import _hip_lib

pytestmark = pytest.mark.gpu

# (m, n, k)
SHAPES = [(1, 1, 1), (2, 3, 15), (15, 17, 16), (16, 16, 17), (17, 31, 63), (31, 33, 64), (33, 63, 65), (63, 64, 79)]
SHAPES += [(64, 65, 80), (65, 127, 129), (129, 66, 257), (100, 1000, 33), (1000, 40, 70), (5, 700, 2000), (700, 9, 2000)]
SHAPES += [(48, 48, 5000), (130, 130, 4099), (16, 2050, 1030), (321, 322, 323), (900, 1000, 500)]


def _product(hip, code, a, b, m, n, k, ta, tb, dtype):
    """C through hp_gemm_layout with NaN around operands held at an odd element offset."""
    def held(host):
        flat = np.full(host.size + 64, np.nan, dtype)
        flat[33 : 33 + host.size] = host.reshape(-1)
        array = p.asarray(flat, backend=hip)
        return array, array._data.ptr + 33 * dtype.itemsize

    (left, pa), (right, pb) = held(np.ascontiguousarray(a.T if ta else a)), held(np.ascontiguousarray(b.T if tb else b))
    out = p.full((m * n + 64,), np.nan, dtype=dtype, backend=hip)
    hip._call("hp_gemm_layout", code, pa, pb, out._data.ptr, m, n, k, int(ta), int(tb))
    got = p.asnumpy(out)
    assert np.isnan(got[m * n :]).all(), "stored past the end of C"
    del left, right
    return got[: m * n].reshape(m, n)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_direct_products_in_every_layout(hip, dtype, m, n, k):
    dtype = np.dtype(dtype)
    rng = np.random.default_rng(m + n + k)
    a, b = rng.uniform(-1, 1, (m, k)).astype(dtype), rng.uniform(-1, 1, (k, n)).astype(dtype)
    exact = a.astype(np.longdouble) @ b.astype(np.longdouble)
    # Any order of k products and sums is off by at most gamma_k |A| |B|
    # (gamma_k ~ k u); the float64 reference of the test adds its own.
    bound = (k + 1) * np.finfo(dtype).eps / 2 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64))
    code = _hip_lib.DTYPE_CODES[dtype]
    first = None
    for ta, tb in ((False, False), (False, True), (True, False), (True, True)):
        got = _product(hip, code, a, b, m, n, k, ta, tb, dtype)
        assert np.all(np.abs(got - exact) <= bound), (ta, tb)
        first = got if first is None else first
        np.testing.assert_array_equal(got, first)
    np.testing.assert_array_equal(_product(hip, code, a, b, m, n, k, False, False, dtype), first)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("left,right", [((7, 20, 45), (7, 45, 33)), ((3, 1, 66, 17), (5, 17, 65)), ((40, 70, 300), (300, 18))])
def test_direct_batches_broadcast(hip, dtype, left, right):
    rng = np.random.default_rng(3)
    a, b = rng.uniform(-1, 1, left).astype(dtype), rng.uniform(-1, 1, right).astype(dtype)
    got = p.asnumpy(p.asarray(a, backend=hip) @ p.asarray(b, backend=hip))
    k = left[-1]
    bound = (k + 1) * np.finfo(dtype).eps / 2 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64))
    assert np.all(np.abs(got - a.astype(np.longdouble) @ b.astype(np.longdouble)) <= bound)


# Shapes for every tile, with and without a K split (test_gemm_plans.py checks that
# the set is complete): narrow extents below, at and above one block of 16.
TILE_SHAPES = [(9, 8200, 300), (16, 4100, 300), (17, 4100, 65), (5, 700, 4099), (16, 700, 4099), (31, 700, 4099)]
TILE_SHAPES += [(n, m, k) for m, n, k in TILE_SHAPES]
TILE_SHAPES += [(5, 9, 4099), (33, 2050, 17), (64, 129, 4099), (64, 4100, 17), (64, 129, 8192), (129, 64, 8192)]
TILE_SHAPES += [(8192, 33, 17), (4100, 70, 64), (300, 70, 8192), (64, 8200, 17), (8200, 64, 17), (64, 300, 8192)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("m,n,k", TILE_SHAPES)
def test_every_direct_tile_in_every_layout(hip, dtype, m, n, k):
    test_direct_products_in_every_layout(hip, dtype, m, n, k)
