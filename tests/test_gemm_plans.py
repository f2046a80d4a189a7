"""Which kernels the products of the GPU tests select, by the library's own rule
(no device): the direct tests reach every tile with and without a K split, and
the large products stay on the staged kernels."""

import ctypes

import numpy as np
import pytest
import test_gpu_gemm_direct as direct

from openpacho import _hip_lib

COMPUTE_UNITS = 256  # of an MI355X
TILES = {(16, 16), (16, 64), (64, 16), (32, 32), (32, 64), (64, 32)}


def plan(dtype, m, n, k, batch=1):
    """(rows, columns of a tile, splits) of a direct product, None for the staged kernels."""
    found = (ctypes.c_int64 * 3)()
    lib = _hip_lib.load()
    code = _hip_lib.DTYPE_CODES[np.dtype(dtype)]
    _hip_lib.check(lib, lib.hp_debug_direct_plan(COMPUTE_UNITS, code, m, n, k, batch, found), "hp_debug_direct_plan")
    return tuple(found) if found[0] else None


@pytest.mark.parametrize("dtype,tiles", [(np.float32, TILES | {(64, 64)}), (np.float64, TILES)])
def test_the_direct_shapes_select_every_tile_and_split(dtype, tiles):
    plans = [plan(dtype, *shape) for shape in direct.SHAPES + direct.TILE_SHAPES]
    assert None not in plans
    assert {(rows, cols, splits > 1) for rows, cols, splits in plans} == {(*t, s) for t in tiles for s in (False, True)}


def test_large_and_whole_products_stay_staged():
    for dtype, m, n, k in [(np.float32, 8192, 8192, 8192), (np.float32, 4097, 2049, 3001), (np.float32, 1024, 1024, 1024)]:
        assert plan(dtype, m, n, k) is None
    assert plan(np.float64, 512, 768, 1024, 64) is None and plan(np.float64, 4096, 4096, 4096) is None


# (type, m, n, k, batch): few K slices in many tiles, either side of the rule.
FEW_STAGED = [(np.float32, 130, 667, 20, 288), (np.float32, 80, 450, 8, 166), (np.float32, 255, 188, 96, 200)]
FEW_STAGED += [(np.float32, 5606, 426, 25, 1), (np.float32, 100, 100, 8, 2000), (np.float32, 80, 450, 32, 600), (np.float32, 200, 40, 8, 400)]
FEW_STAGED += [(np.float64, 290, 3952, 13, 1), (np.float64, 100, 100, 16, 128), (np.float64, 130, 667, 200, 288)]
FEW_DIRECT = [(np.float32, 130, 667, 20, 4), (np.float32, 80, 450, 64, 600), (np.float32, 100, 100, 32, 2000)]
FEW_DIRECT += [(np.float32, 9, 9, 4, 20000), (np.float32, 64, 64, 8, 8000), (np.float32, 20, 300, 20, 1500)]
FEW_DIRECT += [(np.float64, 290, 3952, 20, 1), (np.float64, 130, 667, 300, 288), (np.float64, 64, 64, 16, 256)]


def test_few_slices_in_many_tiles():
    assert [case for case in FEW_STAGED if plan(*case)] == []
    assert [case for case in FEW_DIRECT if not plan(*case)] == []


def test_plans_refuse_what_is_no_product():
    with pytest.raises(ValueError):
        plan(np.int32, 4, 4, 4)
    with pytest.raises(ValueError):
        plan(np.float32, 4, 0, 4)
