"""Row norms around every choice of the row kernels: lanes per short row, the
half and the whole chunk of a wave, rows of several chunks with few rows and
with enough of them for a wave each; lengths that are no multiple of a vector."""

import numpy as np
import pytest

import openpacho as p

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 3, 5, 16, 17, 33, 49, 64, 65, 257, 513, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4097]
SHAPES = [(11, n) for n in LENGTHS] + [(4095, 4099), (4096, 4099), (4099, 2050), (16700, 2051), (70001, 3)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("rows,length", SHAPES)
def test_row_norms(hip, rows, length, dtype):
    rng = np.random.default_rng(length)
    host = rng.standard_normal((rows, length)).astype(dtype)
    tiny, huge = (1e-30, 1e30) if dtype == np.float32 else (1e-250, 1e250)
    host[0] *= dtype(tiny)
    host[1] *= dtype(huge)
    host[2] = 0
    host[3, -1] = np.inf
    host[4, length // 2] = -np.inf
    host[4, 0] = np.nan
    host[5] = 0
    host[5, -1] = np.nan
    got = p.asnumpy(p.linalg.norm(p.asarray(host, backend=hip), axis=1))
    scale = np.ones((rows, 1), np.longdouble)
    scale[0], scale[1] = tiny, huge
    with np.errstate(invalid="ignore"):
        want = np.sqrt(np.sum((host / scale) ** 2, axis=1)) * scale[:, 0]
    # A lane's chain of fused squares is at most 65 long, then 6 butterfly
    # steps and the merges of 5 chunks; the square root halves the error.
    bound = (65 + 6 + 5) / 2 + 1
    finite = np.ones(rows, bool)
    finite[3:6] = False
    np.testing.assert_allclose(got[finite], want[finite].astype(np.float64), rtol=bound * np.finfo(dtype).eps / 2)
    assert got[3] == np.inf and np.isnan(got[4]) and np.isnan(got[5])
    assert got[2] == 0 and not np.signbit(got[2])
