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


# Several chunks of a wave (4096 float32 or 2048 float64), around one, two and four
# butterflies of 64 of them.
LONG = [(np.float32, n) for n in (8190, 4096 * 63 + 5, 4096 * 64, 4096 * 65, 4096 * 127 + 4)]
LONG += [(np.float64, n) for n in (2 * 2048 + 2, 64 * 2048, 129 * 2048 + 1, 255 * 2048 + 8)]


@pytest.mark.parametrize("dtype,length", LONG)
def test_a_norm_does_not_depend_on_the_number_of_rows(hip, dtype, length):
    # 4096 rows are walked by a wave each; fewer leave pairs to a merge kernel.
    rows = 4096
    x = p.random.default_rng(length, backend=hip).normal(0.0, 1.0, (rows, length), dtype=np.dtype(dtype).name)
    walked = p.asnumpy(p.linalg.norm(x, axis=1))
    few = x[: rows - 1000]
    del x
    np.testing.assert_array_equal(p.asnumpy(p.linalg.norm(few, axis=1)), walked[: rows - 1000])
    exact = np.linalg.norm(p.asnumpy(few[:20]).astype(np.longdouble), axis=1)
    # A lane's chain of at most 65 fused squares, the wave's 6 steps, the 6 of
    # the butterfly over chunks and the merges of 4; the root halves the error.
    bound = (65 + 6 + 6 + 4) / 2 + 1
    np.testing.assert_allclose(walked[:20], exact.astype(np.float64), rtol=bound * np.finfo(dtype).eps / 2)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("length", [17, 49, 64, 65, 257, 1024])
def test_short_rows_keep_squares_below_half_a_unit(hip, length, dtype):
    # After a leading 1 each square is just under half a unit in the last place:
    # one chain of a lane's 16 elements drops 15 of them (7.5 units of u for the
    # root). Of four chains the one with the 1 drops at most 4; sums of parts
    # that grew apart from it are off by half a unit each, 2 + 6 of them, and so is the root.
    host = np.full((70, length), 0.99 * np.sqrt(np.finfo(dtype).eps / 2), dtype)
    host[:, 0] = 1
    got = p.asnumpy(p.linalg.norm(p.asarray(host, backend=hip), axis=1))
    exact = np.linalg.norm(host.astype(np.longdouble), axis=1)
    np.testing.assert_allclose(got, exact.astype(np.float64), rtol=(4 + 2 + 6 + 1) / 4 * np.finfo(dtype).eps)


@pytest.mark.parametrize("rows", [(1 << 29) + 3, (1 << 30) + 65])
def test_more_short_rows_than_one_launch_takes(hip, rows):
    # The norm of a single element is its absolute value.
    x = p.random.default_rng(3, backend=hip).normal(0.0, 1.0, (rows, 1), dtype="float32")
    norms = p.linalg.norm(x, axis=1)
    apart = np.max(np.abs(norms - np.abs(x.reshape(rows))))
    assert float(p.asnumpy(apart)) == 0
    del x, apart
    assert float(p.asnumpy(norms[-1:])[0]) > 0  # the last row was written
