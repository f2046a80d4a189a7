"""Mapped reductions at the edges of their kernels: rows around one vector
group, one wave's share, the whole-workgroup rule and a chunk; columns around
the vector width, a column block and a rows-per-step count; every way a leaf
may be broadcast. Elements are small integers, so that every order of a sum
gives the same value and the comparison is exact; one case per kernel checks
that a compiled sum rounds like the eager one and stays within the bound of
its summation order on ordinary values.
"""

import subprocess

import numpy as np
import pytest

import openpacho as p
from openpacho._hip_map_reduce import BLOCK, _column_plan, map_reduce_source
from openpacho._hip_lowering import _Leaf, _identity

# (shape, reduced axes)
ROWS = [((5, n), (1,)) for n in (1, 3, 4, 5, 63, 64, 65, 1008, 1025, 8191, 8192, 8197)]
ROWS += [((4097, 1030), (1,)), ((4096, 1030), (1,)), ((3, 5, 67), (1, 2)), ((100000,), (0,)), ((70001, 3), (1,))]
COLUMNS = [((n, 5), (0,)) for n in (1, 7, 8, 9, 4099)] + [((300, n), (0,)) for n in (2, 3, 4, 63, 1023, 1024, 1025, 1028)]
COLUMNS += [((3, 50, 6), (1,)), ((2, 7, 5, 11), (1, 2)), ((20011, 257), (0,)), ((513, 1, 9), (0,))]
OTHER = [((6, 31, 7), (0, 2)), ((0, 4), (0,)), ((3, 1), (0,))]


def _leaf_shapes(shape):
    """Second operands of every broadcast kind of `shape`."""
    ones = (1,) * len(shape)
    kinds = {shape, ones, shape[-1:], shape[:-1] + (1,), shape[:1] + ones[1:]}
    if len(shape) > 2:
        kinds.add((1, shape[1]) + ones[2:])
    return sorted(kinds)


CASES = [(shape, axes, i) for i, (shape, axes) in enumerate(ROWS + COLUMNS + OTHER)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,axes,index", CASES)
def test_mapped_reductions_are_exact_on_small_integers(hip, shape, axes, index):
    # Types, operations and broadcast kinds rotate over the shapes.
    rng = np.random.default_rng(index)
    kinds = _leaf_shapes(shape)
    for turn in range(2):
        dtype = (np.float32, np.float64, np.int32)[(index + turn) % 3]
        name = "sum" if turn == 0 or not np.prod(shape) else ("min", "max")[index % 2]
        host = rng.integers(-3, 4, shape).astype(dtype)
        other = rng.integers(-3, 4, kinds[(index + turn * 2) % len(kinds)]).astype(dtype)
        function = getattr(np, name)
        compiled = p.compile(lambda x, b: function(x * b - 2, axis=axes))
        got = p.asnumpy(compiled(p.asarray(host, backend=hip), p.asarray(other, backend=hip)))
        np.testing.assert_array_equal(got, function(host * other - 2, axis=axes))


# Rows folded into long ones: by lines and by vectors, with every kind of last
# row, at the edges of the rule (64 long rows of lines, 16 of vectors), batched.
FOLDED = [((rows, 5), (0,)) for rows in (64, 816, 817, 1024, 1027, 2047, 2048, 2049, 2079, 2080)]
FOLDED += [((4 * 1024 + 3, 1025), (0,)), ((3001, 14), (0,)), ((40001, 6), (0,)), ((3, 2051, 7), (1,)), ((2, 30, 71, 9), (1, 2))]
# Past the rows or the bytes of one launch without partials.
FOLDED += [((rows, 5), (0,)) for rows in (8192, 8193, 8223, 8224)] + [((rows, 2051), (0,)) for rows in (2047, 2048, 2079)]
FOLDED += [((9001, 14), (0,)), ((3, 8195, 7), (1,)), ((2, 130, 71, 9), (1, 2))]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,axes", FOLDED)
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int64])
def test_folded_rows_are_exact_on_small_integers(hip, shape, axes, dtype):
    rng = np.random.default_rng(5)
    host = rng.integers(-3, 4, shape).astype(dtype)
    x = p.asarray(host, backend=hip)
    for kind in _leaf_shapes(shape):
        other = rng.integers(-3, 4, kind).astype(dtype)
        sums, most = p.compile(lambda x, b: (np.sum(x * b - 2, axis=axes), np.max(x - b, axis=axes)))(
            x, p.asarray(other, backend=hip)
        )
        np.testing.assert_array_equal(p.asnumpy(sums), np.sum(host * other - 2, axis=axes))
        np.testing.assert_array_equal(p.asnumpy(most), np.max(host - other, axis=axes))


# Rows of each shape that become one, by the rule: as many as start on a line
# where 64 long rows are left, on a vector where 16 are; one where single columns
# need no partials, and where rows are whole vectors. (4- and 8-byte elements)
FOLDS = [(1, 1)] * 10 + [(32, 16), (1, 1), (16, 1), (1, 1), (1, 1)]
FOLDS += [(1, 1), (32, 16), (32, 16), (32, 16), (4, 16), (32, 16), (32, 16), (16, 1), (32, 16), (32, 16)]


@pytest.mark.parametrize("case,folds", list(zip(FOLDED, FOLDS, strict=True)))
@pytest.mark.parametrize("dtype", ["f4", "f8"])
def test_folded_rows_start_on_lines_or_vectors_and_their_plans_cover_them(case, folds, dtype):
    # What the kernel then reads is compared on the device (the exact sums above).
    from openpacho._hip_map_reduce import MOST_PARTIAL_BYTES, _folded_rows, _Mapped

    (shape, axes), dtype = case, np.dtype(dtype)
    leaves = [_Leaf(False, dtype, shape), _Leaf(False, dtype, shape[-1:])]
    m = _Mapped(shape, axes, leaves, [("add", [0, 1], (dtype,) * 2, dtype)], "sum", dtype)
    width = 16 // dtype.itemsize
    folded, lines = _folded_rows(m, width)
    assert folded == folds[dtype.itemsize // 8]
    if folded == 1:
        return
    inner, reduced = folded * m.inner, -(-m.reduced // folded)
    assert inner * dtype.itemsize % (128 if lines else 16) == 0 and reduced >= (64 if lines else 16)
    assert m.outer * inner * dtype.itemsize <= MOST_PARTIAL_BYTES
    unit = 8 if lines else 1
    across, blocks, step, rows, chunks = _column_plan(m.outer, reduced, inner, width, dtype.itemsize, unit)
    assert across * step <= BLOCK and (blocks - 1) * across * width < inner <= blocks * across * width
    assert rows % step == 0 and (chunks - 1) * rows < reduced <= chunks * rows


@pytest.mark.gpu
@pytest.mark.parametrize("shape,axis", [((37, 5000), 1), ((9000, 49), 1), ((3, 20000), 1), ((20000, 129), 0)])
def test_mapped_sums_round_like_the_eager_sum_and_within_their_bound(hip, shape, axis):
    host = np.random.default_rng(1).standard_normal(shape).astype(np.float32)
    x = p.asarray(host, backend=hip)
    got = p.asnumpy(p.compile(lambda x: np.sum(x * 1.5, axis=axis))(x))
    mapped = host * np.float32(1.5)
    if axis == 1:
        np.testing.assert_array_equal(got, p.asnumpy(np.sum(x * 1.5, axis=axis)))
    exact = mapped.astype(np.float64).sum(axis=axis)
    # Recursive summation: depth * u * sum |x|. The longest chain of additions
    # is a thread's rows / 8 or 32 vector groups, then the trees and the merge
    # of the partials: below 160 for these shapes.
    bound = 160 * 2.0**-24 * np.abs(mapped.astype(np.float64)).sum(axis=axis)
    assert np.all(np.abs(got - exact) <= bound)


@pytest.mark.gpu
def test_extrema_of_mapped_rows_and_columns_keep_nan_infinities_and_signed_zeros(hip):
    host = np.full((70, 69), 5, np.float32)
    host[3, 68], host[10, 1], host[20, 40], host[30, 5] = np.nan, np.inf, -np.inf, 0.0
    host[40], host[41] = 0.0, -0.0
    host[41, 68] = 0.0
    x = p.asarray(host, backend=hip)
    for axis in (0, 1):
        for name in ("min", "max"):
            function = getattr(np, name)
            got = p.asnumpy(p.compile(lambda x: function(-x, axis=axis))(x))
            want = p.asnumpy(getattr(p, name)(-x, axis=axis))
            np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
            with np.errstate(invalid="ignore"):
                np.testing.assert_array_equal(got, function(-host, axis=axis))


@pytest.mark.parametrize("width", [2, 4])
def test_column_plans_cover_every_element_once(width):
    rng = np.random.default_rng(width)
    sizes = [1, 2, 3, 15, 16, 17, 255, 256, 257, 1025, 4096, 100003]
    for outer, reduced, inner in [(int(a), int(b), int(c)) for a, b, c in rng.choice(sizes, (400, 3))]:
        for read in (None, outer * reduced * inner * 8):
            across, blocks, step, rows, chunks = _column_plan(outer, reduced, inner, width, 8, read=read)
            groups = -(-inner // width)
            assert across * step <= BLOCK and (blocks - 1) * across < groups <= blocks * across
            assert rows % step == 0 and (chunks - 1) * rows < reduced <= chunks * rows
            assert chunks == 1 or read is None or reduced > 8192 or read > 16 << 20


@pytest.mark.parametrize("shape,axes", [((8, 100, 12), (1,)), ((8, 3, 12), (0, 2)), ((5, 8193), (1,))])
@pytest.mark.parametrize("operation,dtype", [("sum", "f8"), ("min", "u8"), ("max", "?")])
def test_sources_compile(shape, axes, operation, dtype):
    from test_abi import _compiles

    dtype = np.dtype(dtype)
    leaves = [_Leaf(False, dtype, shape), _Leaf(False, dtype, shape[-1:]), _Leaf(True, dtype, ())]
    op = "where" if dtype.kind != "b" else "equal"
    nodes = [(op, [0, 1, 2][: 3 if op == "where" else 2], (dtype,) * 3, dtype)]
    status, log = _compiles(map_reduce_source(shape, axes, leaves, nodes, operation, dtype)[0])
    assert status == 0, log


@pytest.mark.parametrize("dtype", [np.int32, np.int64, np.uint32, np.uint64])
def test_integer_sums_wrap_in_constant_expressions(dtype):
    # A constant expression may not overflow a signed type: the compiler
    # refuses one that does.
    from openpacho._hip_lowering import _combine, ctype

    info, t = np.iinfo(dtype), ctype(dtype)
    first, last = _identity("max", np.dtype(dtype)), _identity("min", np.dtype(dtype))
    source = f"""
constexpr {t} sum({t} a, {t} b) {{ return {_combine("sum", np.dtype(dtype), "a", "b")}; }}
static_assert(sum({last}, 1) == {first} && sum({first}, {last}) == ({t})({info.min + info.max}), "");
static_assert(sum({last}, {last}) == ({t})-2 && sum(({t})-1, 1) == 0, "");
"""
    done = subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-x", "c++", "-"], input=source, capture_output=True, text=True)
    assert done.returncode == 0, done.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("shape", [(7, 50), (3, 5000), (600, 6)])
def test_integer_sums_wrap_in_rows_columns_and_row_programs(hip, dtype, shape):
    host = np.random.default_rng(8).integers(np.iinfo(dtype).min, np.iinfo(dtype).max, shape, dtype=dtype, endpoint=True)

    def sums(x):
        rows = x.sum(axis=1, keepdims=True, dtype=dtype)
        return (x + 1).sum(axis=0, dtype=dtype), (x * 3).sum(axis=1, dtype=dtype), rows, x - rows

    for got, want in zip(p.compile(sums)(p.asarray(host, backend=hip)), sums(host)):
        np.testing.assert_array_equal(p.asnumpy(got), want)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", [(4095, 262144), (8191, 65537), (100003, 36), (70001, 1025), (300, 4096), (41, 9)])
def test_column_sums_keep_what_a_long_chain_would_lose(hip, dtype, shape):
    # After a first row of half the type's digits beyond one, each 1 is less
    # than half a unit in the last place: an accumulator that took the rows, or
    # pairs and fours of them, one after the other would drop them all. Sums of
    # two equal parts drop what comes before the parts reach that unit.
    digits = np.finfo(dtype).nmant
    first = 2.0 ** (digits + 5)  # a unit in the last place is 32
    weights = np.ones((shape[0], 1), dtype)
    weights[0] = first
    compiled = p.compile(lambda x, w: (x * w).sum(axis=0))
    got = p.asnumpy(compiled(p.ones(shape, dtype=dtype, backend=hip), p.asarray(weights, backend=hip)))
    exact = first + (shape[0] - 1)
    # On the way of the first row: 8 rows of a batch, the levels of at most
    # rows / 8 batches, up to 7 single rows, the tree of a step's rows and the
    # merge of the partials (their own chain of at most 16 and a tree): half a
    # unit for each sum.
    bound = (3 + np.log2(max(shape[0], 8)) + 7 + 8 + 16 + 8) * 16
    assert np.all(np.abs(got.astype(np.longdouble) - exact) <= bound), (got[0] - exact, bound)
