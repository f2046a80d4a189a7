"""Elementwise operands broadcast along rows of any length: rows that end inside
a group of four, rows shorter than a group, values per row and per plane, and
their tails; eager and compiled, on small integers, so that the comparison with
NumPy is exact."""

import numpy as np
import pytest

import openpacho as p

pytestmark = pytest.mark.gpu

ROOTS = [(7, 5), (6, 129), (50, 1025), (9, 3), (3, 4, 7), (5, 2, 66), (4, 1, 9), (2, 3, 4, 5)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("root", ROOTS)
def test_broadcast_operands(hip, root, dtype):
    rng = np.random.default_rng(sum(root))
    host = rng.integers(-9, 10, root).astype(dtype)
    rank = len(root)
    shapes = {root[d:] for d in range(rank)} | {root[:d] + (1,) * (rank - d) for d in range(rank + 1)}
    shapes |= {(1,) * d + root[d : d + 1] + (1,) * (rank - d - 1) for d in range(rank)} | {()}
    others = [rng.integers(-9, 10, shape).astype(dtype) for shape in sorted(shapes)]
    x, rest = p.asarray(host, backend=hip), [p.asarray(v, backend=hip) for v in others]
    for value, array in zip(others, rest):
        np.testing.assert_array_equal(p.asnumpy(x * array - 2), host * value - 2)
    compiled = p.compile(lambda x, a, b, c: (x - a) * b + c)
    for i in range(len(rest)):
        at = [i, (i + 1) % len(rest), (i + 3) % len(rest)]
        got = p.asnumpy(compiled(x, *(rest[j] for j in at)))
        a, b, c = (others[j] for j in at)
        np.testing.assert_array_equal(got, (host - a) * b + c)
