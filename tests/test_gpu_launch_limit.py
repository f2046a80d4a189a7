"""Work that would take 2^32 threads or more in one launch: split, or refused,
never a part of the result. (A launch drops the workgroups past that.)"""

import numpy as np
import pytest

import openpacho as p

pytestmark = pytest.mark.gpu
GROUPS = 1 << 24  # of 256 threads


def test_compiled_reductions_of_too_many_column_blocks_are_refused(hip):
    x = p.ones((GROUPS + 2, 2, 2), dtype=np.float32, backend=hip)
    with pytest.raises(ValueError, match="too many threads"):
        p.compile(lambda x: (x * 2).sum(axis=1))(x)
    rows = p.compile(lambda x: (x * 2).sum(axis=(1, 2)))(x)  # many rows share a workgroup
    assert float(p.asnumpy(rows.min())) == float(p.asnumpy(rows.max())) == 8


def test_batches_of_too_many_products_are_refused(hip):
    a, b = (p.ones((GROUPS + 1, 1, 1), dtype=np.float32, backend=hip) for _ in range(2))
    with pytest.raises(ValueError, match="too many tiles"):
        a @ b
    c = a[: GROUPS - 1] @ b[: GROUPS - 1]
    assert float(p.asnumpy(c.min())) == 1
