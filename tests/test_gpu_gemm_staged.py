"""The tables of test_gpu_gemm.py on the LDS-staged kernels that they are about:
the rows that the direct kernels take over are run with those off."""

import numpy as np
import pytest
import test_gpu_gemm as g
from test_gemm_plans import plan

pytestmark = pytest.mark.gpu

F32, F64 = np.float32, np.float64
MODES = [(256, 128, 16), (512, 256, 64), (257, 129, 17), (300, 200, 100), (1, 1, 1), (31, 33, 4099), (640, 384, 48)]
MODES += [(777, 300, 64), (257, 257, 32), (513, 1023, 16)]
ALIGNMENTS = [(300, 260, 64), (512, 256, 48), (129, 70, 37)]
TRANSPOSED = [flags for flags in g.LAYOUTS if any(flags)]


@pytest.fixture
def staged(hip):
    hip._call("hp_debug_staged_products", 1)
    yield hip
    hip._call("hp_debug_staged_products", 0)


def _direct(dtype, m, n, k, batch=()):
    return plan(dtype, m, n, k, int(np.prod(batch, dtype=int))) is not None


@pytest.mark.parametrize("dtype", [F32, F64])
@pytest.mark.parametrize("m,n,k", MODES)
def test_kernel_modes(staged, dtype, m, n, k):
    g.test_kernel_modes_against_float64(staged, dtype, m, n, k)


@pytest.mark.parametrize("case", [c for c in g.STREAM_K_CASES if _direct(c[0], *c[2:], c[1])])
def test_stream_k_splits(staged, case):
    g.test_stream_k_splits_against_float64_and_deterministic(staged, *case)


@pytest.mark.parametrize("dtype", [F32, F64])
@pytest.mark.parametrize("m,n,k", ALIGNMENTS)
def test_operands_at_element_alignment(staged, dtype, m, n, k):
    g.test_operands_at_element_alignment(staged, dtype, m, n, k)


@pytest.mark.parametrize("ta,tb", g.LAYOUTS)
@pytest.mark.parametrize("case", [c for c in g.WIDE_CASES + g.HALF_CASES if _direct(F32, *c[1:], c[0])])
def test_wide_and_half_tiles(staged, ta, tb, case):
    if case[0] and (ta or tb):
        pytest.skip("transposed operands are 2-D")
    g.test_wide_tiles_against_float64_and_deterministic(staged, ta, tb, *case)


@pytest.mark.parametrize("ta,tb", g.LAYOUTS)
@pytest.mark.parametrize("m,n,k", [c for c in g.ODD_K_CASES if _direct(F32, *c)])
def test_odd_k(staged, ta, tb, m, n, k):
    g.test_odd_k_products_against_float64_and_deterministic(staged, ta, tb, m, n, k)


@pytest.mark.parametrize("dtype", [F32, F64])
@pytest.mark.parametrize("ta,tb", TRANSPOSED)
@pytest.mark.parametrize("m,k,n", g.LAYOUT_SHAPES)
def test_transposed_operands(staged, monkeypatch, dtype, ta, tb, m, k, n):
    g.test_compiled_transpose_products_read_operands_in_place(staged, monkeypatch, dtype, ta, tb, m, k, n)


@pytest.mark.parametrize("dtype", [F32, F64])
def test_batch_strides_off_the_16_byte_grid(staged, dtype):
    g.test_batch_strides_off_the_16_byte_grid(staged, dtype)


@pytest.mark.parametrize("dtype", [F32, F64])
@pytest.mark.parametrize("batch,m,n,k", [(3, 300, 280, 77), (2, 256, 256, 1001), (4, 129, 513, 33), (2, 520, 260, 3)])
def test_k_edge_of_adjacent_batch_matrices(staged, dtype, batch, m, n, k):
    g.test_k_edge_of_adjacent_batch_matrices_contracts_zeros(staged, dtype, batch, m, n, k)


@pytest.mark.parametrize("m,k,n", [c for c in g.EDGE_CASES if _direct(F32, c[0], c[2], c[1])])
def test_edge_strips(staged, m, k, n):
    g.test_edge_strips_against_float64_and_repeatable(staged, m, k, n)


@pytest.mark.parametrize("ta,tb", g.LAYOUTS)
@pytest.mark.parametrize("m,k,n", [c for c in g.STRIP_LAYOUT_CASES if _direct(F32, c[0], c[2], c[1])])
def test_edge_strips_in_every_layout(staged, ta, tb, m, k, n):
    g.test_edge_strips_in_every_layout_match_materialized_transposes(staged, ta, tb, m, k, n)


@pytest.mark.parametrize("m,k,n", [(33, 4081, 257), (65, 4095, 1023), (95, 8191, 2051)])
def test_dyadic_products(staged, monkeypatch, m, k, n):
    g.test_dyadic_products_are_exact_and_rebinding_is_copy_free(staged, monkeypatch, m, k, n)


@pytest.mark.parametrize("dtype", [F32, F64])
def test_special_values(staged, dtype):
    g.test_special_values_and_subnormals_propagate(staged, dtype)
