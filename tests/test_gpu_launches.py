"""Regrouped launches of compiled plans: row programs at the edges of their lane
rule, of a lane's groups and of what they refuse; values recomputed by their
readers; independent elementwise steps in one launch. Each plan against NumPy
and against its steps run one by one, which every elementwise output matches
bit for bit, and unchanged explain() steps."""

import numpy as np
import pytest

import openpacho as p
from openpacho import _hip_lowering

pytestmark = pytest.mark.gpu


def _softmax(x):
    e = np.exp(x - x.max(axis=-1, keepdims=True))
    return e / e.sum(axis=-1, keepdims=True)


def _layer_norm(x, gain, shift):
    centred = x - x.mean(axis=-1, keepdims=True)
    variance = (centred * centred).mean(axis=-1, keepdims=True)
    return centred / np.sqrt(variance + 1e-5) * gain + shift, variance


def _standardise(x):
    mean = x.mean(axis=0)
    centred = x - mean
    return centred / np.sqrt((centred * centred).mean(axis=0) + 1e-5), mean


def _update(x, r, d, q, rr, curvature):
    alpha = rr / curvature
    r_new = r - alpha * q
    return x + alpha * d, r_new, (r_new * r_new).sum()


def _square(x):
    total = x.sum(axis=1)  # a row result read along the other axis
    return x - total, x.max(axis=1, keepdims=True) * x


def _stepwise(monkeypatch, function, args):
    """The plan with one launch per step."""
    with monkeypatch.context() as patch:
        patch.setattr(_hip_lowering.HIPLowering, "arrange", lambda self, steps, outputs: steps)
        return p.compile(function)(*args)


def _launches(compiled):
    (plan,) = compiled._plans.values()
    return plan._launches


def _check(hip, monkeypatch, function, host, launches=None, exact=False):
    args = [p.asarray(v, backend=hip) for v in host]
    compiled = p.compile(function)
    got = compiled(*args)
    plain = _stepwise(monkeypatch, function, args)
    want = function(*(v.astype(np.float64) for v in host))
    single = host[0].dtype == np.float32
    for g, s, w in zip(*(v if isinstance(v, tuple) else (v,) for v in (got, plain, want))):
        assert g.shape == s.shape == w.shape and g.dtype == s.dtype == host[0].dtype
        a, b = p.asnumpy(g), p.asnumpy(s)
        if exact:
            np.testing.assert_array_equal(a, b)
        # exp and the quotient of sums of up to 16384 terms in fixed short
        # chains: a few units in the last place of the row's largest value.
        tolerance = 64 * np.finfo(a.dtype).eps
        scale = np.abs(w).max() if w.size else 1.0
        np.testing.assert_allclose(a, w, rtol=tolerance if single else 1e-12, atol=tolerance * scale)
        np.testing.assert_allclose(a, b, rtol=tolerance, atol=tolerance * scale)
    if launches is not None:
        assert len(_launches(compiled)) == launches
    return compiled, args


WIDTHS = [2, 3, 5, 16, 17, 63, 64, 65, 1000, 1009, 1024, 1025, 2048, 2049, 4097, 8192]


@pytest.mark.parametrize("width", WIDTHS)
def test_row_programs(hip, monkeypatch, width):
    rng = np.random.default_rng(width)
    dtype = (np.float32, np.float64)[width % 2]
    rows = 4100 if 1000 <= width <= 2049 else 7
    x = rng.standard_normal((rows, width)).astype(dtype) * 3
    _check(hip, monkeypatch, _softmax, [x], launches=1)
    gain, shift = (rng.uniform(0.5, 1, width).astype(dtype) for _ in range(2))
    if width >= 16:  # the variance of a few values may be nearly zero
        _check(hip, monkeypatch, _layer_norm, [x, gain, shift])


def test_row_programs_of_three_dimensions_and_of_rows_too_long_for_registers(hip, monkeypatch):
    rng = np.random.default_rng(0)
    _check(hip, monkeypatch, _softmax, [rng.standard_normal((3, 5, 130)).astype(np.float32)], launches=1)
    _check(hip, monkeypatch, lambda x: np.exp(x - x.max(axis=(1, 2), keepdims=True)) * 2, [rng.standard_normal((4, 6, 33))], launches=1)
    compiled, _ = _check(hip, monkeypatch, _softmax, [rng.standard_normal((3, 40000)).astype(np.float32)])
    assert len(_launches(compiled)) > 1
    _check(hip, monkeypatch, _square, [rng.standard_normal((40, 40)).astype(np.float32)])


def test_row_programs_keep_nan_and_infinite_rows_apart(hip, monkeypatch):
    x = np.random.default_rng(1).standard_normal((70, 50)).astype(np.float32)
    x[3, 7], x[4, 49], x[5] = np.nan, np.inf, -np.inf
    args = [p.asarray(x, backend=hip)]
    with np.errstate(invalid="ignore"):
        want = _softmax(x)
    got = p.asnumpy(p.compile(_softmax)(*args))
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_allclose(got, want, rtol=1e-5, equal_nan=True)


@pytest.mark.parametrize("shape", [(3000, 129), (257, 1), (2, 64)])
def test_values_recomputed_by_their_readers(hip, monkeypatch, shape):
    x = np.random.default_rng(2).standard_normal(shape) + 1
    compiled, args = _check(hip, monkeypatch, _standardise, [x], exact=True)
    kinds = [s["kind"] for s in compiled.explain(*args)["steps"]]
    assert kinds.count("fused") >= 3 and "map_reduce" in kinds  # the centred array is still a step
    centred = [s for s in compiled._plans[next(iter(compiled._plans))].steps if s.kind == "fused" and s.node.op == "subtract"]
    assert all(launch is not s for s in centred for launch in _launches(compiled))


def test_independent_steps_share_a_launch(hip, monkeypatch):
    rng = np.random.default_rng(3)
    scalars = [np.asarray(v) for v in (2.5, 1.25)]
    for size, outputs in ((1001, 3), (100001, 2)):  # with the sum as one row, and the two vectors alone
        vectors = [rng.standard_normal(size) for _ in range(4)]
        compiled, _ = _check(hip, monkeypatch, _update, [*vectors, *scalars], exact=True)
        joined = [launch for launch in _launches(compiled) if hasattr(launch, "nodes")]
        assert len(joined) == 1 and len(joined[0].nodes) == outputs

    def several(a, b, c):
        return a + 1, b * 2.0, np.exp(c), (a - 3).sum(), b - b

    arrays = [rng.standard_normal(s) for s in ((7, 5), (70000,), (2, 3, 4))]
    compiled, _ = _check(hip, monkeypatch, several, arrays)
    assert len(_launches(compiled)) <= 3


def test_scalars_rebind_and_dtypes_mix_in_regrouped_launches(hip, monkeypatch):
    rng = np.random.default_rng(4)
    host = rng.integers(-5, 6, (60, 33)).astype(np.int32)

    def mixed(x, scale):
        y = x * scale
        return y - y.max(axis=1, keepdims=True), y > 0, (y * y).sum(axis=1)

    compiled = p.compile(mixed)
    x = p.asarray(host, backend=hip)
    for scale in (2, -3):
        for got, want in zip(compiled(x, scale), mixed(host, np.int32(scale))):
            np.testing.assert_array_equal(p.asnumpy(got), want)
    assert compiled.cache_info()["misses"] == 1


@pytest.mark.parametrize("count", [40, 505, 520])
def test_many_operands(hip, count):
    # Several groups whose operands together pass what one launch packs, and one
    # group around that limit (505 and 520 pointers, a flag and a number).
    host = [np.full(70, i % 7, np.int32) for i in range(count)]
    arrays = [p.asarray(v, backend=hip) for v in host]

    def total(values):
        return values[0] if len(values) == 1 else total(values[: len(values) // 2]) + total(values[len(values) // 2 :])

    names = [f"a{i}" for i in range(count)]
    scope = {"total": total}
    result = "total(a) * flag + scale" if count > 100 else "tuple(total(a) * flag + scale + j for j in range(8))"
    exec(f"def function(flag, {', '.join(names)}, scale):\n    a = [{', '.join(names)}]\n    return {result}", scope)
    function = scope["function"]
    got, want = p.compile(function)(True, *arrays, 3), function(True, *host, 3)
    for g, w in zip(*(v if isinstance(v, tuple) else (v,) for v in (got, want))):
        np.testing.assert_array_equal(p.asnumpy(g), w)
