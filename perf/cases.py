"""Workloads of the hip backend, for timing and for comparing results.

Each case is work that a program built on openpacho has the backend do through the public
API: iterations of a dense solver, training steps of a dense network, matrix products, norms,
random arrays, column and row statistics, and layout changes. ``listed()`` names one case per
kind of work and size class; ``draw(rng)`` gives further sizes, types and options of the same
kinds.

Arrays cross between torch and openpacho as views of one device buffer: torch makes the inputs
and reads the results, openpacho computes them. Import torch first: the library then shares
torch's HIP runtime, so that one device synchronisation covers both.
"""

import math
import sys
from pathlib import Path

import numpy as np
import torch

torch.cuda.is_available()  # torch's HIP runtime is in place before the library loads

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "open-pacho_amd"))

import openpacho as p  # noqa: E402

F32, F64 = "float32", "float64"


# ---- the cases -------------------------------------------------------------------


def listed():
    return [
        # A conjugate-gradient solve of a small dense system, float64: four iterations between two looks at
        # the residual. All launches and host dispatch.
        _solve("solve_f64_300", F64, 300, 4),
        # The same solver on a system of 1 GiB: bound by reading the matrix.
        _solve("solve_f32_16384", F32, 16384, 4),
        # One SGD step (forward, backward, update) of a small dense network with ragged sizes.
        _train("train_f32_257x129x65x33", F32, 257, 129, 65, 33),
        # The same step at the batch and width of an ordinary large layer.
        _train("train_f32_8192x1024x4096x1024", F32, 8192, 1024, 4096, 1024),
        # The largest square product.
        _matmul("matmul_f32_8192", F32, 1, 8192, 8192, 8192, False),
        # A product whose every extent is odd, with the padding option.
        _matmul("matmul_f32_4097x3001x2049", F32, 1, 4097, 2049, 3001, True),
        # A batch of double-precision products (m, n, k) = (512, 768, 1024).
        _matmul("matmul_f64_64x512x768x1024", F64, 64, 512, 768, 1024, False),
        # Scaling factors of a matrix: its Frobenius norm and the norms of its columns and rows.
        _norms("norms_f32_65536x4096", F32, 65536, 4096),
        # Normal samples, 1 GiB of them.
        _random("normal_f32_2^28", F32, "normal", 1 << 28),
        # Features standardised by column over an odd number of samples and features.
        _standardise("standardise_f32_100003x1025", F32, 100003, 1025),
        # Softmax of rows.
        _softmax("softmax_f32_16384x4000", F32, 16384, 4000),
        # Layout changes of a batch of matrices: the transposes, and a crop that keeps every other column.
        _rearrange("rearrange_f32_32x1031x4096", F32, 32, 1031, 4096),
    ]


def _solve(name, dtype, n, iterations):
    return {"name": name, "kind": "solve", "dtype": dtype, "n": n, "iterations": iterations}


def _train(name, dtype, n, d, h, o):
    return {"name": name, "kind": "train", "dtype": dtype, "n": n, "d": d, "h": h, "o": o}


def _matmul(name, dtype, batch, m, n, k, padding):
    return {"name": name, "kind": "matmul", "dtype": dtype, "batch": batch, "m": m, "n": n, "k": k, "padding": padding}


def _norms(name, dtype, rows, cols):
    return {"name": name, "kind": "norms", "dtype": dtype, "rows": rows, "cols": cols}


def _random(name, dtype, distribution, count):
    return {"name": name, "kind": "random", "dtype": dtype, "distribution": distribution, "count": count}


def _standardise(name, dtype, rows, cols):
    return {"name": name, "kind": "standardise", "dtype": dtype, "rows": rows, "cols": cols}


def _softmax(name, dtype, rows, cols):
    return {"name": name, "kind": "softmax", "dtype": dtype, "rows": rows, "cols": cols}


def _rearrange(name, dtype, batch, rows, cols):
    return {"name": name, "kind": "rearrange", "dtype": dtype, "batch": batch, "rows": rows, "cols": cols}


def _size(rng, low, high):
    """A size spread over its logarithm; every other one or so is rounded to a multiple of 16."""
    value = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    if rng.random() < 0.5 and value >= 32:
        value = value // 16 * 16
    return max(low, min(high, value))


def _extents(rng, ranges, most):
    """Sizes from (low, high) ranges whose product is at most `most`, none favoured: drawn again until it is."""
    while True:
        sizes = [_size(rng, low, high) for low, high in ranges]
        if math.prod(sizes) <= most:
            return sizes


def draw(rng):
    kind = rng.choice(["solve", "train", "matmul", "norms", "random", "standardise", "softmax", "rearrange"])
    dtype = rng.choice([F32, F32, F64])
    wide = dtype == F64
    if kind == "solve":
        case = _solve("", dtype, _size(rng, 48, 11584 if wide else 16384), 4)
    elif kind == "train":
        # Five products of n x d x h or n x h x o.
        while True:
            n, d, h, o = _size(rng, 32, 16384), _size(rng, 16, 4096), _size(rng, 16, 4096), _size(rng, 8, 2048)
            if n * h * (3 * d + 3 * o) <= (1 << 36 if wide else 1 << 37):
                break
        case = _train("", dtype, n, d, h, o)
    elif kind == "matmul":
        batch = _size(rng, 2, 256) if rng.random() < 0.4 else 1
        side = 8192 if batch == 1 else 1024
        m, n, k = _extents(rng, [(16, side)] * 3, (1 << 37 if wide else 1 << 38) // batch)
        case = _matmul("", dtype, batch, m, n, k, rng.random() < 0.25)
    elif kind == "norms":
        case = _norms("", dtype, *_extents(rng, [(64, 1 << 17), (16, 16384)], 1 << (27 if wide else 28)))
    elif kind == "random":
        distribution = rng.choice(["random", "uniform", "normal", "exponential"])
        case = _random("", dtype, distribution, _size(rng, 1000, 1 << (27 if wide else 28)))
    elif kind == "standardise":
        case = _standardise("", dtype, *_extents(rng, [(256, 1 << 18), (16, 4096)], 1 << (26 if wide else 27)))
    elif kind == "softmax":
        case = _softmax("", dtype, *_extents(rng, [(64, 1 << 17), (16, 16384)], 1 << (25 if wide else 26)))
    else:
        case = _rearrange("", dtype, *_extents(rng, [(1, 64), (32, 8192), (32, 8192)], 1 << (26 if wide else 27)))
    del case["name"]
    return case


# ---- between torch and openpacho ---------------------------------------------------


class _View:
    """The device buffer of an openpacho array, as torch takes one in; it keeps the array."""

    def __init__(self, array):
        self.array = array
        self.__cuda_array_interface__ = {
            "shape": array.shape,
            "typestr": array.dtype.str,
            "data": (array._data.ptr, False),
            "version": 2,
        }


def _tensor(array):
    return torch.as_tensor(_View(array), device="cuda")


def _array(tensor):
    """An openpacho array holding a copy of `tensor`."""
    hip = p.get_backend("hip")
    array = p.empty(tuple(tensor.shape), dtype=str(tensor.dtype).replace("torch.", ""), backend=hip)
    hip.synchronize()  # the block may come from work that is still queued
    _tensor(array).copy_(tensor)
    torch.cuda.synchronize()
    return array


# ---- inputs ------------------------------------------------------------------------


def _inputs(case, seed):
    """The case's inputs as torch tensors, made from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = getattr(torch, case["dtype"])

    def uniform(*shape):
        return torch.rand(shape, generator=gen, device="cuda", dtype=dtype).mul_(2).sub_(1)

    def normal(*shape, scale=1.0):
        return torch.randn(shape, generator=gen, device="cuda", dtype=dtype).mul_(scale)

    kind = case["kind"]
    if kind == "solve":
        # Symmetric, eigenvalues within about 2.5 +- 0.82: condition number about 2.
        n = case["n"]
        a = uniform(n, n)
        a = (a + a.T).mul_(0.5 / math.sqrt(n))
        a.diagonal().add_(2.5)
        return [a.contiguous(), uniform(n)]
    if kind == "train":
        n, d, h, o = (case[k] for k in "ndho")
        return [
            uniform(n, d),
            uniform(n, o),
            normal(d, h, scale=d**-0.5),
            normal(h, scale=0.1),
            normal(h, o, scale=h**-0.5),
            normal(o, scale=0.1),
        ]
    if kind == "matmul":
        lead = (case["batch"],) if case["batch"] > 1 else ()
        return [uniform(*lead, case["m"], case["k"]), uniform(*lead, case["k"], case["n"])]
    if kind == "norms":
        # Rows of very different scale, as before an equilibration.
        x = normal(case["rows"], case["cols"])
        return [x.mul_(torch.pow(10.0, 3 * uniform(case["rows"], 1)))]
    if kind == "standardise":
        # Features with offsets and scales of their own.
        x = normal(case["rows"], case["cols"])
        return [x.mul_(torch.exp(uniform(case["cols"]))).add_(uniform(case["cols"]))]
    if kind == "softmax":
        return [normal(case["rows"], case["cols"], scale=3.0)]
    if kind == "rearrange":
        return [normal(case["batch"], case["rows"], case["cols"])]
    return []


# ---- the work ----------------------------------------------------------------------


@p.compile
def _curvature(a, direction):
    q = a @ direction
    return q, p.dot(direction, q)


@p.compile
def _update(x, r, direction, q, rr, curvature):
    alpha = rr / curvature
    r_new = r - alpha * q
    return x + alpha * direction, r_new, p.dot(r_new, r_new)


@p.compile
def _direction(r, direction, rr_new, rr):
    return r + (rr_new / rr) * direction


@p.compile
def _sgd_step(x, y, w1, b1, w2, b2, rate):
    hidden = np.tanh(x @ w1 + b1)
    residual = hidden @ w2 + b2 - y
    loss = (residual * residual).mean() / 2
    d2 = residual / (x.shape[0] * w2.shape[1])
    dw2 = hidden.T @ d2
    db2 = d2.sum(axis=0)
    d1 = (d2 @ w2.T) * (1 - hidden * hidden)
    dw1 = x.T @ d1
    db1 = d1.sum(axis=0)
    return loss, dw1, db1, dw2, db2, w1 - rate * dw1, b1 - rate * db1, w2 - rate * dw2, b2 - rate * db2


@p.compile
def _standardised(x):
    mean = x.mean(axis=0)
    centred = x - mean
    variance = (centred * centred).mean(axis=0)
    return centred / np.sqrt(variance + 1e-5), mean, variance


@p.compile
def _softmaxed(x):
    e = np.exp(x - x.max(axis=1, keepdims=True))
    return e / e.sum(axis=1, keepdims=True)


_RATE = 0.5


def prepare(case, seed):
    state = {"case": case, "seed": seed, "hip": p.get_backend("hip")}
    arrays = [_array(t) for t in _inputs(case, seed)]
    if case["kind"] == "solve":
        a, b = arrays
        arrays = [a, p.zeros(b.shape, dtype=b.dtype, backend=state["hip"]), b, p.dot(b, b)]
    state["arrays"] = arrays
    return state


def run(state):
    case, arrays = state["case"], state["arrays"]
    kind = case["kind"]
    if kind == "solve":
        a, x, r, rr = arrays
        direction = r
        for _ in range(case["iterations"]):
            q, curvature = _curvature(a, direction)
            x, r, rr_new = _update(x, r, direction, q, rr, curvature)
            direction = _direction(r, direction, rr_new, rr)
            rr = rr_new
        found = x, r, direction, rr
    elif kind == "train":
        found = _sgd_step(*arrays, _RATE)
    elif kind == "matmul":
        found = (p.matmul(*arrays, padding=case["padding"]),)
    elif kind == "norms":
        (x,) = arrays
        found = p.linalg.norm(x), p.linalg.norm(x, axis=0), p.linalg.norm(x, axis=1)
    elif kind == "random":
        rng = p.random.default_rng(state["seed"], backend=state["hip"])
        draws = {
            "random": lambda: rng.random(case["count"], dtype=case["dtype"]),
            "uniform": lambda: rng.uniform(-0.5, 1.5, case["count"], dtype=case["dtype"]),
            "normal": lambda: rng.normal(0.0, 0.01, case["count"], dtype=case["dtype"]),
            "exponential": lambda: rng.exponential(2.0, case["count"], dtype=case["dtype"]),
        }
        found = (draws[case["distribution"]](),)
    elif kind == "standardise":
        found = _standardised(*arrays)
    elif kind == "softmax":
        found = (_softmaxed(*arrays),)
    else:
        (x,) = arrays
        found = x.transpose(0, 2, 1), x[:, 1:, ::2]
    return [_tensor(array) for array in found]


def work(case):
    """Bytes: each input read once and each output written once. Operations: those of the products, and one
    for each element that a statistic or a distribution needs."""
    size = np.dtype(case["dtype"]).itemsize
    kind = case["kind"]
    if kind == "solve":
        n, iterations = case["n"], case["iterations"]
        return {"bytes": iterations * n * n * size, "flops": iterations * 2 * n * n}
    if kind == "train":
        n, d, h, o = (case[k] for k in "ndho")
        weights = d * h + h + h * o + o
        return {"bytes": size * (n * d + n * o + 3 * weights + 1), "flops": 2 * n * h * (2 * d + 3 * o)}
    if kind == "matmul":
        b, m, n, k = (case[key] for key in ("batch", "m", "n", "k"))
        return {"bytes": b * size * (m * k + k * n + m * n), "flops": 2 * b * m * n * k}
    if kind == "random":
        return {"bytes": size * case["count"], "flops": case["count"]}
    count = case["rows"] * case["cols"]
    if kind == "norms":
        return {"bytes": size * (count + case["rows"] + case["cols"] + 1), "flops": 2 * count}
    if kind == "standardise":
        return {"bytes": size * (2 * count + 2 * case["cols"]), "flops": 6 * count}
    if kind == "softmax":
        return {"bytes": size * 2 * count, "flops": 5 * count}
    moved = case["batch"] * case["rows"] * case["cols"] + case["batch"] * (case["rows"] - 1) * ((case["cols"] + 1) // 2)
    return {"bytes": size * 2 * moved, "flops": 0}


# About four times the largest error against 64 bits seen over the listed and 40 drawn cases: residuals of the
# solver 2.4e-6 / 4e-15 (float32 / float64), gradients of the step 7e-7 / 1e-15, products 1.6e-6 / 1e-15,
# everything else 1e-7 / 2e-16.
_TOLERANCES = {"solve": (1e-5, 2e-14), "train": (3e-6, 5e-15), "matmul": (6e-6, 5e-15)}


def tolerance(case):
    """Copies and the random and uniform samples are exact; the rest is what sums in another order differ by."""
    kind = case["kind"]
    if kind == "rearrange" or (kind == "random" and case["distribution"] in ("random", "uniform")):
        return "exact"
    single, double = _TOLERANCES.get(kind, (5e-7, 1e-15))
    return {"rel": double if case["dtype"] == F64 else single}


# ---- the same in 64 bits -------------------------------------------------------------


def exact(case, seed):
    kind = case["kind"]
    if kind == "random":
        return [_samples(case, seed)]
    inputs = _inputs(case, seed)
    if kind == "rearrange":
        (x,) = inputs
        return [x.transpose(1, 2).contiguous(), x[:, 1:, ::2].contiguous()]
    inputs = [t.double() for t in inputs]
    if kind == "solve":
        a, r = inputs
        x, direction, rr = torch.zeros_like(r), r, r.dot(r)
        for _ in range(case["iterations"]):
            q = a.mv(direction)
            alpha = rr / direction.dot(q)
            x, r = x + alpha * direction, r - alpha * q
            rr_new = r.dot(r)
            direction, rr = r + rr_new / rr * direction, rr_new
        return [x, r, direction, rr]
    if kind == "train":
        x, y, w1, b1, w2, b2 = inputs
        hidden = torch.tanh(x.mm(w1) + b1)
        residual = hidden.mm(w2) + b2 - y
        loss = (residual * residual).mean() / 2
        d2 = residual / residual.numel()
        dw2, db2 = hidden.T.contiguous().mm(d2), d2.sum(0)
        d1 = d2.mm(w2.T.contiguous()) * (1 - hidden * hidden)
        dw1, db1 = x.T.contiguous().mm(d1), d1.sum(0)
        steps = [w - _RATE * g for w, g in ((w1, dw1), (b1, db1), (w2, dw2), (b2, db2))]
        return [loss, dw1, db1, dw2, db2, *steps]
    if kind == "matmul":
        return [torch.matmul(*inputs)]
    (x,) = inputs
    if kind == "norms":
        return [x.norm(), x.norm(dim=0), x.norm(dim=1)]
    if kind == "standardise":
        mean = x.mean(0)
        centred = x - mean
        variance = (centred * centred).mean(0)
        return [centred / torch.sqrt(variance + 1e-5), mean, variance]
    return [torch.softmax(x, 1)]


def _words(count, seed, start):
    """The four 32-bit words of the Philox4x32-10 blocks of counters start .. start + count - 1 (Salmon et al.,
    "Parallel random numbers: as easy as 1, 2, 3", 2011), as int64."""
    low = 0xFFFFFFFF
    counter = torch.arange(start, start + count, device="cuda", dtype=torch.int64)
    x0, x1 = counter & low, counter >> 32
    x2 = x3 = torch.zeros_like(counter)
    k0, k1 = seed & low, seed >> 32
    for _ in range(10):
        left, right = x0 * 0xD2511F53, x2 * 0xCD9E8D57  # modulo 2^64: all 64 bits of the product
        x0, x1, x2, x3 = ((right >> 32) & low) ^ x1 ^ k0, right & low, ((left >> 32) & low) ^ x3 ^ k1, left & low
        k0, k1 = (k0 + 0x9E3779B9) & low, (k1 + 0xBB67AE85) & low
    return x0, x1, x2, x3


def _samples(case, seed):
    """The case's samples, from the exact unit values on in 64 bits."""
    count, wide, distribution = case["count"], case["dtype"] == F64, case["distribution"]
    out = torch.empty(count, device="cuda", dtype=torch.float64)

    def unit(high, low):
        return ((high >> 5) * 67108864 + (low >> 6)).double() * 2.0**-53 if wide else (high >> 8).double() * 2.0**-24

    chunk = 1 << 25
    for start in range(0, count, chunk):
        n = min(chunk, count - start)
        w0, w1, w2, w3 = _words(n, seed, start)
        u = unit(w0, w1)
        if distribution == "uniform":
            u = 2.0 * u - 0.5
        elif distribution == "exponential":
            u = -2.0 * torch.log1p(-u)
        elif distribution == "normal":
            u = 0.01 * (torch.sqrt(-2.0 * torch.log1p(-u)) * torch.cos(2 * math.pi * unit(w2, w3)))
        out[start : start + n] = u
    return out
