"""Host side of HIPBackend without a device: its blocks and their lifetime on a
stand-in library that hands out numbers as addresses and keeps account of them,
and the launches that it arranges a plan into."""

import ctypes
import re
import shutil
import subprocess
import sys
import types
from pathlib import Path

import numpy as np
import pytest

import openpacho as p
from openpacho import _hip, _hip_lib
from openpacho._array import ndarray
from openpacho.backends import DeviceInfo


class Library:
    """The entry points that storage uses. ``live`` holds the addresses given
    out; ``after`` is called at the start of an entry point of that name."""

    def __init__(self):
        self.live, self.next, self.limit, self.after = set(), 1 << 20, None, {}
        self.most = None  # live blocks that memory has room for

    def _enter(self, name):
        if name in self.after:
            self.after[name]()

    def hp_init(self, ordinal, out):
        out._obj.value = 1
        return 0

    def hp_alloc(self, ctx, bytes, out):
        self._enter("hp_alloc")
        if self.most is not None and len(self.live) >= self.most:
            return _hip_lib.HP_E_OOM
        self.next += 1 << 20
        out.value = self.next
        self.live.add(self.next)
        return 0

    def hp_dot_new(self, ctx, code, a, b, n, out):
        return self.hp_alloc(ctx, 8, out)

    def hp_gemv(self, ctx, *args):
        """Needs one block of its own while it runs."""
        scratch = ctypes.c_void_p()
        status = self.hp_alloc(ctx, 1, scratch)
        return status or self.hp_free(ctx, scratch.value)

    def hp_free(self, ctx, ptr):
        self.live.remove(ptr)
        return 0

    def hp_set_pool_limit(self, ctx, value):
        self._enter("hp_set_pool_limit")
        self.limit = value
        return 0

    def hp_release_cached(self, ctx):
        return 0

    def hp_destroy(self, ctx):
        return 0

    def hp_last_error(self):
        return b""

    def __getattr__(self, name):  # bound by the backend, unused here
        if name.startswith("hp_"):
            return None
        raise AttributeError(name)


@pytest.fixture
def backend(monkeypatch):
    device = DeviceInfo("0", "stand-in", "AMD", "GPU", True, 256 << 30, "")
    monkeypatch.setattr(_hip, "hip_devices", lambda: [device])
    monkeypatch.setattr(_hip_lib, "load", Library)
    made = _hip.HIPBackend()
    yield made
    made.close()


def _waiting(backend):
    return list(backend._small) + [ptr for kept in backend._kept.values() for ptr in kept]


def _at_instruction(method, number, action, *args):
    """Call ``method``; before its ``number``-th instruction call ``action``.
    False when it has fewer instructions."""
    code, left = method.__func__.__code__, [number]

    def trace(frame, event, arg):
        if frame.f_code is not code:
            return None
        frame.f_trace_opcodes = True
        if event == "opcode":
            left[0] -= 1
            if left[0] == 0:
                sys.settrace(None)
                action()
                sys.settrace(trace)
        return trace

    sys.settrace(trace)
    try:
        method(*args)
    finally:
        sys.settrace(None)
    return left[0] <= 0


def test_a_block_dropped_while_the_waiting_ones_go_back_is_not_lost(backend):
    # The garbage collector may run a finaliser between any two instructions:
    # one drops a block of another class there, and every block is afterwards
    # either back in the library or waiting.
    number, reached = 0, True
    while reached:
        number += 1
        blocks = [backend.empty((n,), np.bool_) for n in (3, 40, 5000, 70000)]
        late = [backend.empty((n,), np.bool_) for n in (9, 300000)]
        blocks.clear()
        with backend._lock:
            reached = _at_instruction(backend._return_small, number, late.clear)
        late.clear()
        assert set(_waiting(backend)) == backend._lib.live, f"before instruction {number}"
        assert len(_waiting(backend)) == len(set(_waiting(backend)))
    assert number > 10


def _out_of_memory(backend, live):
    """``live`` blocks in use, others waiting, and no memory for any more."""
    used = [backend.empty((100000,), np.bool_) for _ in range(live)]
    dropped = [backend.empty((n,), np.bool_) for n in (5000, 5000, 70000)]
    dropped.clear()
    backend._lib.most = len(backend._lib.live)
    assert len(_waiting(backend)) == 3
    return used


def test_waiting_blocks_go_back_before_an_allocation_fails(backend):
    used = _out_of_memory(backend, 2)
    used.append(backend.empty((1 << 21,), np.bool_))  # no block of its class waits
    assert not _waiting(backend) and len(backend._lib.live) == 3
    backend._lib.most = 3
    with pytest.raises(RuntimeError, match="hp_alloc"):
        backend.empty((1 << 21,), np.bool_)


def test_waiting_blocks_go_back_before_a_call_that_needs_memory_fails(backend):
    used = _out_of_memory(backend, 1)
    backend._call("hp_gemv")
    assert not _waiting(backend) and backend._lib.live == {used[0].ptr}
    backend._lib.most = 1
    with pytest.raises(RuntimeError, match="hp_gemv"):
        backend._call("hp_gemv")


def test_waiting_blocks_go_back_before_a_dot_fails(backend):
    used = _out_of_memory(backend, 1)
    vector = ndarray._wrap(used[0], (10,), np.dtype("float32"), backend)
    out = backend.vector_dot(vector, vector)
    assert not _waiting(backend) and backend._lib.live == {used[0].ptr, out.ptr}
    backend._lib.most = 2
    with pytest.raises(RuntimeError, match="hp_dot_new"):
        backend.vector_dot(vector, vector)


def test_no_block_waits_past_a_pool_limit(backend):
    # A block dropped as the limit falls (by a finaliser or another thread) is
    # judged by the new limit.
    number, reached = 0, True
    while reached:
        number += 1
        backend.pool_limit = 1 << 40
        late = [backend.empty((100000,), np.bool_)]
        setter = types.MethodType(type(backend).pool_limit.fset, backend)
        reached = _at_instruction(setter, number, late.clear, 0)
        late.clear()
        assert backend.pool_limit == backend._lib.limit == 0
        assert not any(backend._kept.values()), f"before instruction {number}"
    assert number > 10


def test_a_refused_pool_limit_changes_nothing(backend):
    backend.pool_limit = 1 << 40
    backend._lib.hp_set_pool_limit = lambda ctx, value: _hip_lib.HP_E_HIP
    with pytest.raises(RuntimeError, match="hp_set_pool_limit"):
        backend.pool_limit = 0
    assert backend.pool_limit == 1 << 40


# ---- plans -------------------------------------------------------------------------


def _launches(backend, function, shape, dtype):
    """The launches of a compiled function of one array."""
    plan, _ = p.compile(function)._plan((p.empty(shape, dtype=dtype, backend=backend),), {})
    return plan._launches


def _and_squares(function):
    def result(x):
        y = function(x)
        return y, (y * y).sum(axis=-1)

    return result


def _softmax(x):
    e = np.exp(x - x.max(axis=-1, keepdims=True))
    return e / e.sum(axis=-1, keepdims=True)


POWER, TANH, SIN = (_and_squares(f) for f in (lambda x: x**1.7, np.tanh, np.sin))
# Rows that one launch serves, and rows that stay steps: few long ones of
# operations that keep a lane busy, at 16, 32 and 64 elements a lane and around
# the workgroups that fill the chip; and any whose unrolled code is too long.
ONE = [(POWER, (4, 4096), "f4"), (POWER, (4, 4096), "f8"), (POWER, (1024, 8192), "f4"), (POWER, (1024, 8192), "f8")]
ONE += [(TANH, (4, 4096), "f8"), (TANH, (256, 8192), "f8"), (TANH, (4, 16384), "f4"), (SIN, (4, 8192), "f8")]
ONE += [(SIN, (4, 8192), "f4"), (SIN, (4096, 14336), "f4"), (_softmax, (4, 16384), "f4"), (_softmax, (4, 8192), "f8")]
STEPS = [(POWER, (4, 8192), "f4"), (POWER, (512, 8192), "f4"), (POWER, (64, 8192), "f8"), (POWER, (256, 16384), "f4"), (TANH, (64, 8192), "f8")]
STEPS += [(SIN, (4, 16384), "f4"), (SIN, (16384, 16384), "f4"), (_and_squares(lambda x: np.sin(x) + np.cos(x)), (4096, 10240), "f8")]


@pytest.mark.parametrize("function,shape,dtype", ONE)
def test_rows_that_one_launch_serves(backend, function, shape, dtype):
    assert len(_launches(backend, function, shape, dtype)) == 1


@pytest.mark.parametrize("function,shape,dtype", STEPS)
def test_rows_that_stay_steps(backend, function, shape, dtype):
    assert len(_launches(backend, function, shape, dtype)) == 2


def test_long_rows_stay_in_registers(tmp_path, backend):
    if not (shutil.which("hipcc") or Path("/opt/rocm/bin/hipcc").exists()):
        pytest.skip("hipcc not available")
    import build

    both = _and_squares(lambda x: np.sin(x) + np.cos(x))
    for function, shape, dtype in [(SIN, (4096, 14336), "f4"), (both, (4096, 8192), "f8"), (TANH, (4096, 10240), "f8")]:
        (launch,) = _launches(backend, function, shape, dtype)
        source = tmp_path / "rows.hip"
        source.write_text("#include <hip/hip_runtime.h>\n" + launch.payload.source)
        command = [build.hipcc(), "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-fhip-fp32-correctly-rounded-divide-sqrt"]
        command += ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-c"]
        command += ["-Rpass-analysis=kernel-resource-usage", str(source), "-o", str(tmp_path / "rows.o")]
        remarks = subprocess.run(command, capture_output=True, text=True, check=True).stderr
        assert re.search(r"ScratchSize \[bytes/lane\]: 0\b", remarks), (shape, dtype)
