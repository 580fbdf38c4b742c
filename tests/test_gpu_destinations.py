"""get_state and get_probabilities into pageable, pinned and device memory, at
sizes on both sides of where the route changes."""
import ctypes
import time

import numpy as np
import pytest

from qvnt_amd import QReg, circuits, op
from qvnt_amd._lib import check, lib

pytestmark = pytest.mark.gpu

# (the HIP runtime's entry points, through the library that links it)
HOST, DEVICE = "hipHostMalloc", "hipMalloc"


class Buffer:
    """`size` bytes of pinned or device memory."""

    def __init__(self, kind, size):
        self.kind, self.size, self.p = kind, size, ctypes.c_void_p()
        assert (lib.hipHostMalloc(ctypes.byref(self.p), ctypes.c_size_t(size), ctypes.c_uint(0)) if kind == HOST
                else lib.hipMalloc(ctypes.byref(self.p), ctypes.c_size_t(size))) == 0

    def array(self, dtype):
        out = np.empty(self.size, np.uint8)
        assert lib.hipMemcpy(ctypes.c_void_p(out.ctypes.data), self.p, ctypes.c_size_t(self.size), ctypes.c_int(4)) == 0
        return out.view(dtype)

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        assert (lib.hipHostFree if self.kind == HOST else lib.hipFree)(self.p) == 0


def _reg(n, prec):
    r = QReg(n, prec=prec)
    r.apply(circuits.build(circuits.random_mixed(n, 30, circuits.rng(3, n)), op))
    return r


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [3, 10, 11, 15, 16, 17, 21])
@pytest.mark.parametrize("kind", [HOST, DEVICE])
def test_results_in_other_memory_than_pageable(kind, n, prec):
    with _reg(n, prec) as r:
        state, probs = r.get_state(), r.get_probabilities()
        with Buffer(kind, state.nbytes) as b:
            check(lib.qvnt_reg_get_state(r._h, b.p, state.nbytes))
            assert np.array_equal(b.array(state.dtype), state)
        with Buffer(kind, probs.nbytes) as b:
            check(lib.qvnt_reg_get_probabilities(r._h, ctypes.cast(b.p, ctypes.POINTER(ctypes.c_double)), 1 << n))
            assert np.array_equal(b.array(np.float64), probs)


def _least(call, k=7):
    best = np.inf
    for _ in range(k):
        t = time.perf_counter()
        call()
        best = min(best, time.perf_counter() - t)
    return best


def test_pinned_memory_takes_one_copy():
    """64 MiB: 1.2 ms over the bus; a host thread's second copy makes it 2.7,
    as to pageable memory (3.0)."""
    with _reg(22, "f64") as r:
        page = np.zeros(1 << 22, np.complex128)
        with Buffer(HOST, page.nbytes) as b:
            pageable = _least(lambda: check(lib.qvnt_reg_get_state(r._h, page.ctypes.data, page.nbytes)))
            pinned = _least(lambda: check(lib.qvnt_reg_get_state(r._h, b.p, page.nbytes)))
    assert pinned < 0.65 * pageable
