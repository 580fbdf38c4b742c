"""Results come back whole through the pinned blocks (qvnt_amd/csrc/reg.hpp:
read_back): one block, the edges of a block, more pieces than blocks."""
import numpy as np
import pytest

from qvnt_amd import QReg

pytestmark = pytest.mark.gpu


# 64 KiB is one small block; pieces of 512 KiB, four in flight
@pytest.mark.parametrize("prec, sizes", [("f64", (1, 3, 12, 13, 15, 16, 17, 19, 20)), ("f32", (1, 3, 13, 14, 16, 17, 18, 21))])
def test_state_and_probabilities_come_back_whole(prec, sizes):
    for n in sizes:
        with QReg(n, prec=prec) as reg:
            rng = np.random.default_rng(n)
            psi = (rng.standard_normal(len(reg)) + 1j * rng.standard_normal(len(reg))).astype(np.complex128 if prec == "f64" else np.complex64)
            reg.set_state(psi)
            assert np.array_equal(reg.get_state(), psi)
            w = psi.real.astype(np.float64) ** 2 + psi.imag.astype(np.float64) ** 2
            assert np.array_equal(reg.get_probabilities(), w[:1 << n] * (1.0 / reg.get_absolute()))
