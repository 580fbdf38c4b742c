"""Kernel statistics of the norm: one reduction over the state at every size,
also where no level of its tree is stored (up to 2^11 amplitudes)."""
import pytest

from qvnt_amd import QReg, op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 10, 11, 12, 20, 23])
@pytest.mark.parametrize("prec,amp", [("f64", 16), ("f32", 8)])
def test_norm_is_one_reduction(n, prec, amp):
    with QReg(n, prec=prec) as r:
        r.apply(op.h((1 << n) - 1))
        r.set_timing(True)
        r.kernel_stats(reset=True)
        for calls in (1, 2):
            assert abs(r.get_absolute() - 1.0) < (1e-12 if prec == "f64" else 1e-5)
            got = r.kernel_stats()["reduce"]
            assert got["launches"] == calls and got["bytes"] == calls * amp * max(1 << n, 8) and got["ms"] > 0.0
