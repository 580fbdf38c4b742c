"""The plain form's runs (qvnt_amd/csrc/runs.hip) on the sizes where the split
changes: a queue applied in one call equals its SingleOps applied one call
each (their own kernels), bit for bit, in both precisions."""
import numpy as np
import pytest

from qvnt_amd import QReg, circuits, op

pytestmark = pytest.mark.gpu


# the smallest runs; one tile and two; 8 or 16 amplitudes a thread; one tile
# size and the next
@pytest.mark.parametrize("n", [4, 5, 10, 11, 12, 18, 19, 21, 22, 23])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_run_equals_single_ops(n, prec):
    queue = circuits.build(circuits.random_mixed(n, 150, circuits.rng(n, 7)), op) * op.qft((1 << min(n, 9)) - 1)
    queue *= op.h((1 << n) - 1)
    with QReg.with_state(n, 5 % (1 << n), prec=prec) as run, QReg.with_state(n, 5 % (1 << n), prec=prec) as one:
        run.apply(queue)
        for k in range(len(queue)):
            one.apply(queue[k])
        a, b = run.get_state(), one.get_state()
    assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
