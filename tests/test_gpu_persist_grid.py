"""The grid of the persistent batched launch: few blocks where its rounds are
short (they wait for each other between rounds), every block that fits where
they are long; the same bits as the rounds either way."""
import numpy as np
import pytest

from qvnt_amd import circuits, op
from qvnt_amd.batch import Batch

pytestmark = pytest.mark.gpu


def _run(q, prec, cap):
    ops = [circuits.build(circuits.random_mixed(n, 60, circuits.rng(7, k)), op) for k, n in enumerate(q)]
    with Batch(q, prec=prec) as b:
        info = b.compile(ops, max_qubits=cap, dense_min=0)
        b.run(graph=False)
        want = [b.get_state(k) for k in range(len(q))]
        for _ in range(2):
            b.reset()
            b.run(graph="persistent")
            for k in range(len(q)):
                assert np.array_equal(b.get_state(k), want[k])
        return info


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_short_rounds_take_few_blocks(prec):
    """64 registers of 14 qubits, 1024 tiles of 10 a round, a wave each: some
    hundred blocks, where every tile its own block makes the barriers the time."""
    info = _run([14] * 64, prec, 10)
    phases = info["phases"] * 16 / info["rounds"]
    assert 8 <= info["persist_blocks"] <= max(8.0, (40 * phases) ** 0.5) < 1024


def test_long_rounds_take_all_that_fit():
    """FP32 tiles of 13 (8 waves): two blocks on each of the 256 CUs."""
    assert _run([20] * 64, "f32", 13)["persist_blocks"] == 512
