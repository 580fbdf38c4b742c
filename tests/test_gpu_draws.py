"""Draws and norms on the device (qvnt_amd/csrc/measure.hip) at the edges of
their stages -- one lane's worth of leaves, one wave's, one stored level,
two -- against the pairwise tree in numpy, bit for bit."""
import numpy as np
import pytest

from qvnt_amd import QReg, circuits, op

pytestmark = pytest.mark.gpu


def tree(psi):
    re, im = psi.real.astype(np.float64), psi.imag.astype(np.float64)
    level = [re * re + im * im]
    while len(level[-1]) > 1:
        level.append(level[-1][0::2] + level[-1][1::2])
    return level


def draw(level, u):
    x = u * level[-1][0]
    j = np.zeros(len(u), np.int64)
    for nodes in level[-2::-1]:
        left, right = nodes[2 * j], nodes[2 * j + 1]
        go_left = (x < left) | (right == 0.0)
        x = np.where(go_left, x, x - left)
        j = 2 * j + np.where(go_left, 0, 1)
    return j.astype(np.uint64)


# 4095 draws are the most that go through pinned memory
@pytest.mark.parametrize("n", [1, 2, 3, 5, 6, 7, 10, 11, 12, 13, 17, 18, 21, 22, 23, 24])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_draws_and_norm_equal_the_tree(n, prec):
    ops = op.h((1 << n) - 1) * circuits.build(circuits.random_mixed(max(n, 2), 30, circuits.rng(n, 9)), op) if n > 1 else op.ry(0.7, 1)
    with QReg.with_state(n, 0, prec=prec) as reg:
        reg.apply(ops)
        level = tree(reg.get_state()[:1 << n])
        assert reg.get_absolute() == level[-1][0]
        mask = (1 << n) - 1
        for shots in (1, 2, 4095, 4096):
            u = np.random.default_rng(shots).random(shots)
            u[0] = 0.0 if shots > 1 else u[0]
            assert np.array_equal(reg.sample_mask(mask, u), draw(level, u))
        u = np.random.default_rng(7).random(100)
        assert np.array_equal(reg.sample_mask_noalloc(mask, u), draw(level, u))


# zero subtrees are never entered, wherever they lie
@pytest.mark.parametrize("n", [8, 16, 23])
def test_draws_skip_zero_subtrees(n):
    for state in (0, 1, (1 << n) - 1, (1 << n) // 2, (1 << n) // 3):
        with QReg.with_state(n, state) as reg:
            got = reg.sample_mask((1 << n) - 1, np.array([0.0, 0.3, np.nextafter(1.0, 0.0)]))
            assert np.array_equal(got, np.full(3, state, np.uint64))
