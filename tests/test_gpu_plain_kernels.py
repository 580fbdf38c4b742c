"""The plain form where its kernels change with the size: the single-gate
kernels on the largest registers, runs whose blocks walk several tiles, and
the single-gate kernels as the other side of the fused form's exact check.
Every SingleOp that has to run as its own kernel is applied in a call of its
own (a queue of several is taken as runs)."""
import numpy as np
import pytest

import qvnt_amd
from qvnt_amd import QReg, circuits, op

from test_gpu_fused import permutation_circuit

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,prec", [(34, "f64"), (35, "f32")])
def test_largest_register_gate_by_gate(n, prec):
    """256 GiB of amplitudes: x, h, ry, rxx and swap on the top qubits and a
    controlled x, one call each, then the same pairs as queues (runs).  Each
    pair is a gate and its inverse, so the basis state comes back."""
    start = 0x155555555 & ((1 << n) - 1)
    top, hi2, hi3 = 1 << (n - 1), 1 << (n - 2), 1 << (n - 3)
    pairs = [(op.h(1), op.h(1)), (op.h(top), op.h(top)), (op.ry(0.9, hi2), op.ry(-0.9, hi2)),
             (op.rxx(0.5, top | hi3), op.rxx(-0.5, top | hi3)), (op.swap(hi2 | hi3), op.swap(hi2 | hi3)),
             (op.rz(0.3, hi3), op.rz(-0.3, hi3))]
    with QReg.with_state(n, start, prec=prec) as r:
        r.apply(op.x(top))
        r.apply(op.x(2).c(top))
        for gate, inverse in pairs:
            r.apply(gate)
            r.apply(inverse)
        for gate, inverse in pairs:
            r.apply(gate * inverse)
        want = start ^ top
        want ^= 2 if want & top else 0
        assert abs(r.get_absolute() - 1.0) < (1e-12 if prec == "f64" else 1e-5)
        outs = r.sample_mask((1 << n) - 1, [qvnt_amd.uniform(6, n, k) for k in range(8)])
    assert all(int(o) == want for o in outs), [hex(int(o)) for o in outs]


# 4096 blocks at most: two tiles a block from 25 qubits in FP64 (tiles of
# 2^12), 26 in FP32 (2^13)
@pytest.mark.parametrize("n,prec", [(25, "f64"), (26, "f32"), (27, "f64"), (27, "f32")])
def test_runs_over_several_tiles_a_block(n, prec):
    """Bit for bit what the SingleOps give one call each, from a state without zeros."""
    start = op.h((1 << n) - 1)
    for q in range(n):
        start *= op.rz(0.1 + 0.2 * q, 1 << q)
    queue = circuits.build(circuits.random_mixed(n, 60, circuits.rng(n, 9)), op) * op.qft(0b1111 << (n - 4))
    with QReg(n, prec=prec) as run, QReg(n, prec=prec) as one:
        run.apply(start * queue)
        whole = start * queue
        for k in range(len(whole)):
            one.apply(whole[k])
        a, b = run.get_state(), one.get_state()
    assert np.array_equal(a.view(np.uint64), b.view(np.uint64))


@pytest.mark.parametrize("n,tq,prec", [(10, 10, "f64"), (16, 10, "f64"), (20, 12, "f32"), (22, 11, "f64")])
def test_fused_permutations_equal_single_kernels(n, tq, prec):
    """A circuit of permutations through the fused form equals its SingleOps
    through their own kernels, exactly: the two share no tile code."""
    g = np.random.default_rng(7300 + n + tq)
    circ = permutation_circuit(g, n, 200)
    dt = np.complex128 if prec == "f64" else np.complex64
    psi = (g.standard_normal(1 << n) + 1j * g.standard_normal(1 << n)).astype(dt)
    with QReg(n, prec=prec) as r:
        r.set_state(psi)
        for k in range(len(circ)):
            r.apply(circ[k])
        want = r.get_state()
        r.set_state(psi)
        r.apply_fused(circ, max_qubits=tq)
        got = r.get_state()
    assert np.array_equal(got, want)


@pytest.mark.parametrize("n", [26, 27])
def test_a_run_ends_before_gates_with_many_controls(n):
    """FP32: the planner leaves gates with many controls behind a run to their
    own kernels, after it has looked at them as part of it (more phases, more
    tile qubits); between two stretches of other gates they stay in.  The same
    bits as one SingleOp a call."""
    plain, many = None, None
    for k in range(14):
        o = op.ry(0.2 + k, 1 << (4 + k % 7)) * op.rzz(0.3 + k, (1 << (4 + k % 7)) | (1 << (n - 1 - k % 3)))
        plain = o if plain is None else plain * o
    for k in range(30):
        o = (op.rx if k % 2 else op.ry)(0.4 + k, 1 << (12 + k % 4)).c(0b11111 << (17 + k % 2))
        many = o if many is None else many * o
    start = op.h((1 << n) - 1)
    for queue in (plain * many, plain * many * plain, many * plain):
        with QReg(n, prec="f32") as run, QReg(n, prec="f32") as one:
            run.apply(start)
            one.apply(start)
            run.apply(queue)
            for k in range(len(queue)):
                one.apply(queue[k])
            a, b = run.get_state(), one.get_state()
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64))
