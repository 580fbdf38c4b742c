"""The work that users of this engine have it do, as cases that can be timed.

A case is a register (or a batch, or a served mix) taken through the public
entry points: basis state, circuit, readout.  The circuits are the package's
own families (qvnt_amd.circuits) drawn from the seed.  Registers that a
program keeps are made in prepare() and reset at the start of each pass;
the short-lived ones are made and dropped inside the pass.

The readout is what the size allows: the whole state or its probabilities
while they fit a few MiB, shots of measured qubits and the norm beyond.  FP32
states of 2^25 amplitudes and more are measured on their top eight qubits, and
their norm is given in FP32: finer than that is below the rounding of the
amplitudes.
"""
import math
import random

import numpy as np
import torch

from qvnt_amd import QReg, circuits, op
from qvnt_amd.batch import Batch
from qvnt_amd.program import Program, Sym
from qvnt_amd.serve import Server

SHOTS = 1024


def listed():
    return [
        # smallest calls: a fresh register, its QFT, its state -- launches and latency
        dict(name="qft-10q-f64", kind="fresh", form="plain", prec="f64", circuit="qft", n=10, depth=1),
        # the reference's own benchmark loop: register made, two small QFTs, one qubit measured, register dropped
        dict(name="reference-loop-18q", kind="loop", form="plain", prec="f64", circuit="qft", n=18, depth=1),
        # an algorithm in FP32 on an odd size, gate by gate as the reference applies it
        dict(name="mixed-15q-f32", kind="state", form="plain", prec="f32", circuit="mixed", n=15, depth=300),
        # the 20-qubit workload: qft, h, 200 random gates, shots on the low byte, probabilities
        dict(name="plain-20q-f64", kind="probs", form="plain", prec="f64", circuit="plain20", n=20, depth=200),
        # a QASM program: measure, branch on the classical bits, reset, go on
        dict(name="program-17q-f64", kind="program", form="plain", prec="f64", circuit="mixed", n=17, depth=120),
        # one Trotter step of the Ising ring in FP32, gate by gate
        dict(name="tfim-27q-f32", kind="shots", form="plain", prec="f32", circuit="tfim", n=27, depth=1),
        # the headline: one layer of the 30-qubit brickwork circuit (16 GiB), gate by gate
        dict(name="brickwork-30q-f64", kind="shots", form="plain", prec="f64", circuit="brickwork", n=30, depth=1),
        # the fused form on an ordinary circuit: compile, passes and the state back
        dict(name="fused-mixed-16q-f64", kind="state", form="fused", prec="f64", circuit="mixed", n=16, depth=400),
        # ten brickwork layers in one fused call
        dict(name="fused-brickwork-30q-f64", kind="shots", form="fused", prec="f64", circuit="brickwork", n=30, depth=10),
        # time evolution: one fused call per Trotter step, FP32, an odd number of qubits
        dict(name="fused-tfim-31q-f32", kind="evolve", form="fused", prec="f32", circuit="tfim", n=31, depth=3),
        # many small uneven registers in one batch, each with its own circuit and shots
        dict(name="batch-96-10..18q-f64", kind="batch", form="fused", prec="f64", circuit="mixed", n=18, low=10, count=96, depth=400),
        # requests of mixed sizes served side by side
        dict(name="serve-24-12..24q-f64", kind="serve", form="fused", prec="f64", circuit="mixed", n=24, low=12, count=24, depth=1000),
    ]


def draw(rng):
    kind = rng.choice(["fresh", "loop", "state", "state", "probs", "program", "shots", "shots", "shots", "evolve", "batch", "serve"])
    form = rng.choice(["plain", "fused"])
    prec = rng.choice(["f64", "f32"])
    if kind == "fresh":
        return dict(kind=kind, form=form, prec=prec, circuit="qft", n=rng.randint(4, 14), depth=1)
    if kind == "loop":
        return dict(kind=kind, form="plain", prec=prec, circuit="qft", n=rng.randint(16, 21), depth=1)
    if kind == "state":
        return dict(kind=kind, form=form, prec=prec, circuit=rng.choice(["mixed", "mixed", "brickwork", "tfim"]), n=rng.randint(8, 18),
                    depth=_log(rng, 20, 800))
    if kind == "probs":
        return dict(kind=kind, form=form, prec="f64", circuit="plain20", n=rng.randint(17, 21), depth=_log(rng, 50, 500))
    if kind == "program":
        return dict(kind=kind, form="plain", prec="f64", circuit="mixed", n=rng.randint(9, 19), depth=_log(rng, 20, 200))
    if kind == "shots":
        circuit = rng.choice(["brickwork", "tfim", "mixed"])
        n = rng.randint(22, 29) if form == "plain" else rng.randint(22, 31)
        depth = rng.randint(1, 2) if form == "plain" else rng.randint(1, 8)
        return dict(kind=kind, form=form, prec=prec, circuit=circuit, n=n, depth=depth * n if circuit == "mixed" else depth)
    if kind == "evolve":
        return dict(kind=kind, form="fused", prec=prec, circuit="tfim", n=rng.randint(22, 30), depth=rng.randint(2, 6))
    if kind == "batch":
        low = rng.randint(8, 12)
        return dict(kind=kind, form="fused", prec=prec, circuit="mixed", n=low + rng.randint(4, 7), low=low, count=_log(rng, 24, 200),
                    depth=_log(rng, 60, 500))
    low = rng.randint(10, 14)
    return dict(kind=kind, form="fused", prec="f64", circuit="mixed", n=low + rng.randint(5, 11), low=low, count=_log(rng, 6, 32),
                depth=_log(rng, 150, 1500))


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# ------------------------------------------------------------------ inputs

def _gates(case, seed):
    """The circuit's calls, each a list of (constructor, arguments, control)."""
    n, depth = case["n"], case["depth"]
    if case["circuit"] == "qft":
        if case["kind"] == "loop":
            return [[("qft", (0b0111,), 0), ("qft", (0b1110,), 0)]]
        return [[("qft", ((1 << n) - 1,), 0)]]
    if case["circuit"] == "plain20":
        return [circuits.plain_20q(seed, n, depth)[1]]
    if case["circuit"] == "mixed":
        return [circuits.random_mixed(n, depth, circuits.rng(seed, 11))]
    if case["circuit"] == "brickwork":
        # (small registers: depth counts gates, large ones: layers)
        layers = depth if case["kind"] != "state" else max(1, depth // (5 * n))
        return [sum((circuits.brickwork_layer(n, k, seed) for k in range(layers)), [])]
    steps = depth if case["kind"] != "state" else max(1, depth // (2 * n))
    # angles of the order of 1 from the seed first: the ring starts in no basis state
    start = [("u3", tuple(circuits.rng(seed, 12 + q).uniform(0.0, math.pi, 3)) + (1 << q,), 0) for q in range(n)]
    start = [(c, tuple(float(x) for x in a[:3]) + a[3:], k) for c, a, k in start]
    step = circuits.tfim_step(n, seed=seed)
    if case["kind"] == "evolve":
        return [start + step] + [step] * (steps - 1)
    return [start + step * steps]


def _basis(case, seed):
    return random.Random(seed).getrandbits(case["n"])


def _mask(case, seed):
    """The measured qubits of a large register."""
    n = case["n"]
    if case["prec"] == "f32":
        return 0xFF << (n - 8)
    return sum(1 << q for q in random.Random(seed + 1).sample(range(n), 8))


def _draws(seed, count=SHOTS):
    return np.random.default_rng(seed).random(count)


def _program(case, seed):
    """Three stretches of gates: measure three qubits, branch on them, reset one, measure two more."""
    n, r = case["n"], random.Random(seed + 2)
    q = r.sample(range(n), 6)
    part = [circuits.random_mixed(n, case["depth"], circuits.rng(seed, 20 + k)) for k in range(3)]
    first, second = (1 << q[0]) | (1 << q[1]) | (1 << q[2]), (1 << q[3]) | (1 << q[4])
    branch = [("x", (1 << q[3],), 0), ("rx", (r.uniform(0, 6), 1 << q[5]), 0)]
    return part, first, second, branch, r.randrange(8), 1 << q[5], [r.random(), r.random()]


def _registers(case, seed):
    r = random.Random(seed + 3)
    out = []
    for k in range(case["count"]):
        n = r.randint(case["low"], case["n"])
        specs = circuits.random_mixed(n, r.randint(max(20, case["depth"] // 10), case["depth"]), circuits.rng(seed, 100 + k))
        mask = sum(1 << q for q in r.sample(range(n), 8))
        out.append((n, specs, mask, _draws(seed * 1000 + k)))
    return out


def prepare(case, seed):
    kind, n, prec = case["kind"], case["n"], case["prec"]
    s = dict(case=case)
    if kind == "batch":
        regs = _registers(case, seed)
        s["regs"] = regs
        s["batch"] = Batch([r[0] for r in regs], prec=prec)
        s["batch"].compile([circuits.build(r[1], op) for r in regs], max_qubits=11)
        return s
    if kind == "serve":
        s["reqs"] = [(k, circuits.build(specs, op), m, mask, u) for k, (m, specs, mask, u) in enumerate(_registers(case, seed))]
        s["server"] = Server(8 << 30, slots=4)
        return s
    if kind == "program":
        part, first, second, branch, value, reset, draws = _program(case, seed)
        p = Program(n, 5)
        p.apply(circuits.build(part[0], op)).measure(first, 0b00111).if_eq(0b00111, value, circuits.build(branch, op))
        p.apply(circuits.build(part[1], op)).reset(reset)
        p.apply(circuits.build(part[2], op)).measure(second, 0b11000)
        s["sym"], s["draws"] = Sym(p, prec=prec), draws
        return s
    s["ops"] = [circuits.build(g, op) for g in _gates(case, seed)]
    s["basis"] = _basis(case, seed)
    if kind in ("fresh", "loop"):
        s["u"] = float(_draws(seed, 1)[0])
        return s
    s["mask"] = 0xFF if kind == "probs" else _mask(case, seed) if kind != "state" else 0
    s["draws"] = _draws(seed)
    s["reg"] = QReg(n, prec=prec)
    return s


# --------------------------------------------------------------- the passes

def _apply(reg, case, ops):
    for o in ops:
        if case["form"] == "plain":
            reg.apply(o)
        else:
            reg.apply_fused(o)


def _norm(reg, case):
    """The norm of the state, in the register's precision."""
    total = reg.get_absolute()
    return total if case["prec"] == "f64" else np.float32(total)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "fresh":
        with QReg.with_state(case["n"], s["basis"], prec=case["prec"]) as reg:
            _apply(reg, case, s["ops"])
            return {"state": reg.get_state()}
    if kind == "loop":
        with QReg.with_state(case["n"], s["basis"], prec=case["prec"]) as reg:
            _apply(reg, case, s["ops"])
            outcome = reg.measure_mask(0b100, u=s["u"]).get()
            return {"outcome": outcome, "weight": _norm(reg, case)}
    if kind == "batch":
        b = s["batch"]
        b.reset()
        b.run(graph=True)
        got = [b.sample_mask(k, mask, u) for k, (_, _, mask, u) in enumerate(s["regs"])]
        total = np.array([t for _, t in got])
        return {"outcomes": np.stack([o for o, _ in got]), "total": total if case["prec"] == "f64" else total.astype(np.float32)}
    if kind == "serve":
        server = s["server"]
        for k, o, n, mask, u in s["reqs"]:
            server.submit(k, n, o, mask, u, dense_min=3)
        got = sorted(server.drain(len(s["reqs"])), key=lambda r: r["id"])
        return {"outcomes": np.stack([r["outcomes"] for r in got]), "total": np.array([r["total"] for r in got])}
    if kind == "program":
        sym = s["sym"]
        sym.reset()
        sym.finish(draws=s["draws"])
        return {"class": sym.get_class().get(), "probabilities": sym.get_probabilities()}
    reg = s["reg"]
    reg.reset(s["basis"])
    _apply(reg, case, s["ops"])
    if kind == "state":
        return {"state": reg.get_state()}
    outcomes = reg.sample_mask(s["mask"], s["draws"])
    if kind == "probs":
        return {"outcomes": outcomes, "probabilities": reg.get_probabilities()}
    return {"outcomes": outcomes, "norm": _norm(reg, case)}


def work(case):
    """The state written once by the reset or read once by the readout, and
    each call's circuit read and written once; 7 operations an amplitude for
    each constructor of a circuit (u3 is three of them)."""
    amp = 16 if case["prec"] == "f64" else 8
    kind = case["kind"]

    def flops(specs, n):
        k = 0
        for ctor, args, _ in specs:
            w = bin(args[0]).count("1") if ctor in ("h", "qft") else 1
            k += {"u3": 3, "h": (w + 1) // 2, "qft": w * (w + 1) // 2}.get(ctor, 1)
        return 7.0 * k * 2.0 ** n

    if kind in ("batch", "serve"):
        regs = _registers(case, 0)
        return {"bytes": float(sum(4 * (amp << n) + 16 * SHOTS for n, _, _, _ in regs)), "flops": sum(flops(g, n) for n, g, _, _ in regs)}
    n = case["n"]
    if kind == "program":
        part = _program(case, 0)[0]
        return {"bytes": 10.0 * (amp << n) + 8.0 * (1 << n), "flops": sum(flops(g, n) for g in part)}
    calls = _gates(case, 0)
    back = {"state": amp << n, "fresh": amp << n, "probs": 8 << n}.get(kind, 0)
    return {"bytes": (2.0 * len(calls) + 2.0) * (amp << n) + back, "flops": sum(flops(g, n) for g in calls)}


# --------------------------------------------------- the same in 64 bits

class _Plain:
    """A state vector in torch, complex128: textbook matrices on its axes."""

    def __init__(self, n, state):
        self.n = n
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.psi = torch.zeros(1 << n, dtype=torch.complex128, device=self.dev)
        self.psi[state] = 1.0

    def _parts(self, bits, ctrl):
        """Views of the amplitudes whose control qubits are 1, by the values of the qubits `bits` (bits[0] lowest)."""
        v = self.psi.view([2] * self.n)
        where = [slice(None)] * self.n
        for q in range(self.n):
            if ctrl >> q & 1:
                where[self.n - 1 - q] = 1
        out = []
        for k in range(1 << len(bits)):
            at = list(where)
            for j, q in enumerate(bits):
                at[self.n - 1 - q] = k >> j & 1
            out.append(v[tuple(at)])
        return out

    def matrix(self, m, bits, ctrl=0):
        x = self._parts(bits, ctrl)
        y = [sum(complex(m[r][c]) * x[c] for c in range(len(x)) if m[r][c] != 0) for r in range(len(x))]
        for v, w in zip(x, y):
            v.copy_(w)

    def diag(self, d, bits, ctrl=0):
        for v, f in zip(self._parts(bits, ctrl), d):
            if f != 1:
                v.mul_(complex(f))

    def apply(self, specs):
        for ctor, args, ctrl in specs:
            self.gate(ctor, args, ctrl)

    def gate(self, ctor, args, ctrl):
        bits = [q for q in range(self.n) if args[-1] >> q & 1]
        i, h = 1j, math.sqrt(0.5)
        if ctor == "h":
            for q in bits:
                self.matrix([[h, h], [h, -h]], [q], ctrl)
        elif ctor == "qft":
            for k, q in enumerate(bits):
                self.matrix([[h, h], [h, -h]], [q], ctrl)
                for j, t in enumerate(bits[k + 1:], 1):
                    self.gate("rz", (math.pi / 2 ** j, 1 << t), ctrl | 1 << q)
        elif ctor == "u3":
            the, phi, lam = args[:3]
            for c, a in (("rz", lam), ("ry", the), ("rz", phi)):
                self.gate(c, (a, args[-1]), ctrl)
        elif ctor in ("x", "y"):
            m = [[0, 1], [1, 0]] if ctor == "x" else [[0, -i], [i, 0]]
            for q in bits:
                self.matrix(m, [q], ctrl)
        elif ctor in ("z", "s", "t"):
            f = {"z": -1, "s": i, "t": complex(h, h)}[ctor]
            for q in bits:
                self.diag([1, f], [q], ctrl)
        elif ctor == "swap":
            self.matrix([[1, 0, 0, 0], [0, 0, 1, 0], [0, 1, 0, 0], [0, 0, 0, 1]], bits, ctrl)
        elif ctor == "i_swap":
            self.matrix([[1, 0, 0, 0], [0, 0, i, 0], [0, i, 0, 0], [0, 0, 0, 1]], bits, ctrl)
        else:
            c, s = math.cos(args[0] / 2), math.sin(args[0] / 2)
            if ctor == "phi":
                self.diag([1, complex(math.cos(args[0]), math.sin(args[0]))], bits, ctrl)
            elif ctor == "rz":
                self.diag([complex(c, -s), complex(c, s)], bits, ctrl)
            elif ctor == "rzz":
                self.diag([complex(c, -s), complex(c, s), complex(c, s), complex(c, -s)], bits, ctrl)
            elif ctor == "rx":
                self.matrix([[c, -i * s], [-i * s, c]], bits, ctrl)
            elif ctor == "ry":
                self.matrix([[c, -s], [s, c]], bits, ctrl)
            elif ctor == "rxx":
                self.matrix([[c, 0, 0, -i * s], [0, c, -i * s, 0], [0, -i * s, c, 0], [-i * s, 0, 0, c]], bits, ctrl)
            elif ctor == "ryy":
                self.matrix([[c, 0, 0, i * s], [0, c, -i * s, 0], [0, -i * s, c, 0], [i * s, 0, 0, c]], bits, ctrl)
            else:
                raise ValueError(ctor)

    def weights(self):
        return self.psi.real ** 2 + self.psi.imag ** 2

    def measure(self, mask, u):
        """The drawn outcome on `mask`; the state keeps the amplitudes that agree with it, not rescaled."""
        w = torch.cumsum(self.weights(), 0)
        r = int(torch.searchsorted(w, u * w[-1], right=True))
        at = torch.arange(1 << self.n, device=self.dev)
        self.psi[((at ^ r) & mask) != 0] = 0
        return r & mask

    def reset(self, mask):
        at = torch.arange(1 << self.n, device=self.dev)
        self.psi[(at & mask) != 0] = 0
        norm = math.sqrt(float(self.weights().sum()))
        if norm <= 1e-15:
            self.psi.zero_()
            self.psi[0] = 1.0
        elif 1.0 - norm > 1e-9:
            self.psi /= norm


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    if kind in ("batch", "serve"):
        return {"outcomes": None, "total": np.ones(case["count"])}
    if kind in ("shots", "evolve"):
        return {"outcomes": None, "norm": 1.0}
    if kind == "program":
        part, first, second, branch, value, reset, draws = _program(case, seed)
        p = _Plain(n, 0)
        p.apply(part[0])
        got = p.measure(first, draws[0])
        packed = sum(1 << k for k, q in enumerate(q for q in range(n) if first >> q & 1) if got >> q & 1)
        if packed == value:
            p.apply(branch)
        p.apply(part[1])
        p.reset(reset)
        p.apply(part[2])
        p.measure(second, draws[1])
        w = p.weights()
        return {"class": None, "probabilities": (w / w.sum()).cpu().numpy()}
    p = _Plain(n, _basis(case, seed))
    for g in _gates(case, seed):
        p.apply(g)
    if kind == "loop":
        p.measure(0b100, float(_draws(seed, 1)[0]))
        return {"outcome": None, "weight": float(p.weights().sum())}
    if kind == "probs":
        return {"outcomes": None, "probabilities": p.weights().cpu().numpy()}
    return {"state": p.psi.cpu().numpy()}
