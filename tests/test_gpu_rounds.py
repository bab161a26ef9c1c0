"""Gate circuits on small states against the oracle, or beyond its sizes against
the gate-by-gate tile passes (explicit tile shapes).  Tolerance 1e-12 per
amplitude of a normalised state: a gate adds at most 4 roundings of 1.1e-16, so
1000 gates stay below 5e-13 on each side."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-12

PERM = [("X", False), ("cX", False), ("SWAP", False), ("acX", False)]
PHASE = [("Z", False), ("S", False), ("T", False), ("Rz", True), ("R", True), ("cZ", False), ("cR", True), ("cRz", True)]
DENSE = [("H", False), ("Y", False), ("V", False), ("Rx", True), ("Ry", True), ("cY", False), ("cV", False)]
KINDS = {"all": PERM + PHASE + DENSE, "moves": PERM, "phases": PHASE, "dense": DENSE}
TWO = {"cX", "acX", "cY", "cZ", "cV", "SWAP", "cR", "cRz"}


def _draw(rng, n, count, kinds, targets=None):
    out = []
    while len(out) < count:
        name, angle = kinds[int(rng.integers(len(kinds)))]
        t = int(rng.choice(targets)) if targets is not None else int(rng.integers(n))
        c = t
        if name in TWO:
            if n == 1:
                continue
            c = int((t + rng.integers(1, n)) % n)
        out.append((name, t, c, float(rng.uniform(-3.0, 3.0)) if angle else 0.0))
    return out


def _circuit(qf, gates):
    c = qf.Circuit()
    for name, t, ctl, a in gates:
        c.add(qf.gate(name, t, ctl, a) if a else qf.gate(name, t, ctl))
    return c


def _state(n, seed):
    r = np.random.default_rng(seed)
    v = r.normal(size=1 << n) + 1j * r.normal(size=1 << n)
    return v / np.linalg.norm(v)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8, 9, 11, 12, 13, 14])
@pytest.mark.parametrize("kind,count", [("all", 300), ("moves", 40), ("phases", 90), ("dense", 120), ("all", 9), ("all", 25)])
def test_random_gates_match_oracle(qf, oracle, n, kind, count):
    gates = _draw(np.random.default_rng(1000 * n + count), n, count, KINDS[kind])
    psi = _state(n, n)
    qc = qf.Computer(n)
    qc.set_coeff_vec(psi)
    qc.apply_circuit(_circuit(qf, gates))
    expect = oracle.apply_circuit(psi, n, [oracle.G(*g) for g in gates])
    assert np.max(np.abs(qc.get_coeff_vec() - expect)) < TOL


@pytest.mark.parametrize("n", [4, 12, 13])
def test_many_gates_on_one_qubit(qf, oracle, n):
    # rotations under changing conditions on one qubit (one flip, long lists)
    # and more phases between two of them than one round holds
    rng = np.random.default_rng(n)
    gates = _draw(rng, n, 80, [("cV", False), ("cY", False), ("Ry", True)], targets=[1])
    gates += _draw(rng, n, 60, PHASE) + [("H", 1, 1, 0.0)] + _draw(rng, n, 60, PHASE)
    psi = _state(n, n)
    qc = qf.Computer(n)
    qc.set_coeff_vec(psi)
    qc.apply_circuit(_circuit(qf, gates))
    expect = oracle.apply_circuit(psi, n, [oracle.G(*g) for g in gates])
    assert np.max(np.abs(qc.get_coeff_vec() - expect)) < TOL


@pytest.mark.parametrize("n", [17, 20, 22, 23])
@pytest.mark.parametrize("kind,count", [("all", 400), ("moves", 60), ("phases", 60)])
def test_multi_tile_states_match_tile_passes(qf, n, kind, count):
    gates = _draw(np.random.default_rng(n + count), n, count, KINDS[kind])
    psi = _state(n, n)
    saved = qf.get_tuning()
    got = []
    try:
        for shape in ((-1, -1, -1), (11, 4, 24)):
            qf.set_tuning(*shape)
            qc = qf.Computer(n)
            qc.set_coeff_vec(psi)
            qc.apply_circuit(_circuit(qf, gates))
            qc.apply_circuit(_circuit(qf, gates[:30]).adjoint())
            got.append(np.array(qc.get_coeff_vec()))
    finally:
        qf.set_tuning(*saved)
    assert np.max(np.abs(got[0] - got[1])) < TOL
