"""Gate circuits on states beyond 22 qubits: tile passes as rounds, in place,
against the gate-by-gate passes of an explicit tile shape.  Tolerance 1e-12 per
amplitude (at most 4 roundings of 1.1e-16 per gate, 300 gates)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-12
ONE = [("H", 0), ("X", 0), ("Y", 0), ("Z", 0), ("S", 0), ("T", 0), ("V", 0), ("Rx", 1), ("Ry", 1), ("Rz", 1)]
TWO = [("cX", 0), ("cY", 0), ("cZ", 0), ("cV", 0), ("SWAP", 0), ("cR", 1), ("cRz", 1)]
MOVES = [("X", 0), ("cX", 0), ("SWAP", 0)]


def _gates(rng, n, count, kinds):
    out = []
    for _ in range(count):
        name, angle = kinds[int(rng.integers(len(kinds)))]
        t = int(rng.integers(n))
        c = int((t + rng.integers(1, n)) % n) if (name, angle) in TWO else t
        out.append((name, t, c, float(rng.uniform(-3.0, 3.0)) if angle else 0.0))
    return out


@pytest.mark.parametrize("n", [23, 24])
@pytest.mark.parametrize("kind,count", [("all", 300), ("moves", 40), ("few", 3), ("with_a", 30)])
def test_large_states_match_tile_passes(qf, gpu, n, kind, count):
    rng = np.random.default_rng(n + count)
    gates = _gates(rng, n, count, MOVES if kind == "moves" else ONE + TWO)
    if kind == "with_a":  # a two-qubit gate that has no rounds
        gates.insert(11, ("A", 3, n - 2, 1.1))
    c = qf.Circuit()
    for name, t, ctl, a in gates:
        c.add(qf.gate(name, t, ctl, a) if a else qf.gate(name, t, ctl))
    r = np.random.default_rng(n)
    psi = r.normal(size=1 << n) + 1j * r.normal(size=1 << n)
    psi /= np.linalg.norm(psi)
    saved = qf.get_tuning()
    got = []
    try:
        for shape in ((-1, -1, -1), (11, 4, 24)):
            qf.set_tuning(*shape)
            qc = qf.Computer(n)
            qc.set_coeff_vec(psi)
            qc.apply_circuit(c)
            got.append(np.array(qc.get_coeff_vec()))
    finally:
        qf.set_tuning(*saved)
    assert np.max(np.abs(got[0] - got[1])) < TOL
