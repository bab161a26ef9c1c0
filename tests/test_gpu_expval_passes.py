"""Expectation passes where their shape changes: passes padded to full width
(Z strings alone, one X mask, several diagonal operators in one call), all
passes in one launch (16 to 23 qubits) and one launch per pass from 24 on;
the group kernel below 16 qubits and the sliced operator application.
Oracle: the same sums in numpy on the downloaded state, 1e-12 relative to the
sum of the coefficients' magnitudes (each value is a mean of +-1)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _parity(v):
    for s in (16, 8, 4, 2, 1):
        v = v ^ (v >> s)
    return v & 1


def _value(psi, terms):
    index = np.arange(len(psi), dtype=np.uint32)
    total = 0.0
    for c, string in terms:
        x = sum(1 << q for p, q in string if p != "Z")
        z = sum(1 << q for p, q in string if p != "X")
        src = index ^ np.uint32(x)
        sign = 1.0 - 2.0 * _parity(src & np.uint32(z))
        total += c * (1j ** sum(p == "Y" for p, _ in string)) * np.vdot(psi, sign * psi[src])
    return total


@pytest.mark.parametrize("n", [16, 20, 21, 23, 24])
def test_padded_and_diagonal_passes(qf, n):
    from qforte_amd.engine import workloads as W

    qc = qf.Computer(n)
    qc.apply_circuit(W.to_circuit(qf, W.brickwork_layers(n, 2, seed=n)))
    psi = np.asarray(qc.get_coeff_vec())
    top = n - 1
    operators = [
        [(0.5, [("Z", 0)]), (-1.5, [("Z", top)]), (0.25, [("Z", 3), ("Z", 7), ("Z", top)])],
        [(0.7, [("X", 0), ("Y", 1)]), (0.3, [("Y", 0), ("X", 1)])],
        [(1.0, [("X", top)]), (0.5, [("Y", top), ("Z", 6)]), (0.4, [("Z", 8)])],
    ]
    operators += [[(1.0, [("Z", q)])] for q in range(0, n, 1)]
    pool = qf.QubitOpPool()
    for terms in operators:
        pool.add(1.0, W.to_operator(qf, terms))
    got = qc.direct_oppl_exp_val(pool)
    for k, terms in enumerate(operators[:8]):
        scale = sum(abs(c) for c, _ in terms)
        assert abs(got[k] - _value(psi, terms)) < 1e-12 * scale, (n, k)
        assert abs(qc.direct_op_exp_val(W.to_operator(qf, terms)) - got[k]) < 1e-12 * scale, (n, k)
    assert abs(got[-1] - _value(psi, operators[-1])) < 1e-12


def _random_terms(n, count, seed, imaginary):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(count):
        qubits = rng.choice(n, size=int(rng.integers(1, n + 1)), replace=False)
        c = float(rng.normal()) + (1j * float(rng.normal()) if imaginary else 0.0)
        out.append((c, [("XYZ"[int(rng.integers(3))], int(q)) for q in sorted(qubits)]))
    return out


@pytest.mark.parametrize("n,count", [(1, 3), (2, 10), (5, 60), (9, 300), (12, 700), (15, 40), (17, 90)])
@pytest.mark.parametrize("imaginary", [False, True])
def test_expectations_and_application_against_numpy(qf, n, count, imaginary):
    """More terms per X mask than one staged block, odd counts of pairs, real
    and complex coefficients; <bra|O|ket> and O|psi> on the same terms."""
    from qforte_amd.engine import workloads as W

    rng = np.random.default_rng(n)
    states = []
    for _ in range(2):
        v = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
        states.append(v / np.linalg.norm(v))
    bra, ket = qf.Computer(n), qf.Computer(n)
    bra.set_coeff_vec(states[0])
    ket.set_coeff_vec(states[1])
    terms = _random_terms(n, count, n + count, imaginary)
    if n == 9:
        terms += [(0.1 + 0.01 * k, [("X", 0)] + [("Z", q) for q in range(1, 9) if (k >> (q - 1)) & 1]) for k in range(256)]
        terms += [(0.2, [("X", 0), ("Z", 8)]), (0.3, [("Y", 0)])] * 2
    op = W.to_operator(qf, terms)
    scale = sum(abs(c) for c, _ in terms)
    index = np.arange(1 << n, dtype=np.uint32)
    out = np.zeros(1 << n, complex)
    for c, string in terms:
        x = sum(1 << q for p, q in string if p != "Z")
        z = sum(1 << q for p, q in string if p != "X")
        src = index ^ np.uint32(x)
        out += c * (1j ** sum(p == "Y" for p, _ in string)) * (1.0 - 2.0 * _parity(src & np.uint32(z))) * states[1][src]
    assert abs(ket.direct_op_exp_val(op) - np.vdot(states[1], out)) < 1e-12 * scale
    assert abs(qf.cross_expectations(bra, ket, [op])[0] - np.vdot(states[0], out)) < 1e-12 * scale
    ket.apply_operator(op)
    assert np.max(np.abs(np.asarray(ket.get_coeff_vec()) - out)) < 1e-12 * scale
