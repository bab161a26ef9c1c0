"""The Pauli form that a circuit keeps while gates are appended, against the
product of its gates' matrices on three qubits (exact: entries 0, +-1, +-i)."""

import numpy as np
import pytest

_M = {
    "I": np.eye(2, dtype=complex),
    "X": np.array([[0, 1], [1, 0]], dtype=complex),
    "Y": np.array([[0, -1j], [1j, 0]]),
    "Z": np.diag([1.0 + 0j, -1.0]),
}
_N = 3


def _matrix(letters):
    u = np.eye(2**_N, dtype=complex)
    for p, q in letters:
        m = np.eye(1, dtype=complex)
        for k in reversed(range(_N)):
            m = np.kron(m, _M[p] if k == q else _M["I"])
        u = m @ u
    return u


def _from_masks(x, z, phase):
    u = np.zeros((2**_N, 2**_N), dtype=complex)
    for j in range(2**_N):
        u[j ^ x, j] = phase * (-1) ** bin(j & z).count("1")
    return u


def _circuit(qf, letters):
    c = qf.Circuit()
    for p, q in letters:
        c.add(qf.gate(p, q))
    return c


@pytest.mark.parametrize("how", ["append", "join", "insert", "remove", "replace", "swap", "insert_circuit", "remove_gates", "adjoint", "canonical", "grown"])
@pytest.mark.parametrize("seed", [0, 1, 2])
def test_form_follows_the_gates(qf, how, seed):
    rng = np.random.default_rng(seed)

    def draw(k):
        return [("IXYZ"[int(rng.integers(4))], int(rng.integers(_N))) for _ in range(k)]

    a, b = draw(7), draw(5)
    c = _circuit(qf, a)
    scale = 1.0
    if how == "append":
        pass
    elif how == "join":
        c.add(_circuit(qf, b))
        a = a + b
    elif how == "insert":
        c.insert_gate(2, qf.gate(*b[0]))
        a = a[:2] + b[:1] + a[2:]
    elif how == "remove":
        c.remove_gate(3)
        a = a[:3] + a[4:]
    elif how == "replace":
        c.replace_gate(3, qf.gate(*b[0]))
        a = a[:3] + b[:1] + a[4:]
    elif how == "swap":
        c.swap_gates(1, 4)
        a[1], a[4] = a[4], a[1]
    elif how == "insert_circuit":
        c.insert_circuit(2, _circuit(qf, b))
        a = a[:2] + b + a[2:]
    elif how == "remove_gates":
        c.remove_gates(1, 4)
        a = a[:1] + a[4:]
    elif how == "adjoint":
        c = c.adjoint()
        a = a[::-1]
    elif how == "canonical":
        a = [g for g in a if g[0] != "I"]  # refuses I
        c = _circuit(qf, a)
        scale = c.canonicalize_pauli_circuit()
        a = a[::-1]  # its coefficient is that of the product in written order
    elif how == "grown":  # append after a mutation that drops the form
        c.swap_gates(0, 5)
        a[0], a[5] = a[5], a[0]
        c.add(qf.gate(*b[0]))
        c.add(_circuit(qf, b[1:]))
        a = a + b
    assert np.array_equal(scale * _from_masks(*qf._core.pauli_masks(c)), _matrix(a))


def test_other_gates_have_no_form(qf):
    c = _circuit(qf, [("X", 0)])
    c.add(qf.gate("Rz", 1, 1, 0.3))
    assert qf._core.pauli_masks(c) is None
    c.set_parameters([0.4])
    assert qf._core.pauli_masks(c) is None
    c.set_parameter(1, 0.5)
    assert qf._core.pauli_masks(c) is None
    c.remove_gate(1)
    assert qf._core.pauli_masks(c) == (1, 0, 1)
    d = _circuit(qf, [("Z", 0)])
    d.add(qf.gate("H", 0))
    c.add(d)
    assert qf._core.pauli_masks(c) is None
    assert qf._core.pauli_masks(qf.Circuit()) == (0, 0, 1)
