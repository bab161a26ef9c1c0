"""Runs of Pauli exponentials whose flip masks span more dimensions than a
register orbit holds: against the oracle, or beyond its sizes against lane
orbits (six dimensions).  Tolerance 1e-12 per amplitude of a normalised state:
at most 4 roundings of 1.1e-16 per exponential, 120 of them."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-12


def _sequence(n, count, seed):
    # random strings, repeated ones, products of earlier flips, pure Z strings
    # and strings confined to the lowest qubits (inside every tile's runs)
    r = np.random.default_rng(seed)
    seq = []
    for _ in range(count):
        kind = int(r.integers(7))
        if kind == 0 and seq:
            term = seq[int(r.integers(len(seq)))][1]
        elif kind == 1:
            term = [("Z", int(q)) for q in sorted(r.choice(n, size=3, replace=False))]
        elif kind == 2:
            term = [("XY"[int(r.integers(2))], q) for q in range(int(r.integers(1, 4)))]
        else:
            qs = sorted(int(v) for v in r.choice(n, size=int(r.integers(2, 9)), replace=False))
            term = [("XYZ"[int(r.integers(3))], q) for q in qs]
        seq.append((float(r.normal()), term))
    return seq


def _state(n):
    r = np.random.default_rng(n)
    v = r.normal(size=1 << n) + 1j * r.normal(size=1 << n)
    return v / np.linalg.norm(v)


def _run(qf, n, seq, psi):
    from qforte_amd.engine import workloads as W

    U, phase = qf.trotterize(W.exp_operator(qf, seq))
    assert phase == 1.0
    qc = qf.Computer(n)
    qc.set_coeff_vec(psi)
    qf.reset_counters()
    qc.apply_circuit(U)
    passes = qf.get_counters()["fused_passes"]
    return np.array(qc.get_coeff_vec()), passes


@pytest.mark.parametrize("n", [12, 13, 14, 16])
@pytest.mark.parametrize("count", [12, 90])
def test_wide_passes_match_oracle(qf, oracle, n, count):
    seq = _sequence(n, count, n + count)
    psi = _state(n)
    got, _ = _run(qf, n, seq, psi)
    expect = psi
    for theta, term in seq:
        expect = oracle.exp_pauli(expect, -1j * theta, term)
    assert np.max(np.abs(got - expect)) < TOL


@pytest.mark.parametrize("n", [19, 22, 24])
def test_wide_passes_match_lane_orbits(qf, gpu, n):
    seq = _sequence(n, 120, n)
    psi = _state(n)
    wide, fewer = _run(qf, n, seq, psi)
    saved = qf.get_pass_tuning()
    try:
        qf.set_pass_tuning(6)
        lanes, more = _run(qf, n, seq, psi)
    finally:
        qf.set_pass_tuning(saved)
    assert fewer < more
    assert np.max(np.abs(wide - lanes)) < TOL
