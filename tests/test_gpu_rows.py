"""Hamiltonian rows of the sector engine against the full-space program (1e-10
Ha and 1e-10 on gradients, as the other sector tests) at the forms where they
can go wrong: Hamiltonians that the rows take in part or not at all, one-sided
fillings, a beta space wider than one workgroup, a single determinant pair."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _random_operator(qf, n, seed, count, hopping):
    """Real-coefficient Pauli sum: Z strings, number-conserving XX + YY pairs
    over random qubits (any Z string between them) and random strings with an
    even number of Y."""
    rng = np.random.default_rng(seed)
    op = qf.QubitOperator()

    def add(c, letters):
        op.add(c, qf.build_circuit(" ".join(f"{p}_{q}" for q, p in sorted(letters.items()))))

    for _ in range(count):
        qubits = rng.choice(n, size=int(rng.integers(1, 5)), replace=False)
        add(float(rng.normal()), {int(q): "Z" for q in qubits})
    for _ in range(hopping):
        spin = int(rng.integers(2))
        p, q = (int(v) for v in 2 * rng.choice(n // 2, size=2, replace=False) + spin)
        rest = {int(r): "Z" for r in rng.choice(n, size=int(rng.integers(0, n)), replace=False) if r not in (p, q)}
        c = float(rng.normal())
        add(c, {p: "X", q: "X", **rest})
        add(c, {p: "Y", q: "Y", **rest})
    for _ in range(count):
        letters = {int(q): "XYZ"[int(rng.integers(3))] for q in rng.choice(n, size=int(rng.integers(2, min(n, 7))), replace=False)}
        if sum(p == "Y" for p in letters.values()) % 2 == 0:
            add(float(rng.normal()), letters)
    op.simplify()
    return op


def _compare(qf, n, na, nb, hamiltonian, inputs, operator, step=1):
    ref = qf.system.hamiltonians.hf_occupation(n // 2, na, nb)
    pool = qf.SQOpPool()
    pool.set_orb_spaces(ref)
    pool.fill_pool("SD")
    tops = list(range(0, len(pool), step))
    tpl = qf.compile_ucc_template(n, ref, hamiltonian, pool, tops)
    prog = qf.compile_ucc_program(n, ref, operator, pool, tops)
    t = np.random.default_rng(n + na).normal(0.0, 0.2, len(tops)).tolist()
    e_p, g_p = prog.gradient(t)
    args = (t,) if inputs is None else (t, inputs)
    e, g = tpl.gradient(*args)
    scale = max(1.0, abs(e_p))
    assert abs(tpl.energy(*args) - e_p) < 1e-10 * scale
    assert abs(e - e_p) < 1e-10 * scale
    assert np.max(np.abs(np.array(g) - np.array(g_p))) < 1e-10 * scale


@pytest.mark.parametrize("n,na,nb", [(4, 1, 1), (8, 2, 2), (10, 4, 1), (12, 3, 3)])
@pytest.mark.parametrize("seed", [1, 2])
def test_general_hamiltonians(qf, n, na, nb, seed):
    op = _random_operator(qf, n, 10 * n + seed, 40, 60)
    _compare(qf, n, na, nb, op, None, op)


@pytest.mark.parametrize("n,na,nb,step", [(4, 1, 1, 1), (6, 2, 1, 1), (14, 1, 6, 3), (14, 6, 1, 3), (16, 4, 4, 11), (22, 1, 5, 40)])
def test_molecular_hamiltonians(qf, n, na, nb, step):
    h, g = qf.synthetic_integrals(n // 2, n + nb)
    hmap = qf.HamiltonianMap(n // 2)
    inputs = hmap.pack(0.7, h, g)
    _compare(qf, n, na, nb, hmap, inputs, hmap.operator(inputs), step)


def test_rows_and_term_loops_share_a_launch(qf):
    """Templates whose Hamiltonian the rows take whole, in part and not at
    all, served together: each as alone."""
    n, ref = 8, [1, 1, 1, 1, 0, 0, 0, 0]
    pool = qf.SQOpPool()
    pool.set_orb_spaces(ref)
    pool.fill_pool("SD")
    tops = list(range(len(pool)))
    h, g = qf.synthetic_integrals(4, 5)
    hmap = qf.HamiltonianMap(4)
    inputs = hmap.pack(0.0, h, g)
    odd = qf.QubitOperator()  # X X on one spin without its Y Y: no sector flip keeps to its strings
    for k, c in enumerate((0.3, -0.4, 0.5)):
        odd.add(c, qf.build_circuit(f"X_{k} X_{k + 1} Z_7 X_{k + 2} X_{k + 3}"))
    cases = [(qf.compile_ucc_template(n, ref, hmap, pool, tops), inputs)]
    cases += [(qf.compile_ucc_template(n, ref, op, pool, tops), []) for op in (_random_operator(qf, n, 3, 20, 30), odd)]
    t = np.random.default_rng(4).normal(0.0, 0.2, len(tops)).tolist()
    eng = qf.ServingEngine(hbm_budget_bytes=1 << 30, max_active=64)
    ids = [(eng.submit(tpl, t, inp), eng.submit(tpl, t, inp, gradient=True)) for tpl, inp in cases]
    eng.drain()
    for (e_id, g_id), (tpl, inp) in zip(ids, cases):
        e, gr = tpl.gradient(t, inp)
        assert abs(eng.results[e_id] - tpl.energy(t, inp)) < 1e-12
        assert abs(eng.results[g_id] - e) < 1e-12
        assert np.max(np.abs(np.array(eng.gradients[g_id]) - np.array(gr))) < 1e-12
