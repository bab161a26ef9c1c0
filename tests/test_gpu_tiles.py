"""Component tiles of the sector engine: ansatz, inverse and reverse sweep
against the full-space compiled program (1e-10 Ha for energies and gradients,
1e-11 for residual amplitudes: the tolerances of the other sector tests) where
the tiling can go wrong: one tile for the whole sector, many, generators of
several runs, generators whose components exceed a tile, programs longer than
one staged chunk of records, no generator at all."""

import random

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "n,na,nb,pool_type,count,combo",
    [
        (4, 1, 1, "SD", 0, 0),  # the smallest sector
        (8, 2, 2, "SD", -1, 0),  # no generator
        (8, 2, 2, "sa_SD", 0, 0),  # several runs per generator
        (12, 3, 3, "sa_SD", 0, 0),  # more than 128 records in one pass
        (14, 4, 3, "SD", 40, 0),  # random order, several segments
        (14, 4, 4, "GSD", 30, 20),  # a generator of 20 excitations: components beyond a tile
        (16, 1, 7, "SD", 0, 0),  # few alpha strings, a tile of one alpha block
    ],
)
def test_tiles_match_the_full_space_program(qf, n, na, nb, pool_type, count, combo):
    ref = qf.system.hamiltonians.hf_occupation(n // 2, na, nb)
    pool = qf.SQOpPool()
    pool.set_orb_spaces(ref)
    pool.fill_pool(pool_type)
    rng = random.Random(n * 100 + combo)
    tops = list(range(len(pool))) if count == 0 else [rng.randrange(len(pool)) for _ in range(max(count, 0))]
    gens, idx, scale = qf.ucc_generators(pool, tops, pool_type)
    if combo:
        wide = qf.QubitOperator()
        for g in gens[:combo]:
            wide.add_op(g)
        gens, idx, scale = list(gens) + [wide], list(idx) + [len(tops)], list(scale) + [0.5]
    nparam = max(idx) + 1 if idx else 1
    h, g = qf.synthetic_integrals(n // 2, n)
    hmap = qf.HamiltonianMap(n // 2)
    inputs = hmap.pack(0.1, h, g)
    ridx = qf.ref_to_basis_idx(ref)
    prog = qf.UCCProgram(n, ridx, gens, idx, scale, nparam, hmap.operator(inputs))
    tpl = qf.SectorTemplate(n, ridx, gens, idx, scale, nparam, hmap)
    t = np.random.default_rng(n + nb).normal(0.0, 0.1, nparam).tolist()
    assert abs(tpl.energy(t, inputs) - prog.energy(t)) < 1e-10
    e, gr = tpl.gradient(t, inputs)
    e_p, gr_p = prog.gradient(t)
    assert abs(e - e_p) < 1e-10
    assert np.max(np.abs(np.array(gr) - np.array(gr_p))) < 1e-10
    state = qf.Computer(n)
    tpl.prepare(t, state)
    amps = np.abs(np.asarray(state.get_coeff_vec()))
    sel = [int(ridx)] + [int(i) for i in np.argsort(-amps)[:8] if amps[i] > 0.0]
    r, r_p = np.asarray(tpl.residuals(t, sel, inputs)), np.asarray(prog.residuals(t, sel))
    assert np.max(np.abs(r - r_p)) < 1e-11
    # the same request served in a launch with another size
    other = qf.compile_ucc_template(8, [1, 1, 1, 1, 0, 0, 0, 0], qf.HamiltonianMap(4), _sd(qf), list(range(26)))
    h4, g4 = qf.synthetic_integrals(4, 3)
    inputs4 = qf.HamiltonianMap(4).pack(0.0, h4, g4)
    eng = qf.ServingEngine(hbm_budget_bytes=1 << 30, max_active=64)
    ids = [eng.submit(tpl, t, inputs, gradient=True), eng.submit(other, [0.05] * 26, inputs4, gradient=True),
           eng.submit(tpl, t, inputs, gradient=True)]
    eng.drain()
    assert abs(eng.results[ids[0]] - e) < 1e-12 and eng.results[ids[0]] == eng.results[ids[2]]
    assert np.max(np.abs(np.array(eng.gradients[ids[0]]) - np.array(gr))) < 1e-12
    e4, g4r = other.gradient([0.05] * 26, inputs4)
    assert abs(eng.results[ids[1]] - e4) < 1e-12
    assert np.max(np.abs(np.array(eng.gradients[ids[1]]) - np.array(g4r))) < 1e-12


def _sd(qf):
    pool = qf.SQOpPool()
    pool.set_orb_spaces([1, 1, 1, 1, 0, 0, 0, 0])
    pool.fill_pool("SD")
    return pool


def test_complex_generators_on_the_sector(qf):
    """Imaginary hopping, i (a+_p a_q + a+_q a_p), makes the state complex:
    the template keeps complex amplitudes, beside a real template in one
    serving queue."""
    n, ref = 8, [1, 1, 1, 1, 0, 0, 0, 0]
    gens = []
    for p, q in ((0, 4), (1, 5), (2, 6), (0, 2)):
        string = " ".join(f"Z_{k}" for k in range(p + 1, q))
        op = qf.QubitOperator()
        op.add(0.5j, qf.build_circuit(f"X_{p} {string} X_{q}"))
        op.add(0.5j, qf.build_circuit(f"Y_{p} {string} Y_{q}"))
        gens.append(op)
    hmap = qf.HamiltonianMap(4)
    h, g = qf.synthetic_integrals(4, 12)
    inputs = hmap.pack(0.2, h, g)
    ridx = qf.ref_to_basis_idx(ref)
    args = (n, ridx, gens, [0, 1, 2, 3], [1.0] * 4, 4)
    prog = qf.UCCProgram(*args, hmap.operator(inputs))
    tpl = qf.SectorTemplate(*args, hmap)
    t = [0.3, -0.2, 0.4, 0.25]
    e, gr = tpl.gradient(t, inputs)
    e_p, gr_p = prog.gradient(t)
    assert abs(e - e_p) < 1e-10 and abs(tpl.energy(t, inputs) - e_p) < 1e-10
    assert np.max(np.abs(np.array(gr) - np.array(gr_p))) < 1e-10
    a, b = qf.Computer(n), qf.Computer(n)
    prog.prepare(t, a)
    tpl.prepare(t, b)
    amps = np.asarray(a.get_coeff_vec())
    assert np.abs(amps.imag).max() > 1e-2
    assert np.max(np.abs(amps - np.asarray(b.get_coeff_vec()))) < 1e-12
    sel = [int(i) for i in np.argsort(-np.abs(amps))[:6]]
    assert np.max(np.abs(np.asarray(tpl.residuals(t, sel, inputs)) - np.asarray(prog.residuals(t, sel)))) < 1e-11
    real = qf.compile_ucc_template(n, ref, hmap, _sd(qf), list(range(26)))
    eng = qf.ServingEngine(hbm_budget_bytes=1 << 30, max_active=64)
    ids = [eng.submit(x, y, inputs, gradient=True) for x, y in ((tpl, t), (real, [0.05] * 26), (tpl, t), (real, [0.05] * 26))]
    eng.drain()
    assert abs(eng.results[ids[0]] - e) < 1e-12 and eng.results[ids[0]] == eng.results[ids[2]]
    assert np.max(np.abs(np.array(eng.gradients[ids[2]]) - np.array(gr))) < 1e-12
    assert abs(eng.results[ids[3]] - real.energy([0.05] * 26, inputs)) < 1e-12
