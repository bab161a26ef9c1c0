"""Arguments of the compiled UCC calls: the sequence forms they take, and pool
tables of every size (one operator, none, more than the kept workspace holds).
Repeated operators give the same sums in the same order: compared exactly."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _template(qf):
    n = 6
    ref = qf.system.hamiltonians.hf_occupation(3, 2, 1)
    h, g = qf.synthetic_integrals(3, 5)
    hmap = qf.HamiltonianMap(3)
    inputs = hmap.pack(0.3, h, g)
    pool = qf.SQOpPool()
    pool.set_orb_spaces(ref)
    pool.fill_pool("SD")
    tops = list(range(len(pool)))
    t = np.random.default_rng(3).normal(0.0, 0.3, len(tops))
    ops = [o.jw_transform() for _, o in pool.terms()]
    return qf.compile_ucc_template(n, ref, hmap, pool, tops), qf.compile_ucc_program(n, ref, hmap.operator(inputs), pool, tops), t, inputs, ops


def test_sequence_forms(qf):
    tpl, prog, t, inputs, _ = _template(qf)
    e = tpl.energy(t.tolist(), inputs)
    e_p = prog.energy(t.tolist())
    for form in (t, tuple(t.tolist()), list(t)):
        assert tpl.energy(form, inputs) == e
        assert prog.energy(form) == e_p
    assert tpl.energy(t.tolist(), tuple(inputs)) == e
    z = len(t) * [0.0]
    assert tpl.energy(len(t) * [0], inputs) == tpl.energy(z, inputs)
    mixed = [0] + z[1:]
    assert tpl.energy(mixed, inputs) == tpl.energy(z, inputs)
    for bad in ("x", None, len(t) * ["a"], 1.0):
        with pytest.raises(TypeError):
            tpl.energy(bad, inputs)
    with pytest.raises(Exception):
        tpl.energy(z[1:], inputs)


@pytest.mark.parametrize("copies", [0, 1, 65, 60000])
def test_pool_tables_of_any_size(qf, copies):
    tpl, prog, t, inputs, ops = _template(qf)
    one = tpl.pool_gradients(t.tolist(), ops, inputs=inputs)
    many = tpl.pool_gradients(t.tolist(), ops * copies, inputs=inputs)
    assert many == one * copies
    assert np.max(np.abs(np.array(one) - np.array(prog.pool_gradients(t.tolist(), ops)))) < 1e-10
