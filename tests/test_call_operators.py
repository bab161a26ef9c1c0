"""Operators of a call as any iterable: the forms whose items live only while
they are read (a generator, a map, a sequence that makes its items on access)
give the terms that a list gives."""

import pytest

from host_runtime import on_host  # noqa: F401

FORMS = """
class Lazy:
    def __init__(self, make, n): self.make, self.n = make, n
    def __len__(self): return self.n
    def __getitem__(self, i):
        if not 0 <= i < self.n: raise IndexError(i)
        return self.make(i)
import collections.abc
collections.abc.Sequence.register(Lazy)
def forms(make, n):
    yield [make(i) for i in range(n)]
    yield tuple(make(i) for i in range(n))
    yield (make(i) for i in range(n))
    yield map(make, range(n))
    yield Lazy(make, n)
    yield {i: make(i) for i in range(n)}.values()
"""

SETUP = """
import gc
ref = qf.system.hamiltonians.hf_occupation(3, 2, 1)
h, g = qf.synthetic_integrals(3, 5)
hmap = qf.HamiltonianMap(3)
inputs = hmap.pack(0.3, h, g)
pool = qf.SQOpPool()
pool.set_orb_spaces(ref)
pool.fill_pool("SD")
tops = list(range(len(pool)))
tpl = qf.compile_ucc_template(6, ref, hmap, pool, tops)
prog = qf.compile_ucc_program(6, ref, hmap.operator(inputs), pool, tops)
t = [0.1] * len(tops)
ops = [o for _, o in pool.terms()]
make = lambda i: ops[i % len(ops)].jw_transform()
a, b = qf.Computer(6), qf.Computer(6)
calls = {
    "template": lambda x: tpl.pool_gradients(t, x, inputs=inputs),
    "program": lambda x: prog.pool_gradients(t, x),
    "cross": lambda x: qf.cross_expectations(a, b, x),
}
"""


@pytest.mark.parametrize("call", ["template", "program", "cross"])
def test_operators_of_any_iterable(on_host, call):  # noqa: F811
    # the entry points refuse what they do not understand (a term outside the
    # register, a gate that is no Pauli letter) while compiling the operators:
    # with freed operators they crash or refuse these
    out = on_host(FORMS + SETUP + f"""
call = calls[{call!r}]
n = 3 * len(ops)
want = len(call([make(i) for i in range(n)]))
for form in forms(make, n):
    host.host_forget()
    assert len(call(form)) == want == n
def bad(i):
    if i != n - 1: return make(i)
    c = qf.Circuit(); c.add(qf.gate("H", 0)); o = qf.QubitOperator(); o.add_term(1.0, c)
    return o
for form in forms(bad, n):
    try: call(form)
    except ValueError as e: assert "Pauli sums" in str(e)
    else: raise SystemExit("accepted")
for wrong in ("x", None, 1, [1], [None], (None for _ in range(2))):
    try: call(wrong)
    except TypeError: pass
    else: raise SystemExit("accepted " + repr(wrong))
print("ok")
""")
    assert out.strip() == "ok"


@pytest.mark.gpu
@pytest.mark.parametrize("call", ["template", "program", "cross"])
def test_values_of_any_iterable(qf, call):
    ns = {"qf": qf}
    exec(FORMS + SETUP, ns)
    a, b = ns["a"], ns["b"]
    ns["tpl"].prepare(ns["t"], a)
    ns["prog"].prepare([0.2] * len(ns["t"]), b)
    n = 3 * len(ns["ops"])
    values = [list(ns["calls"][call](form)) for form in ns["forms"](ns["make"], n)]
    assert any(abs(v) > 1e-6 for v in values[0])
    assert all(v == values[0] for v in values)
