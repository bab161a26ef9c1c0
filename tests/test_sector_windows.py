"""Partial sums of the sector's reverse sweep: kept for a window of passes, so
their memory is bounded on large sectors and for long ansaetze, energy calls
allocate none, and no budget is refused for them."""

import pytest

from host_runtime import on_host  # noqa: F401

SETUP = """
def template(norb, ne, layers, pick):
    n = 2 * norb
    ref = qf.system.hamiltonians.hf_occupation(norb, ne, ne)
    pool = qf.SQOpPool()
    pool.set_orb_spaces(ref)
    pool.fill_pool("SD")
    tops = [k for k in range(len(pool)) if k in pick] if pick else list(range(len(pool)))
    gens, idx, scale = qf.ucc_generators(pool, tops)
    H = qf.QubitOperator()
    for q in range(n):
        c = qf.Circuit()
        c.add(qf.gate("Z", q))
        H.add_op(qf.build_operator(f"{0.1 * (q + 1)}, Z_{q}"))
    for q in range(0, n - 2, 2):
        H.add_op(qf.build_operator(f"{0.05 * (q + 1)}, X_{q} Z_{q + 1} X_{q + 2}; {0.05 * (q + 1)}, Y_{q} Z_{q + 1} Y_{q + 2}"))
    ridx = qf.ref_to_basis_idx(ref)
    return [n, ridx, gens * layers, idx * layers, [s / layers for s in scale] * layers, len(tops), H]
"""


@pytest.mark.parametrize("norb,ne,layers,pick", [(12, 6, 1, None), (16, 8, 1750, range(8))])
def test_memory_is_bounded(on_host, norb, ne, layers, pick):  # noqa: F811
    # 16 orbitals: 14000 generators over 161 thousand tiles, more partial sums
    # than a 32-bit number counts
    out = on_host(SETUP + f"""
args = template({norb}, {ne}, {layers}, {list(pick) if pick else None})
tpl = qf.SectorTemplate(*args)
t = [0.1] * tpl.nparam
state = 16 * tpl.dim  # complex amplitudes
base = host.host_used()
tpl.energy(t, [])
assert host.host_used() - base <= state, host.host_used() - base
base = host.host_used()
host.host_forget()
tpl.gradient(t, [])
took = host.host_used() - base
assert took <= 2 * state, took
sweeps = [s for name, s in launches() if "k_sec_tile" in name and "Li2E" in name]
tiles, waves = sweeps[0][0], sweeps[0][3] // 64
# every pass's sums (eight bytes per tile, wave and generator) fit what was allocated
gens = len(args[2])
assert len(sweeps) * took >= 8 * tiles * waves * gens, (len(sweeps), tiles, gens, took)
print("ok")
""", timeout=300)
    assert out.strip() == "ok"


def test_budget_of_a_gradient_request(on_host):  # noqa: F811
    # two states, (cos, sin) per generator and the arguments of a real template
    out = on_host(SETUP + """
args = template(9, 4, 4, None)
tpl = qf.SectorTemplate(*args)
t = [0.1] * tpl.nparam
need = 32 * tpl.dim + 16 * len(args[2]) + 8 * (tpl.nparam + 2 * len(args[2])) + (64 << 10)
eng = qf.BatchEngine(3 * need, 4)
ids = [eng.submit(tpl, t, [], True) for _ in range(6)]
done = []
while len(done) < 6: done += eng.step(6)
try: qf.BatchEngine(3 * 8 * tpl.dim, 4).submit(tpl, t, [], True)
except Exception as e: assert "budget" in str(e)
else: raise SystemExit("accepted")
print("ok")
""")
    assert out.strip() == "ok"


def test_audit_takes_its_buffers_itself(on_host):  # noqa: F811
    out = on_host(SETUP + """
tpl = qf.SectorTemplate(*template(9, 4, 1, None))
tpl.gradient([0.1] * tpl.nparam, [])
base = host.host_used()
try: tpl.graph_audit(True)  # nothing is captured without a device
except RuntimeError: pass
assert host.host_used() - base >= 8 * tpl.dim // 256
print("ok")
""")
    assert out.strip() == "ok"


LONG = (9, 4, 30, None)  # 18 qubits, 16800 generators


def test_long_ansatz_takes_several_windows(on_host):  # noqa: F811
    out = on_host(SETUP + f"""
args = template(*{LONG})
tpl = qf.SectorTemplate(*args)
host.host_forget()
tpl.gradient([0.1] * tpl.nparam, [])
print(len(args[2]), sum("k_sec_tile_sum" in name for name, _ in launches()))
""")
    gens, sums = map(int, out.split())
    assert gens == 16800 and sums >= 3


@pytest.mark.gpu
def test_gradient_over_several_windows(qf):
    """The template's windows against the full-space program, alone and in a
    launch with a request that has one window."""
    import numpy as np

    ns = {"qf": qf}
    exec(SETUP, ns)
    args = ns["template"](*LONG)
    tpl, prog = qf.SectorTemplate(*args), qf.UCCProgram(*args)
    t = list(np.random.default_rng(7).normal(0.0, 0.1, tpl.nparam))
    e, g = tpl.gradient(t, [])
    e_p, g_p = prog.gradient(t)
    assert abs(e - e_p) < 1e-10
    assert np.max(np.abs(np.array(g) - np.array(g_p))) < 1e-10
    small = qf.SectorTemplate(*ns["template"](9, 4, 1, None))
    eng = qf.BatchEngine(8 << 30, 8)
    ids = [eng.submit(x, t, [], True) for x in (tpl, small, tpl)]
    done = dict()
    while len(done) < 3:
        done.update(eng.step(8))
    for i in (ids[0], ids[2]):
        assert abs(done[i] - e) < 1e-12
        assert np.max(np.abs(np.array(eng.take_gradient(i, tpl.nparam)) - np.array(g))) < 1e-12
    assert np.max(np.abs(np.array(eng.take_gradient(ids[1], tpl.nparam)) - np.array(small.gradient(t, [])[1]))) < 1e-12
