"""Launches of the serving engine whatever the number of requests: more small
energy requests than a grid's second dimension holds (65535) run in one launch."""

import pytest

from host_runtime import on_host  # noqa: F401

SETUP = """
ref = qf.system.hamiltonians.hf_occupation(2, 1, 1)
hmap = qf.HamiltonianMap(2)
h, g = qf.synthetic_integrals(2, 3)
inputs = hmap.pack(0.1, h, g)
pool = qf.SQOpPool()
pool.set_orb_spaces(ref)
pool.fill_pool("SD")
tpl = qf.compile_ucc_template(4, ref, hmap, pool, list(range(len(pool))))
t = [0.1] * tpl.nparam
"""


@pytest.mark.parametrize("gradient", [False, True])
def test_many_small_requests(on_host, gradient):  # noqa: F811
    out = on_host(SETUP + f"""
n = 66000
eng = qf.BatchEngine(64 << 30, 1 << 20)
for _ in range(n): eng.submit(tpl, t, inputs, {gradient})
host.host_forget()
done = 0
while eng.pending() != (0, 0) and done < n: done += len(eng.step(1 << 20))
assert done == n
for name, shape in launches():
    assert max(shape[1:3]) <= 65535 and min(shape[:6]) >= 1, (name, shape)
sums = [s[0] for name, s in launches() if "k_sec_sum" in name]
assert {gradient} or max(sums) > 65535, sums
print("ok")
""")
    assert out.strip() == "ok"


@pytest.mark.parametrize("gradient", [False, True])
def test_a_launch_that_fails_keeps_its_requests(on_host, gradient):  # noqa: F811
    out = on_host(SETUP + f"""
eng = qf.BatchEngine(64 << 30, 1 << 20)
ids = [eng.submit(tpl, t, inputs, {gradient}) for _ in range(5)]
host.host_limit(host.host_used())
for _ in range(2):
    try: eng.step()
    except RuntimeError as e: assert "out of memory" in str(e)
    else: raise SystemExit("launched")
    assert eng.pending() == (5, 0)
host.host_limit(2**63)
done = []
while len(done) < 5: done += eng.step()
assert sorted(i for i, _ in done) == ids and eng.pending() == (0, 0)
print("ok")
""")
    assert out.strip() == "ok"


@pytest.mark.gpu
def test_many_small_requests_values(qf):
    ns = {"qf": qf}
    exec(SETUP, ns)
    tpl, t, inputs = ns["tpl"], ns["t"], ns["inputs"]
    eng = qf.BatchEngine(64 << 30, 1 << 20)
    n = 66000
    scaled = [[x * k for x in t] for k in (1.0, 2.0, 3.0)]
    ids = {eng.submit(tpl, scaled[i % 3], inputs, False): i % 3 for i in range(n)}
    want = [tpl.energy(s, inputs) for s in scaled]
    got = {}
    while len(got) < n:
        got.update(dict(eng.step(1 << 20)))
    assert all(got[i] == want[k] for i, k in ids.items())
