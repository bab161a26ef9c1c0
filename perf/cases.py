"""The work that users of qforte_amd have it do, as measurable cases.

Kinds of case and what each stands for:

* ``circuit``   a gate circuit on a ``Computer`` and the energy of a Pauli sum
* ``trotter``   brickwork layers, a Trotter product of Pauli exponentials, an energy and <Z> of every qubit
* ``expval``    the energy of a molecular Hamiltonian (its full Pauli sum) and one-electron properties in a given state
* ``energy``    one UCCSD energy on the determinant sector: a call of a gradient-free optimizer
* ``gradient``  one UCCSD energy and adjoint gradient on the sector: a call of a VQE optimizer
* ``pool``      the pool gradients of one ADAPT iteration
* ``residual``  the residual amplitudes of one PQE iteration
* ``program``   one UCCSD energy and gradient on the full state (generators outside the sector engine's reach)
* ``serve``     a batch of requests of mixed sizes, each with its own integrals, through ``ServingEngine``

Inputs are drawn from the seed: gates and angles, Pauli strings, integrals,
amplitudes and states.  ``exact`` restates each kind in numpy on plain bit
strings.  ``ops`` is the number of singles and doubles in a UCC ansatz, picked
in random order as ADAPT grows one; 0 is the whole pool in its own order.
"""

import itertools
import math

import numpy as np

import qforte_amd as qf
from qforte_amd.system.hamiltonians import hf_occupation

ONE_QUBIT = ("H", "X", "Y", "Z", "S", "T", "Rx", "Ry", "Rz")
TWO_QUBIT = ("cX", "cZ", "SWAP")
ROTATIONS = ("Rx", "Ry", "Rz")
LETTERS = "XYZ"
# qubits, alpha and beta electrons of the size classes that a mixed batch draws from
MIX = ((8, 2, 2), (10, 3, 2), (12, 3, 3), (14, 4, 3), (16, 4, 4), (18, 5, 4), (20, 5, 5))
ONE_WORKGROUP = 8000  # determinants of a state that one workgroup's LDS holds
EXACT_AMPS = 1 << 27  # amplitudes a numpy sweep over all ops or terms may touch (about 10 s)


def listed():
    return [
        # the plain workload of a first program: 500 random gates, 200 terms, amplitudes read back
        {"name": "circuit-12", "kind": "circuit", "n": 12, "gates": 500, "terms": 200},
        # a longer circuit that no longer fits one compute unit, on an odd number of qubits
        {"name": "circuit-17", "kind": "circuit", "n": 17, "gates": 800, "terms": 300},
        # time evolution at an ordinary size: state beyond the L2 caches, many exponentials
        {"name": "trotter-23", "kind": "trotter", "n": 23, "layers": 4, "strings": 400, "terms": 400},
        # the largest state: 16 GiB
        {"name": "trotter-30", "kind": "trotter", "n": 30, "layers": 4, "strings": 120, "terms": 100},
        # <H> and dipole-like properties of a 9-orbital molecule in a full-space state (gate-level VQE, analysis)
        {"name": "expval-18", "kind": "expval", "n": 18, "properties": 3},
        # the smallest UCC call: latency and launches
        {"name": "energy-8", "kind": "energy", "n": 8, "na": 2, "nb": 2, "ops": 0},
        # an ordinary VQE gradient
        {"name": "gradient-16", "kind": "gradient", "n": 16, "na": 4, "nb": 4, "ops": 0},
        # one ADAPT screening over the generalized singles and doubles, 30 operators into the ansatz
        {"name": "pool-14", "kind": "pool", "n": 14, "na": 4, "nb": 3, "ops": 30, "pool": "GSD"},
        # the largest size class, one request alone over the whole chip: residuals of a PQE step
        {"name": "residual-20", "kind": "residual", "n": 20, "na": 5, "nb": 5, "ops": 0},
        # the full-space gradient
        {"name": "program-14", "kind": "program", "n": 14, "na": 4, "nb": 3, "ops": 0},
        # energies for many optimizers at once (a server's queue)
        {"name": "serve-energy", "kind": "serve", "requests": 512, "largest": 20, "gradient": False},
        # the same with gradients
        {"name": "serve-gradient", "kind": "serve", "requests": 128, "largest": 20, "gradient": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _electrons(rng, n, most):
    """Numbers of alpha and beta electrons, neither space empty nor full, at most ``most`` determinants."""
    half = n // 2
    while True:
        na = rng.randint(1, half - 1)
        nb = max(1, na - rng.randint(0, 1))
        if math.comb(half, na) * math.comb(half, nb) <= most:
            return na, nb


def draw(rng):
    kind = rng.choice(("circuit", "trotter", "expval", "energy", "energy", "gradient", "gradient", "pool", "residual", "program", "serve"))
    if kind == "circuit":
        return {"kind": kind, "n": rng.randint(6, 22), "gates": _log_int(rng, 60, 1000), "terms": _log_int(rng, 20, 400)}
    if kind == "trotter":
        n = rng.randint(18, 29)
        most = min(500, 120 << (30 - n))
        return {"kind": kind, "n": n, "layers": rng.randint(1, 4), "strings": _log_int(rng, 40, most), "terms": _log_int(rng, 40, most)}
    if kind == "expval":
        return {"kind": kind, "n": 2 * rng.randint(4, 10), "properties": rng.randint(1, 9)}
    if kind == "serve":
        return {"kind": kind, "requests": _log_int(rng, 8, 256), "largest": 2 * rng.randint(4, 10), "gradient": rng.random() < 0.4}
    n = 2 * rng.randint(3, 7 if kind in ("pool", "program") else 10)
    na, nb = _electrons(rng, n, ONE_WORKGROUP if kind in ("energy", "gradient") else 1 << 16)
    whole = _sector_work(n, na, nb)[3]
    case = {"kind": kind, "n": n, "na": na, "nb": nb, "ops": 0 if rng.random() < 0.5 else _log_int(rng, min(4, whole), min(100, whole))}
    if kind == "pool":
        case["pool"] = rng.choice(("SD", "GSD"))
    return case


# ---- inputs as plain data ----------------------------------------------------------------


def _gates(rng, n, count):
    """(type, target, control, angle) of a random circuit on uniformly random qubits."""
    out = []
    kinds = ONE_QUBIT + TWO_QUBIT
    for _ in range(count):
        g = kinds[int(rng.integers(len(kinds)))]
        if g in TWO_QUBIT:
            t, c = (int(v) for v in rng.choice(n, size=2, replace=False))
            out.append((g, t, c, 0.0))
        else:
            q = int(rng.integers(n))
            out.append((g, q, q, float(rng.uniform(0.0, 2.0 * math.pi)) if g in ROTATIONS else 0.0))
    return out


def _brickwork(rng, n, layers):
    out = []
    for layer in range(layers):
        for q in range(n):
            out.append(("Ry", q, q, float(rng.uniform(0.0, 2.0 * math.pi))))
            out.append(("Rz", q, q, float(rng.uniform(0.0, 2.0 * math.pi))))
        out += [("cX", lo + 1, lo, 0.0) for lo in range(layer % 2, n - 1, 2)]
    return out


def _pauli_strings(rng, n, count, wmin, wmax, width):
    """(real number ~ N(0, width), [(letter, qubit), ...]) of random weights."""
    out = []
    for _ in range(count):
        w = int(rng.integers(min(wmin, n), min(wmax, n) + 1))
        qubits = sorted(int(v) for v in rng.choice(n, size=w, replace=False))
        out.append((float(rng.normal(0.0, width)), [(LETTERS[int(rng.integers(3))], q) for q in qubits]))
    return out


def _integrals(rng, norb):
    """(h, g): h symmetric, g with the 8-fold symmetry of real chemist-notation integrals."""
    h = rng.normal(0.0, 0.1, (norb, norb))
    h = 0.5 * (h + h.T)
    h[np.diag_indices(norb)] -= 2.0 * np.arange(norb) / norb
    g = rng.normal(0.0, 0.01, (norb,) * 4)
    g = g + g.transpose(1, 0, 2, 3)
    g = g + g.transpose(0, 1, 3, 2)
    g = (g + g.transpose(2, 3, 0, 1)) / 8.0
    for p in range(norb):
        g[p, p, p, p] += 0.5
    return h, g


def _properties(rng, norb, count):
    """Symmetric one-electron matrices (dipole components and the like)."""
    m = rng.normal(0.0, 0.3, (count, norb, norb))
    return 0.5 * (m + m.transpose(0, 2, 1))


def _amplitudes(rng, count):
    return rng.normal(0.0, 0.05, count)


def _tops(case, rng):
    """Indices into the SD pool of the ansatz's operators, in the order of their application."""
    whole = _sector_work(case["n"], case["na"], case["nb"])[3]
    return rng.permutation(whole)[:case["ops"]].tolist() if case["ops"] else list(range(whole))


def _random_state(rng, n):
    v = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    return v / np.linalg.norm(v)


def _excited(n, na, nb):
    """The singly and doubly excited determinants of the aufbau determinant, as integers in ascending order."""
    occ = [2 * i for i in range(na)] + [2 * i + 1 for i in range(nb)]
    virt = [p for p in range(n) if p not in occ]
    ref = sum(1 << p for p in occ)
    out = [ref ^ (1 << i) ^ (1 << a) for i in occ for a in virt if (i - a) % 2 == 0]
    for i, j in itertools.combinations(occ, 2):
        for a, b in itertools.combinations(virt, 2):
            if (i & 1) + (j & 1) == (a & 1) + (b & 1):
                out.append(ref ^ (1 << i) ^ (1 << j) ^ (1 << a) ^ (1 << b))
    return sorted(out)


def _requests(case, rng):
    """(size class, integrals, amplitude seed) of every request of a mixed batch."""
    classes = [m for m in MIX if m[0] <= case["largest"]]
    out = []
    for k in rng.permutation(case["requests"]):
        m = classes[int(k) % len(classes)]
        out.append((m, _integrals(rng, m[0] // 2), int(rng.integers(1 << 30))))
    return out


# ---- qforte_amd objects from plain data ----------------------------------------------------


def _circuit(gates):
    c = qf.Circuit()
    for g, t, ctl, angle in gates:
        if t != ctl:
            c.add(qf.gate(g, t, ctl))
        elif g in ROTATIONS:
            c.add(qf.gate(g, t, t, angle))
        else:
            c.add(qf.gate(g, t, t))
    return c


def _operator(terms, factor=1.0):
    op = qf.QubitOperator()
    for c, string in terms:
        op.add(factor * c, _circuit([(p, q, q, 0.0) for p, q in string]))
    return op


def _pool(ref, kind):
    pool = qf.SQOpPool()
    pool.set_orb_spaces(ref)
    pool.fill_pool(kind)
    return pool


def _template(n, na, nb, tops=None):
    """The compiled template of one ansatz and its map from integrals."""
    ref = hf_occupation(n // 2, na, nb)
    pool = _pool(ref, "SD")
    hmap = qf.HamiltonianMap(n // 2)
    return qf.compile_ucc_template(n, ref, hmap, pool, list(range(len(pool))) if tops is None else tops), hmap, ref


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "circuit":
        gates = _gates(rng, case["n"], case["gates"])
        terms = _pauli_strings(rng, case["n"], case["terms"], 1, 6, 1.0)
        return {"kind": kind, "qc": qf.Computer(case["n"]), "circuit": _circuit(gates), "operator": _operator(terms)}
    if kind == "trotter":
        n = case["n"]
        layers = _brickwork(rng, n, case["layers"])
        strings = _pauli_strings(rng, n, case["strings"], 4, 8, 0.1)
        terms = _pauli_strings(rng, n, case["terms"], 1, 6, 1.0)
        evolution, _ = qf.trotterize(_operator(strings, -1j))
        pool = qf.QubitOpPool()
        for q in range(n):
            pool.add(1.0, _operator([(1.0, [("Z", q)])]))
        return {"kind": kind, "qc": qf.Computer(n), "circuit": _circuit(layers), "evolution": evolution,
                "operator": _operator(terms), "spins": pool}
    if kind == "expval":
        n = case["n"]
        hmap = qf.HamiltonianMap(n // 2)
        operator = hmap.operator(hmap.pack(0.5, *_integrals(rng, n // 2)))
        pool = qf.QubitOpPool()
        for m in _properties(rng, n // 2, case["properties"]):
            one = qf.SQOperator()
            for p in range(n // 2):
                for q in range(n // 2):
                    one.add(m[p, q], [2 * p], [2 * q])
                    one.add(m[p, q], [2 * p + 1], [2 * q + 1])
            pool.add(1.0, one.jw_transform())
        qc = qf.Computer(n)
        qc.set_coeff_vec(_random_state(rng, n))
        return {"kind": kind, "qc": qc, "operator": operator, "properties": pool}
    if kind == "serve":
        compiled = {m: _template(*m) for m in MIX if m[0] <= case["largest"]}
        requests = []
        for m, (h, g), s in _requests(case, rng):
            template, hmap, _ = compiled[m]
            t = _amplitudes(np.random.default_rng(s), template.nparam)
            requests.append((m[0], template, t.tolist(), hmap.pack(0.0, h, g)))
        return {"kind": kind, "engine": qf.ServingEngine(), "requests": requests, "gradient": case["gradient"]}
    n, na, nb = case["n"], case["na"], case["nb"]
    h, g = _integrals(rng, n // 2)
    tops = _tops(case, rng)
    if kind == "program":
        ref = hf_occupation(n // 2, na, nb)
        pool = _pool(ref, "SD")
        hmap = qf.HamiltonianMap(n // 2)
        program = qf.compile_ucc_program(n, ref, hmap.operator(hmap.pack(0.0, h, g)), pool, tops)
        return {"kind": kind, "program": program, "t": _amplitudes(rng, len(tops)).tolist()}
    template, hmap, ref = _template(n, na, nb, tops)
    state = {"kind": kind, "template": template, "t": _amplitudes(rng, template.nparam).tolist(), "inputs": hmap.pack(0.0, h, g)}
    if kind == "residual":
        excited = _excited(n, na, nb)
        state["determinants"] = [excited[k] for k in tops]
    if kind == "pool":
        pool = _pool(ref, case["pool"])
        state["operators"], _, _ = qf.ucc_generators(pool, list(range(len(pool))))
    return state


def run(state):
    kind = state["kind"]
    if kind == "circuit":
        qc = state["qc"]
        qc.reset()
        qc.apply_circuit(state["circuit"])
        return {"energy": np.complex128(qc.direct_op_exp_val(state["operator"])), "amplitudes": qc.get_coeff_vec()}
    if kind == "trotter":
        qc = state["qc"]
        qc.reset()
        qc.apply_circuit(state["circuit"])
        qc.apply_circuit(state["evolution"])
        return {"energy": np.complex128(qc.direct_op_exp_val(state["operator"])),
                "spins": np.array(qc.direct_oppl_exp_val(state["spins"]))}
    if kind == "expval":
        qc = state["qc"]
        return {"energy": np.complex128(qc.direct_op_exp_val(state["operator"])),
                "properties": np.array(qc.direct_oppl_exp_val(state["properties"]))}
    if kind == "energy":
        return {"energy": state["template"].energy(state["t"], state["inputs"])}
    if kind == "gradient":
        e, g = state["template"].gradient(state["t"], state["inputs"])
        return {"energy": e, "gradient": np.array(g)}
    if kind == "program":
        e, g = state["program"].gradient(state["t"])
        return {"energy": e, "gradient": np.array(g)}
    if kind == "residual":
        return {"residuals": np.array(state["template"].residuals(state["t"], state["determinants"], state["inputs"]))}
    if kind == "pool":
        return {"gradients": np.array(state["template"].pool_gradients(state["t"], state["operators"], 64, state["inputs"]))}
    engine, want = state["engine"], state["gradient"]
    ids = [(n, engine.submit(template, t, inputs, gradient=want)) for n, template, t, inputs in state["requests"]]
    engine.drain()
    out = {}
    for n in sorted({n for n, _ in ids}):
        out["energy-%d" % n] = np.array([engine.results.pop(i) for m, i in ids if m == n])
        if want:
            out["gradient-%d" % n] = np.concatenate([engine.gradients.pop(i) for m, i in ids if m == n])
    return out


# ---- what a pass cannot do without -----------------------------------------------------------


def _sector_work(n, na, nb):
    """(determinants, amplitude pairs of the SD rotations, determinants that H connects one with, parameters)."""
    no = n // 2
    va, vb = no - na, no - nb
    c = math.comb
    dets = c(no, na) * c(no, nb)
    single = na * va * c(no - 2, na - 1) * c(no, nb) + nb * vb * c(no - 2, nb - 1) * c(no, na)
    same = (c(na, 2) * c(va, 2) * (c(no - 4, na - 2) if no >= 4 and na >= 2 else 0) * c(no, nb)
            + c(nb, 2) * c(vb, 2) * (c(no - 4, nb - 2) if no >= 4 and nb >= 2 else 0) * c(no, na))
    mixed = na * va * nb * vb * c(no - 2, na - 1) * c(no - 2, nb - 1)
    count = na * va + nb * vb + c(na, 2) * c(va, 2) + c(nb, 2) * c(vb, 2) + na * va * nb * vb
    return dets, single + same + mixed, 1 + count, count


def _ucc_work(n, na, nb, gradient, ops=0):
    dets, pairs, linked, params = _sector_work(n, na, nb)
    if ops:
        pairs, params = pairs * ops / params, ops
    norb = n // 2
    p = norb * (norb + 1) // 2
    flops = 6.0 * pairs + (2.0 if gradient else 1.0) * dets * linked
    if gradient:
        flops += 16.0 * pairs  # both states un-rotated, and the overlap of every pair
    return 8.0 * (params + 1 + p + p * (p + 1) // 2) + (8.0 * params if gradient else 8.0), flops


def work(case):
    kind = case["kind"]
    if kind == "circuit":
        size = 2.0 ** case["n"]
        return {"bytes": 32.0 * size, "flops": size * (14.0 * case["gates"] + 4.0 * case["terms"])}
    if kind == "trotter":
        size = 2.0 ** case["n"]
        ops = 2 * case["n"] * case["layers"] + case["strings"]
        return {"bytes": 32.0 * size, "flops": size * (10.0 * ops + 4.0 * case["terms"])}
    if kind == "expval":
        size, norb = 2.0 ** case["n"], case["n"] // 2
        return {"bytes": 16.0 * size, "flops": size * 4.0 * norb ** 4 / 8.0}
    if kind == "serve":
        classes = [m for m in MIX if m[0] <= case["largest"]]
        each = [_ucc_work(*m, case["gradient"]) for m in classes]
        share = case["requests"] / len(classes)
        return {"bytes": share * sum(b for b, _ in each), "flops": share * sum(f for _, f in each)}
    b, f = _ucc_work(case["n"], case["na"], case["nb"], kind != "energy", case["ops"])
    return {"bytes": b, "flops": f}


# ---- the same in numpy, 64 bits ----------------------------------------------------------------

_R = math.sqrt(0.5)
_FIXED = {
    "X": [[0, 1], [1, 0]], "Y": [[0, -1j], [1j, 0]], "Z": [[1, 0], [0, -1]], "H": [[_R, _R], [_R, -_R]],
    "S": [[1, 0], [0, 1j]], "T": [[1, 0], [0, complex(_R, _R)]],
}


def _matrix(g, angle):
    if g in _FIXED:
        return np.array(_FIXED[g], dtype=np.complex128)
    c, s = math.cos(angle / 2.0), math.sin(angle / 2.0)
    if g == "Rx":
        return np.array([[c, -1j * s], [-1j * s, c]])
    if g == "Ry":
        return np.array([[c, -s], [s, c]], dtype=np.complex128)
    return np.array([[complex(c, -s), 0], [0, complex(c, s)]])


def _apply_gates(psi, n, gates):
    for g, t, ctl, angle in gates:
        if t == ctl:
            v = psi.reshape(-1, 2, 1 << t)
            psi = np.einsum("ij,ajb->aib", _matrix(g, angle), v).reshape(-1)
            continue
        hi, lo = max(t, ctl), min(t, ctl)
        v = psi.reshape(1 << (n - 1 - hi), 2, 1 << (hi - lo - 1), 2, 1 << lo).copy()
        if g == "SWAP":
            v[:, 0, :, 1], v[:, 1, :, 0] = v[:, 1, :, 0].copy(), v[:, 0, :, 1].copy()
        elif g == "cZ":
            v[:, 1, :, 1] *= -1.0
        elif ctl == hi:
            v[:, 1] = v[:, 1, :, ::-1].copy()
        else:
            v[:, :, :, 1] = v[:, ::-1, :, 1].copy()
        psi = v.reshape(-1)
    return psi


def _parity(v):
    v = v.astype(np.uint64)
    for s in (16, 8, 4, 2, 1):
        v = v ^ (v >> np.uint64(s))
    return (v & np.uint64(1)).astype(np.int64)


def _apply_pauli(psi, index, string):
    """P |psi>: X flips, Z signs, Y = i X Z on each of its qubits."""
    x = sum(1 << q for p, q in string if p != "Z")
    z = sum(1 << q for p, q in string if p != "X")
    ny = sum(1 for p, _ in string if p == "Y")
    src = index ^ x
    return (1j ** ny) * (1.0 - 2.0 * _parity(src & z)) * psi[src]


def _exact_circuit(case, seed):
    n = case["n"]
    rng = np.random.default_rng(seed)
    trotter = case["kind"] == "trotter"
    gates = _brickwork(rng, n, case["layers"]) if trotter else _gates(rng, n, case["gates"])
    strings = _pauli_strings(rng, n, case["strings"], 4, 8, 0.1) if trotter else []
    terms = _pauli_strings(rng, n, case["terms"], 1, 6, 1.0)
    if (len(gates) + 2 * len(strings) + 2 * len(terms)) << n > EXACT_AMPS:
        return None
    psi = np.zeros(1 << n, dtype=np.complex128)
    psi[0] = 1.0
    psi = _apply_gates(psi, n, gates)
    index = np.arange(1 << n, dtype=np.int64)
    for theta, string in strings:
        psi = math.cos(theta) * psi - 1j * math.sin(theta) * _apply_pauli(psi, index, string)
    energy = sum(c * np.vdot(psi, _apply_pauli(psi, index, string)) for c, string in terms)
    if not trotter:
        return {"energy": np.complex128(energy), "amplitudes": psi}
    p = np.abs(psi) ** 2
    return {"energy": np.complex128(energy), "spins": np.array([np.sum(p * (1.0 - 2.0 * ((index >> q) & 1))) for q in range(n)]) + 0j}


class _Determinants:
    """Fermionic operators on a list of determinants (bit p = spin orbital p, alpha even, beta odd)."""

    def __init__(self, n, na=None, nb=None):
        j = np.arange(1 << n, dtype=np.int64)
        if na is not None:
            even = sum(1 << p for p in range(0, n, 2))
            bits = lambda v: sum((v >> p) & 1 for p in range(n))  # noqa: E731
            j = j[(bits(j & even) == na) & (bits(j & (even << 1)) == nb)]
        self.n, self.dets = n, j
        self.rank = np.full(1 << n, -1, dtype=np.int64)
        self.rank[j] = np.arange(len(j))

    def ladder(self, create, annihilate):
        """(source, target, sign) of a+_c0 a+_c1 .. a_a0 a_a1 .. on every determinant that it does not kill."""
        need = sum(1 << p for p in annihilate)
        src = np.nonzero((self.dets & need) == need)[0]
        j = self.dets[src]
        odd = np.zeros(len(j), dtype=np.int64)
        alive = np.ones(len(j), dtype=bool)
        for p, make in [(p, False) for p in reversed(annihilate)] + [(p, True) for p in reversed(create)]:
            odd ^= _parity(j & ((1 << p) - 1))
            alive &= ((j >> p) & 1) == (0 if make else 1)
            j = j ^ (1 << p)
        src, j, odd = src[alive], j[alive], odd[alive]
        return src, self.rank[j], 1.0 - 2.0 * odd

    def hamiltonian(self, psi, constant, h, g):
        """sum h_pq E_pq + 1/2 sum (pq|rs) (E_pq E_rs - delta_qr E_ps) + constant on psi."""
        norb = self.n // 2
        moves = []
        d = np.zeros((norb * norb, len(psi)), dtype=psi.dtype)
        for p in range(norb):
            for q in range(norb):
                for spin in (0, 1):
                    src, dst, sign = self.ladder([2 * p + spin], [2 * q + spin])
                    moves.append((p * norb + q, src, dst, sign))
                    d[p * norb + q, dst] += sign * psi[src]
        one = (h - 0.5 * np.einsum("prrq->pq", g)).reshape(-1)
        out = constant * psi + one @ d
        d = ((0.5 * g.reshape(norb * norb, norb * norb)) @ d.view(np.float64)).view(psi.dtype)
        for k, src, dst, sign in moves:
            out[dst] += sign * d[k, src]
        return out

    def transitions(self, psi, matrices):
        """<psi| sum m_pq E_pq |psi> of every one-electron matrix."""
        out = np.zeros(len(matrices), dtype=np.complex128)
        for p in range(self.n // 2):
            for q in range(self.n // 2):
                for spin in (0, 1):
                    src, dst, sign = self.ladder([2 * p + spin], [2 * q + spin])
                    out += matrices[:, p, q] * np.sum(psi[dst].conj() * sign * psi[src])
        return out

    def excitations(self, na, nb):
        """(reference, (creators, annihilators) of every excited determinant), orbitals descending."""
        ref = sum(1 << (2 * i) for i in range(na)) + sum(1 << (2 * i + 1) for i in range(nb))
        out = []
        for d in _excited(self.n, na, nb):
            down = [p for p in range(self.n - 1, -1, -1) if ((d ^ ref) >> p) & 1]
            out.append(([p for p in down if not (ref >> p) & 1], [p for p in down if (ref >> p) & 1]))
        return ref, out


def _exact_ucc(n, na, nb, h, g, tops, t, want):
    """``want`` "energy" or "gradient": (energy, gradient or None); "pool" or "residual": those numbers."""
    space = _Determinants(n, na, nb)
    ref, excitations = space.excitations(na, nb)
    psi = np.zeros(len(space.dets))
    psi[space.rank[ref]] = 1.0
    pairs = [space.ladder(*e) for e in excitations]

    def rotate(v, k, angle):
        src, dst, sign = pairs[tops[k]]
        c, s = math.cos(angle), math.sin(angle)
        a, b = v[src], v[dst]
        v[src], v[dst] = c * a - s * sign * b, c * b + s * sign * a

    def overlap(op):
        src, dst, sign = pairs[op]
        return 2.0 * float(np.sum(sign * (sigma[dst] * psi[src] - sigma[src] * psi[dst])))

    for k in range(len(t)):
        rotate(psi, k, t[k])
    sigma = space.hamiltonian(psi, 0.0, h, g)
    energy = float(psi @ sigma)
    if want == "pool":
        return np.array([overlap(k) for k in range(len(pairs))])
    if want == "residual":
        for k in reversed(range(len(t))):
            rotate(sigma, k, -t[k])
        excited = _excited(n, na, nb)
        return sigma[space.rank[[excited[k] for k in tops]]] + 0j
    if want == "energy":
        return energy, None
    grad = np.zeros(len(t))
    for k in reversed(range(len(t))):
        grad[k] = overlap(tops[k])
        rotate(psi, k, -t[k])
        rotate(sigma, k, -t[k])
    return energy, grad


def exact(case, seed):
    kind = case["kind"]
    if kind in ("circuit", "trotter"):
        return _exact_circuit(case, seed)
    rng = np.random.default_rng(seed)
    if kind == "expval":
        n = case["n"]
        if n > 18:
            return None
        h, g = _integrals(rng, n // 2)
        one = _properties(rng, n // 2, case["properties"])
        psi = _random_state(rng, n)
        space = _Determinants(n)
        return {"energy": np.complex128(np.vdot(psi, space.hamiltonian(psi, 0.5, h, g))),
                "properties": space.transitions(psi, one)}
    if kind == "serve":
        out, left = {}, 12
        rows = _requests(case, rng)
        for m in sorted({m for m, _, _ in rows}):
            mine = [(hg, s) for k, hg, s in rows if k == m]
            left -= len(mine) * _sector_work(*m)[1] / 1e6
            got = [None] * len(mine) if left < 0 or m[0] > 14 else [
                _exact_ucc(*m, *hg, range(_sector_work(*m)[3]), _amplitudes(np.random.default_rng(s), _sector_work(*m)[3]),
                           "gradient" if case["gradient"] else "energy") for hg, s in mine]
            known = got[0] is not None
            out["energy-%d" % m[0]] = np.array([e for e, _ in got]) if known else None
            if case["gradient"]:
                out["gradient-%d" % m[0]] = np.concatenate([d for _, d in got]) if known else None
        return out
    n, na, nb = case["n"], case["na"], case["nb"]
    h, g = _integrals(rng, n // 2)
    tops = _tops(case, rng)
    t = _amplitudes(rng, len(tops))
    if kind == "pool" and case["pool"] != "SD":
        return None
    got = _exact_ucc(n, na, nb, h, g, tops, t, "gradient" if kind == "program" else kind)
    if kind in ("pool", "residual"):
        return {"gradients" if kind == "pool" else "residuals": got}
    return {"energy": got[0]} if kind == "energy" else {"energy": got[0], "gradient": got[1]}
