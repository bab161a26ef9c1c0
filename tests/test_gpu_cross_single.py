"""Two-state expectation values around the rule that takes one pair per thread
(from 18 qubits, fewer than two terms per mask), against numpy."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _masks(word):
    x = z = 0
    ph = 1.0 + 0j
    for letter, q in word:
        if letter in "XY":
            x |= 1 << q
        if letter in "YZ":
            z |= 1 << q
        if letter == "Y":
            ph *= 1j
    return x, z, ph


def _exact(a, b, terms):
    j = np.arange(a.size)
    total = 0j
    for c, word in terms:
        x, z, ph = _masks(word)
        v = j & z
        s = np.zeros_like(j)
        while v.any():
            s ^= v & 1
            v >>= 1
        total += c * ph * np.sum(np.conj(a[j ^ x]) * (1 - 2 * s) * b)
    return total


# per mask: its number of strings
@pytest.mark.parametrize("n", [17, 18, 20])
@pytest.mark.parametrize("sizes", [[1], [1, 1, 1], [2, 1], [2, 2], [1, 3, 1], [3, 2, 1, 1, 1]])
def test_few_terms_per_mask(qf, n, sizes):
    from qforte_amd.engine import workloads as W

    rng = np.random.default_rng(100 * n + len(sizes) + sum(sizes))
    states = []
    for _ in range(2):
        v = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
        v /= np.linalg.norm(v)
        qc = qf.Computer(n)
        qc.set_coeff_vec(v)
        states.append((qc, v))
    terms = []
    for g, count in enumerate(sizes):
        flips = [] if g == 1 else sorted(int(q) for q in rng.choice(n, 2 + g, replace=False))  # mask 1: diagonal
        free = [q for q in range(n) if q not in flips]
        for k in range(count):
            zs = sorted(int(q) for q in rng.choice(free, k + 1, replace=False))
            word = [("Y" if (k + i) % 3 == 1 else "X", q) for i, q in enumerate(flips)] + [("Z", q) for q in zs]
            terms.append((complex(rng.normal(), rng.normal()), word))
    (qa, a), (qb, b) = states
    got = qf.cross_expectations(qa, qb, [W.to_operator(qf, terms), W.to_operator(qf, terms[:1])])
    # sums of 2^n products of modulus about 2^-n, rounded in another order
    assert abs(got[0] - _exact(a, b, terms)) < 1e-14 * len(terms)
    assert abs(got[1] - _exact(a, b, terms[:1])) < 1e-14
