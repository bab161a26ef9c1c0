"""Which generators of a full-space program go as pair rotations: those whose
strings have one weight on all pairs that they move, to rounding.  A generator
whose weights differ by more keeps its exponentials, and a string that is not
Hermitian is refused as one exponential is."""

import numpy as np
import pytest

from host_runtime import on_host  # noqa: F401

CODE = """
class C64(ctypes.Structure):
    _fields_ = [("re", ctypes.c_double), ("im", ctypes.c_double)]
class Pauli(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint64), ("z", ctypes.c_uint64), ("phase", C64), ("coeff", C64)]
lib = ctypes.CDLL(os.path.join(os.path.dirname(qf.__file__), "libqfe.so"))
lib.qfe_last_error.restype = ctypes.c_char_p
def energy(terms):
    gen = (Pauli * len(terms))(*[Pauli(x, z, C64(*ph), C64(0.0, c)) for x, z, ph, c in terms])
    ham = (Pauli * 1)(Pauli(0, 1, C64(1, 0), C64(1, 0)))
    off = (ctypes.c_uint64 * 2)(0, len(terms))
    p, e = ctypes.c_void_p(), ctypes.c_double()
    rc = lib.qfe_program_create(4, ctypes.c_uint64(3), gen, off, ctypes.c_uint64(1), (ctypes.c_int32 * 1)(0), (ctypes.c_double * 1)(1.0),
                                ctypes.c_uint64(1), ham, ctypes.c_uint64(1), ctypes.byref(p))
    assert rc == 0, lib.qfe_last_error()
    host.host_forget()
    rc = lib.qfe_program_energy(p, (ctypes.c_double * 1)(0.3), ctypes.byref(e))
    return rc, any("k_program_tile" in n for n, _ in launches())
"""


def test_one_weight_to_rounding(on_host):  # noqa: F811
    out = on_host(CODE + """
X, Y = (1, 0), (0, 1)
for d, tiles in ((0.0, True), (2.0**-52, True), (2e-14, False), (5e-13, False), (0.1, False)):
    # X0 X1 and Y0 Y1: weights 2 and 0 on the pairs; X0 and X0 Z1: the same
    assert energy([(3, 0, X, 0.5), (3, 3, (-1, 0), 0.5 * (1 + d))]) == (0, tiles), d
    assert energy([(1, 0, X, 0.5), (1, 2, X, 0.5 * (1 + d))]) == (0, tiles), d
    # two pairs of weights 1 and 1 + d
    assert energy([(1, 0, X, 1 + d / 2), (1, 2, X, d / 2)]) == (0, tiles), d
print("ok")
""")
    assert out.strip() == "ok"


def test_strings_that_are_not_hermitian(on_host):  # noqa: F811
    out = on_host(CODE + """
for im, rc in ((0.0, 0), (4e-16, 0), (6e-16, 1), (9e-16, 1), (2e-15, 1), (0.5, 1)):
    assert energy([(1, 0, (1, im), 0.5)])[0] == rc, (im, lib.qfe_last_error())
    assert energy([(1, 1, (im, 1), 0.5)])[0] == rc, (im, lib.qfe_last_error())
assert energy([(1, 0, (1 + 1e-11, 0), 0.5)])[0] == 1
print("ok")
""")
    assert out.strip() == "ok"


@pytest.mark.gpu
@pytest.mark.parametrize("d", [0.0, 2e-14, 5e-13, 0.1])
def test_small_weights_are_kept(qf, d):
    """exp(t K), K = i/2 (X0 + (1 + d) X0 Z1), on |q1 = 1>: a rotation by t d / 2."""
    gen = qf.QubitOperator()
    for c, word in ((0.5, "X_0"), (0.5 * (1 + d), "X_0 Z_1")):
        gen.add_op(qf.build_operator(f"{c!r}j, {word}"))
    H = qf.build_operator("1.0, Z_0")
    prog = qf.UCCProgram(2, 2, [gen], [0], [1.0], 1, H)
    qc = qf.Computer(2)
    prog.prepare([0.8], qc)
    a = np.asarray(qc.get_coeff_vec())
    d = 0.5 * (1 + d) - 0.5  # as the coefficients hold it
    assert abs(a[2] - np.cos(0.8 * d)) < 4e-16
    assert abs(a[3] + 1j * np.sin(0.8 * d)) < 4e-16
