"""Generators of a full-space program: a string that is not Hermitian is
refused as one exponential is."""

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


def test_strings_that_are_not_hermitian(on_host):  # noqa: F811
    out = on_host(CODE + """
for im, rc in ((0.0, 0), (4e-16, 0), (6e-16, 1), (9e-16, 1), (2e-15, 1), (0.5, 1)):
    assert energy([(1, 0, (1, im), 0.5)])[0] == rc, (im, lib.qfe_last_error())
    assert energy([(1, 1, (im, 1), 0.5)])[0] == rc, (im, lib.qfe_last_error())
assert energy([(1, 0, (1 + 1e-11, 0), 0.5)])[0] == 1
print("ok")
""")
    assert out.strip() == "ok"
