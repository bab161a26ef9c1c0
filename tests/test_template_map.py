"""The coefficient map of a sector template: an index outside the inputs or
offsets that decrease are refused for every term that connects determinants
of the sector, in real and in complex templates; a term that connects none is
read by nothing."""

import pytest

from host_runtime import on_host  # noqa: F401

CODE = """
class C64(ctypes.Structure):
    _fields_ = [("re", ctypes.c_double), ("im", ctypes.c_double)]
class Pauli(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint64), ("z", ctypes.c_uint64), ("phase", C64), ("coeff", C64)]
lib = ctypes.CDLL(os.path.join(os.path.dirname(qf.__file__), "libqfe.so"))
lib.qfe_last_error.restype = ctypes.c_char_p
N = 8  # 4 orbitals, 2 + 2 electrons: alpha on even bits, beta on odd ones
REF = 0b00001111
# term: (x, z): diagonal, alpha flip, beta flip, flips of both, three alpha flips' worth of bits (odd), one flip of each
TERMS = {"diagonal": (0, 0b101), "alpha": (0b00010001, 0), "beta": (0b00100010, 0b10000), "both": (0b00110011, 0), "none": (0b00000001, 0), "mixed": (0b11, 0)}
def create(off, idx, ninputs, imag):
    names = list(TERMS)
    ham = (Pauli * len(names))(*[Pauli(*TERMS[k], C64(1, 0), C64(1, 0)) for k in names])
    val = (C64 * len(idx))(*[C64(0.5, imag) for _ in idx])
    goff = (ctypes.c_uint64 * 1)(0)
    t = ctypes.c_void_p()
    rc = lib.qfe_template_create(N, ctypes.c_uint64(REF), None, goff, ctypes.c_uint64(0), None, None, ctypes.c_uint64(0), ham,
                                 ctypes.c_uint64(len(names)), (ctypes.c_uint64 * len(off))(*off), (ctypes.c_uint32 * len(idx))(*idx), val,
                                 ctypes.c_uint64(ninputs), ctypes.byref(t))
    if t: lib.qfe_template_destroy(t)
    return rc, lib.qfe_last_error()
n = len(TERMS)
for imag in (0.0, 0.25):
    good = list(range(n))
    assert create(list(range(n + 1)), good, n, imag)[0] == 0
    for k, name in enumerate(TERMS):
        connects = name not in ("none", "mixed")
        for bad in (n, n + 1, 2**32 - 1):
            rc, msg = create(list(range(n + 1)), good[:k] + [bad] + good[k + 1:], n, imag)
            assert (rc == 1 and b"map index" in msg) if connects else rc == 0, (imag, name, bad, rc, msg)
        if connects:
            off = list(range(n + 1))
            off[k], off[k + 1] = off[k + 1], off[k]
            rc, msg = create(off, good, n, imag)
            assert rc == 1 and b"offsets" in msg, (imag, name, rc, msg)
print("ok")
"""


def test_map_is_checked_for_every_connecting_term(on_host):  # noqa: F811
    assert on_host(CODE).strip() == "ok"
