"""The T2 rows by column lists and A^T y gathered by shared orbitals (csrc/t2rows.hpp) on the CPU, with every index checked,
against the oracle: the rows of A.x, and A^T.y of a y that is zero elsewhere."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle_py as orc

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib():
    subprocess.check_call(["make", "-s", "-C", os.path.join(HERE, "emu"), "build/libv2g_emu_t2.so"])
    lib = ctypes.CDLL(os.path.join(HERE, "emu", "build", "libv2g_emu_t2.so"))
    lib.emu_t2.restype = ctypes.c_longlong
    lib.emu_t2.argtypes = ([ctypes.c_int, ctypes.POINTER(ctypes.c_int)] + [ctypes.c_int] * 5
                           + [ctypes.c_void_p] * 4 + [ctypes.c_longlong] * 2)
    lib.emu_t2_rows.argtypes = ([ctypes.c_int, ctypes.POINTER(ctypes.c_int)] + [ctypes.c_int] * 5
                                + [ctypes.c_void_p])
    return lib


# the last has blocks of several chunks of columns
@pytest.mark.parametrize("amopi,na,nb,mult,pos,sz", [
    ([1], 1, 0, 2, "DQGT2", True),
    ([2], 1, 1, 1, "DQGT2", True),
    ([5], 3, 2, 2, "DQGT2", True),
    ([4], 2, 2, 1, "DQGT2", False),
    ([2, 1, 1, 1], 2, 2, 1, "DQGT2", True),
    ([3, 0, 1, 1, 0, 2, 1, 1], 4, 3, 2, "DQGT2", True),
    ([2, 1, 1, 1], 3, 2, 2, "DQGT1T2", True),
    ([11], 3, 3, 1, "DQGT2", True),
])
def test_t2_rows_match_oracle(lib, amopi, na, nb, mult, pos, sz):
    L = orc.Layout(amopi, na, nb, mult, pos, constrain_sz=sz)
    a = (ctypes.c_int * 8)(*(amopi + [0] * (8 - len(amopi))))
    args = (len(amopi), a, na, nb, mult, int("T1" in pos), int(sz))
    t2 = np.zeros(L.ncon, dtype=np.int8)
    lib.emu_t2_rows(*args, t2.ctypes.data)
    rng = np.random.default_rng(5)
    x, y = rng.normal(size=L.dimx), rng.normal(size=L.ncon) * t2
    ax, aty = np.zeros(L.ncon), np.zeros(L.dimx)
    assert lib.emu_t2(*args, x.ctypes.data, ax.ctypes.data, y.ctypes.data, aty.ctypes.data, L.dimx, L.ncon) == 0
    ref = L.Au(x) * t2
    assert np.linalg.norm(ax - ref) <= 1e-13 * np.linalg.norm(ref)
    ref = L.ATu(y)
    assert np.linalg.norm(aty - ref) <= 1e-13 * np.linalg.norm(ref)
