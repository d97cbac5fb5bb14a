"""The reduced form of the plain CG (csrc/redrows.hpp) on the CPU.

The host build runs the exact row functions of the HIP kernels, with every index
checked, through whole CG solves; they must follow CGSolver::solve
(cg_solver.cc:125-177) on the oracle's maps.

The first four iterates are compared with the plain recurrence, to 1e-12 or ten
times what its own two forms (p.A A^T p and ||A^T p||^2) differ by where that is
more: once a Ritz value has converged (with CONSTRAIN_SZ off after two iterations)
rounding is amplified in any form.  Later iterates of two correct forms may part, so
from there on what is held is what does not depend on the path: y and the residual
norm that the recurrence reports belong together, ||rhs - A A^T y||, to 1e-12 of the
first residual.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle_py as orc

HERE = os.path.dirname(os.path.abspath(__file__))

# amopi, na, nb, positivity, constrain_sz, constrain_spin
LAYOUTS = [
    ([4], 2, 2, "DQG", True, True),
    ([5], 3, 2, "DQG", True, True),
    ([6], 4, 2, "DQG", True, True),
    ([1], 1, 0, "DQG", True, True),
    ([2, 1, 1, 0], 2, 2, "DQG", True, True),
    ([0, 3, 2, 1], 3, 1, "DQG", False, True),
    ([2, 1, 1, 1, 0, 1, 1, 1], 3, 3, "DQG", True, True),
    ([4], 2, 2, "DQG", False, True),
    ([5], 2, 2, "DQG", True, False),
    ([5], 2, 2, "DQ", True, True),
    ([3, 2], 3, 2, "DQ", True, True),
    ([5], 2, 2, "DG", True, True),
    ([4], 3, 1, "DG", True, False),
    ([5], 2, 2, "D", True, True),
    ([4], 3, 1, "D", False, True),
    ([7], 3, 3, "DQG", True, True),
    ([5, 0, 0, 0, 0, 5, 0, 0], 5, 5, "DQG", True, True),
]


@pytest.fixture(scope="module")
def lib():
    subprocess.check_call(["make", "-s", "-C", os.path.join(HERE, "emu"), "build/libv2g_emu_red.so"])
    lib = ctypes.CDLL(os.path.join(HERE, "emu", "build", "libv2g_emu_red.so"))
    lib.emu_red_cg.restype = ctypes.c_int
    lib.emu_red_cg.argtypes = ([ctypes.c_int, ctypes.POINTER(ctypes.c_int)] + [ctypes.c_int] * 9
                               + [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_longlong,
                                  ctypes.c_double, ctypes.c_int, ctypes.c_void_p])
    return lib


def _emu(lib, amopi, na, nb, pos, sz, spin, rhs, y, tol, maxiter):
    a = (ctypes.c_int * 8)(*(amopi + [0] * (8 - len(amopi))))
    q2, g2, t1, t2 = orc.positivity_flags(pos)
    y = y.copy()
    res = np.zeros(max(1, maxiter))
    it = lib.emu_red_cg(len(amopi), a, na, nb, na - nb + 1, q2, g2, t2, t1, int(spin), int(sz),
                        rhs.ctypes.data, y.ctypes.data, len(rhs), tol, maxiter, res.ctypes.data)
    return it, y, res


def _plain(L, rhs, y0, maxiter, squares=True):
    y = y0.copy()
    r = rhs - L.Au(L.ATu(y))
    p, rz, res = r.copy(), r @ r, []
    for _ in range(maxiter):
        t = L.ATu(p)
        ap = L.Au(t)
        alpha = rz / (t @ t if squares else p @ ap)
        y += alpha * p
        r = r - alpha * ap
        rz, old = r @ r, rz
        res.append(np.sqrt(rz))
        p = r + rz / old * p
    return y, np.array(res)


@pytest.mark.parametrize("amopi,na,nb,pos,sz,spin", LAYOUTS)
def test_reduced_cg_follows_the_plain_cg(lib, amopi, na, nb, pos, sz, spin):
    L = orc.Layout(amopi, na, nb, na - nb + 1, pos, constrain_sz=sz, constrain_spin=spin)
    rng = np.random.default_rng(3)
    rhs = L.Au(rng.normal(size=L.dimx))
    y0 = rng.normal(size=L.ncon)
    for n in (1, 2, 3, 4) if L.ncon > 60 else (1, 2):
        it, y, res = _emu(lib, amopi, na, nb, pos, sz, spin, rhs, y0, 0.0, n)
        assert it == n
        yr, resr = _plain(L, rhs, y0, n)
        assert np.abs(res - resr).max() <= 1e-12 * resr[0]
        own = np.linalg.norm(_plain(L, rhs, y0, n, squares=False)[0] - yr)
        assert np.linalg.norm(y - yr) <= max(1e-12 * np.linalg.norm(yr), 10 * own)
    if L.ncon > 60:
        r0 = np.linalg.norm(rhs - L.Au(L.ATu(y0)))
        for n in (7, 10, 20):
            it, y, res = _emu(lib, amopi, na, nb, pos, sz, spin, rhs, y0, 0.0, n)
            assert abs(np.linalg.norm(rhs - L.Au(L.ATu(y))) - res[n - 1]) <= 1e-12 * r0


def test_reduced_cg_converges(lib):
    """To a tolerance 1e-11 below the first residual, as a direct CG does."""
    amopi, na, nb = [2, 1, 1, 1, 0, 1, 1, 1], 3, 3
    L = orc.Layout(amopi, na, nb, 1, "DQG")
    rng = np.random.default_rng(4)
    rhs = L.Au(rng.normal(size=L.dimx))
    tol = 1e-11 * np.linalg.norm(rhs)
    it, y, res = _emu(lib, amopi, na, nb, "DQG", True, True, rhs, np.zeros(L.ncon), tol, 1000)
    assert 0 < it < 999 and res[it] < tol
    assert np.linalg.norm(rhs - L.Au(L.ATu(y))) < 10 * tol


def test_layouts_with_second_pass_rows_are_left_out(lib):
    for pos in ("DQGT1", "DQGT2"):
        L = orc.Layout([4], 2, 2, 1, pos)
        assert _emu(lib, [4], 2, 2, pos, True, True, np.zeros(L.ncon), np.zeros(L.ncon), 0.0, 1)[0] == -1
