"""The capped CG of single handles, iterate by iterate, over every kind of layout: the
reduced form with and without Q2, G2, spin rows and S_z, and the fused general form with
T2 rows in one and in several chunks of columns (t2rows.hpp).

y, the residual norm and the count after n iterations, odd and even, against the plain
recurrence of CGSolver::solve (cg_solver.cc:125-177) on the oracle's maps: 1e-12, or ten
times what the recurrence's own two forms (p.A A^T p and ||A^T p||^2) differ by where that
is more.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle_py as orc  # noqa: E402
from test_red_cg import LAYOUTS, _plain  # noqa: E402

pytestmark = pytest.mark.gpu

T2 = [
    ([5], 3, 2, "DQGT2", True, True),
    ([2, 1, 1, 1], 2, 2, "DQGT2", True, True),
    ([8, 6], 5, 5, "DQGT2", False, True),   # aba columns in two chunks
    ([14], 4, 4, "DQGT2", True, True),      # 1 274 aab and 2 744 aba columns: two and three
]


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _pair(amopi, na, nb, pos, sz, spin):
    from v2rdm_casscf_amd import V2RDMSolver
    s = V2RDMSolver(amopi, na, nb, na - nb + 1, pos, constrain_sz=sz, constrain_spin=spin)
    return s, orc.Layout(amopi, na, nb, na - nb + 1, pos, constrain_sz=sz, constrain_spin=spin)


@pytest.mark.parametrize("amopi,na,nb,pos,sz,spin", LAYOUTS + T2)
def test_capped_cg_matches_recurrence(amopi, na, nb, pos, sz, spin):
    s, L = _pair(amopi, na, nb, pos, sz, spin)
    rng = np.random.default_rng(3)
    rhs = L.Au(rng.normal(size=L.dimx))
    y0 = rng.normal(size=L.ncon)
    for n in (1, 2) if L.ncon <= 60 or L.ncon > 10 ** 6 else (1, 2, 3, 4):
        yr, resr = _plain(L, rhs, y0, n)
        own = np.linalg.norm(_plain(L, rhs, y0, n, squares=False)[0] - yr)
        y = _dev(y0)
        it, res = s.cg_solve(_dev(rhs), y, 0.0, n)
        dy = np.linalg.norm(y.cpu().numpy() - yr)
        print(f"[cg {amopi} {pos} n {n}] |dy| {dy / np.linalg.norm(yr):.1e} "
              f"own {own / np.linalg.norm(yr):.1e}", flush=True)
        assert it == n
        assert abs(res - resr[-1]) <= 1e-12 * resr[0]
        assert dy <= max(1e-12 * np.linalg.norm(yr), 10 * own)


@pytest.mark.parametrize("pos,precond", [("DQG", 0), ("DQG", 1), ("DQGT1", 0), ("DQGT2", 0)])
def test_no_iterations_leave_y_alone(pos, precond):
    """maxiter 0: y keeps every bit, whatever the right-hand side holds."""
    s, L = _pair([4], 2, 2, pos, True, True)
    rng = np.random.default_rng(8)
    y0 = rng.normal(size=L.ncon)
    y0[::7] = -0.0
    for bad in (1.0, np.inf, np.nan):
        rhs = rng.normal(size=L.ncon)
        rhs[::5] = bad
        y = _dev(y0)
        assert s.cg_solve(_dev(rhs), y, 1e-9, 0, precond=precond) == (0, 0.0)
        assert np.array_equal(y.cpu().numpy().view(np.int64), y0.view(np.int64)), bad


@pytest.mark.parametrize("amopi,na,nb,pos", [([5], 3, 2, "DQG"), ([5], 3, 2, "DQGT1"), ([5], 3, 2, "DQGT2"),
                                             ([2, 1, 1, 1], 3, 2, "DQGT1T2"), ([8, 6], 5, 5, "DQGT2")])
def test_capped_preconditioned_cg_matches_recurrence(amopi, na, nb, pos):
    """The general form with a diagonal, fused (D, Q, G and T2) and not (T1), same bounds."""
    s, L = _pair(amopi, na, nb, pos, True, True)
    rng = np.random.default_rng(9)
    rhs = L.Au(rng.normal(size=L.dimx))
    y0 = rng.normal(size=L.ncon)
    minv = rng.uniform(0.5, 2.0, size=L.ncon)
    s.set_precond_diag(_dev(minv))

    def plain(n, squares):
        y = y0.copy()
        r = rhs - L.Au(L.ATu(y))
        p = minv * r
        rz = r @ p
        for _ in range(n):
            t = L.ATu(p)
            ap = L.Au(t)
            alpha = rz / (t @ t if squares else p @ ap)
            y += alpha * p
            r = r - alpha * ap
            z = minv * r
            rz, old = r @ z, rz
            p = z + rz / old * p
        return y, np.linalg.norm(r)

    r0 = np.linalg.norm(rhs - L.Au(L.ATu(y0)))
    for n in (1, 2, 3):
        yr, resr = plain(n, True)
        own = np.linalg.norm(plain(n, False)[0] - yr)
        y = _dev(y0)
        it, res = s.cg_solve(_dev(rhs), y, 0.0, n, precond=2)
        assert it == n
        assert abs(res - resr) <= 1e-12 * max(r0, resr)
        assert np.linalg.norm(y.cpu().numpy() - yr) <= max(1e-12 * np.linalg.norm(yr), 10 * own)


@pytest.mark.parametrize("amopi,na,nb,pos", [([5], 2, 2, "DQG"), ([5], 3, 2, "DQG"), ([5], 2, 2, "DG"),
                                             ([2, 0, 1, 1, 0, 2, 1, 1], 5, 5, "DQG")])
def test_cg_past_its_last_digit_stays_finite(amopi, na, nb, pos):
    """A A^T is singular: iterations beyond the solution's last digit run along directions that
    A^T maps to zero, where ||A^T p||^2 is what rounding leaves of it.  As a sum of squares that
    is (eps ||p||)^2, and y stays finite; a difference of squares can be zero or negative."""
    s, L = _pair(amopi, na, nb, pos, True, True)
    rng = np.random.default_rng(1)
    rhs = L.Au(rng.normal(size=L.dimx))
    for n in (150, 250, 400):
        y = _dev(np.zeros(L.ncon))
        it, res = s.cg_solve(_dev(rhs), y, 0.0, n)
        print(f"[cg {amopi} {pos} n {n}] |r| {res:.1e} |y| {float(y.norm()):.1e}", flush=True)
        assert it == n and np.isfinite(res)
        assert bool(torch.isfinite(y).all())
