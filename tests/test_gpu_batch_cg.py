"""One outer iteration of a batch, problem by problem, against the plain recurrence of
CGSolver::solve (cg_solver.cc:125-177) on the oracle's maps and the oracle's Update_xz.

The CG is capped after n iterations, so that y is a given iterate and not a solution that
any path reaches.  y agrees to 1e-12, or ten times what the recurrence's own two forms
(p.A A^T p and ||A^T p||^2) differ by where that is more; the split of that y to 1e-10, as
the other splits, and what the difference of the two y makes of it.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import fci_tools as ft  # noqa: E402
import oracle_py as orc  # noqa: E402

pytestmark = pytest.mark.gpu

C1 = dict(amopi=[5], nalpha=3, nbeta=2)
D2H = dict(amopi=[2, 0, 1, 1, 0, 2, 1, 1], nalpha=5, nbeta=5)
SMALL = dict(amopi=[3], nalpha=2, nbeta=1)

BATCHES = {
    # batches of the general form: rows of a segment above one tile's 256, a problem in
    # front of others, D, Q, G problems beside those that send the batch there
    "t2": [dict(C1, positivity="DQGT2"), dict(amopi=[6], nalpha=3, nbeta=3, positivity="DQGT2")],
    "t1 and plain": [D2H, dict(C1, positivity="DQGT1"), dict(amopi=[9], nalpha=4, nbeta=4)],
    "spin adapted": [dict(amopi=[5], nalpha=2, nbeta=2, spin_adapt_q2=True), C1,
                     dict(D2H, constrain_spin=False, spin_adapt_q2=True, spin_adapt_g2=True)],
    # batches of the reduced form: closed shells with every condition, and one problem or
    # more without, which takes all of the batch to the kernels that ask the layout
    "reduced": [dict(amopi=[4], nalpha=2, nbeta=2), D2H, dict(amopi=[7], nalpha=3, nbeta=3)],
    "reduced, mixed": [D2H, C1, dict(amopi=[3, 2], nalpha=3, nbeta=2, positivity="DQ"),
                       dict(amopi=[5], nalpha=2, nbeta=2, positivity="DG"),
                       dict(amopi=[4], nalpha=3, nbeta=1, positivity="DG", constrain_spin=False),
                       dict(amopi=[0, 3, 2, 1], nalpha=3, nbeta=1, constrain_sz=False),
                       dict(amopi=[6], nalpha=4, nbeta=2), dict(amopi=[7], nalpha=3, nbeta=3)],
}


def _layout(pb):
    kw = {k: v for k, v in pb.items() if k not in ("amopi", "nalpha", "nbeta", "positivity")}
    return orc.Layout(pb["amopi"], pb["nalpha"], pb["nbeta"], None, pb.get("positivity", "DQG"), **kw)


def _plain(L, rhs, y0, n, squares):
    y = y0.copy()
    r = rhs - L.Au(L.ATu(y))
    p, rz = r.copy(), r @ r
    for _ in range(n):
        t = L.ATu(p)
        ap = L.Au(t)
        alpha = rz / (t @ t if squares else p @ ap)
        y += alpha * p
        r = r - alpha * ap
        rz, old = r @ r, rz
        p = r + rz / old * p
    return y


def _norm(v):
    return np.linalg.norm(v)


def _run(probs, which, n):
    from v2rdm_casscf_amd.batch import BatchSolver
    bs = BatchSolver(probs, options=dict(MAXITER=1, CG_MAXITER=n, CG_CONVERGENCE=0.0))
    Ls = {q: _layout(probs[q]) for q in which}
    ham = {}
    h1s, eris = [], []
    for pb in probs:
        key = tuple(pb["amopi"])
        if key not in ham:
            irreps = [h for h, k in enumerate(pb["amopi"]) for _ in range(k)]
            ham[key] = ft.random_hamiltonian(sum(key), 3, irreps if len(key) > 1 else None)
        h1s.append(ham[key][0])
        eris.append(ham[key][1])
    bs.set_integrals(h1s, eris)
    before = {q: [bs.x_of(q, v).cpu().numpy() for v in (bs.c, bs.x, bs.z)]
              + [bs.y_of(q, v).cpu().numpy() for v in (bs.b, bs.y)] for q in which}
    st = bs.compute_energy()
    for q in which:
        L = Ls[q]
        c, x0, z0, b, y0 = before[q]
        rhs = L.Au(c - z0) - (L.Au(x0) - b)
        yr = _plain(L, rhs, y0, n, False)
        own = _norm(_plain(L, rhs, y0, n, True) - yr)
        y = bs.y_of(q).cpu().numpy()
        print(f"[batch cg] problem {q} {probs[q]} n {n} |dy| {_norm(y - yr) / _norm(yr):.1e} "
              f"own {own / _norm(yr):.1e}", flush=True)
        assert st[q]["cg_iters"] == n
        assert _norm(y - yr) <= max(1e-12 * _norm(yr), 10 * own)
        xr, zr = L.update_xz(1.0, y, c, x0)
        assert _norm(bs.x_of(q).cpu().numpy() - xr) < 1e-10 * _norm(xr)
        assert _norm(bs.x_of(q, bs.z).cpu().numpy() - zr) < 1e-10 * _norm(zr)


@pytest.mark.parametrize("n", [1, 4])
@pytest.mark.parametrize("name", BATCHES, ids=str)
def test_batch_iteration_matches_recurrence(name, n):
    probs = BATCHES[name]
    _run(probs, range(len(probs)), n)


def test_batch_of_many_problems():
    """More problems than the reduced form of the CG takes in one batch (1 024)."""
    _run([SMALL] * 1025, (0, 511, 1024), 3)


def test_batch_of_many_mid_sized_blocks():
    """More blocks of 33 to 64 indices in a launch than its 1 024-thread workgroups take
    (kFewMid, 512): even and odd sizes from 33 to 64, with 256 threads each."""
    probs = ([dict(amopi=[5, 4], nalpha=4, nbeta=4)] * 50 + [dict(amopi=[6], nalpha=3, nbeta=3)]
             + [dict(amopi=[7], nalpha=4, nbeta=3), dict(amopi=[8], nalpha=4, nbeta=4),
                dict(amopi=[11, 3], nalpha=4, nbeta=4, positivity="D"),
                dict(amopi=[9, 7], nalpha=4, nbeta=4, positivity="D")]
             + [dict(amopi=[7], nalpha=3, nbeta=3)] * 10)
    mid = [n for pb in probs for n in _layout(pb).block_dims if 32 < n <= 64]
    assert len(mid) > 512 and {33, 36, 40, 41, 49, 57, 63, 64} <= set(mid)
    _run(probs, (0, 49, 50, 51, 52, 53, 54, 64), 2)
