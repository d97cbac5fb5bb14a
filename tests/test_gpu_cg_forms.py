"""Edges of the CG's calls on single handles (cg_solver.cc:125-177)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle_py as orc  # noqa: E402

pytestmark = pytest.mark.gpu


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _pair(amopi, na, nb, pos, sz, spin):
    from v2rdm_casscf_amd import V2RDMSolver
    s = V2RDMSolver(amopi, na, nb, na - nb + 1, pos, constrain_sz=sz, constrain_spin=spin)
    return s, orc.Layout(amopi, na, nb, na - nb + 1, pos, constrain_sz=sz, constrain_spin=spin)


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
