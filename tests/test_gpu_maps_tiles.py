"""A.x and A^T.y where the work is dealt out otherwise than in the small layouts: G2 blocks visited
by tiles (from 512 pairs on), several items a thread (from two million rows on), T2 rows in
several chunks of columns.  Against the oracle, 1e-12 relative as the other maps."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda:0")


@pytest.mark.parametrize("amopi,na,nb,mult,pos", [
    ([23], 4, 4, 1, "DQG"),                # 529 pairs: one tile row short of full, 2.7 million rows
    ([24, 9], 4, 4, 1, "DG"),              # 657 and 432 pairs: one irrep by tiles, one not
    ([12], 4, 3, 2, "DQGT2"),              # aba triplets in two chunks
    ([3, 0, 1, 1, 0, 2, 1, 1], 4, 3, 2, "DQGT2"),
], ids=str)
def test_maps_match_oracle(amopi, na, nb, mult, pos):
    import oracle_py as orc
    from v2rdm_casscf_amd import V2RDMSolver
    L = orc.Layout(amopi, na, nb, mult, pos)
    s = V2RDMSolver(amopi, na, nb, mult, pos)
    rng = np.random.default_rng(23)
    x, y = rng.normal(size=L.dimx), rng.normal(size=L.ncon)
    ax, aty = _dev(np.full(L.ncon, np.nan)), _dev(np.full(L.dimx, np.nan))
    s.bpsdp_Au(ax, _dev(x))
    s.bpsdp_ATu(aty, _dev(y))
    for got, ref in ((ax, L.Au(x)), (aty, L.ATu(y))):
        assert np.linalg.norm(got.cpu().numpy() - ref) < 1e-12 * np.linalg.norm(ref)
