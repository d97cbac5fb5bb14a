"""Update_xz of small blocks at the edges of their kernels: 256 threads up to 32 indices,
1 024 up to 64 (256 where a launch has more than 512 such blocks: test_gpu_batch_cg.py),
the block Jacobi above; odd sizes, a block of one index, matrices whose
squares leave the range of the fast rotation, and ones with nothing to rotate.  Against the
oracle (LAPACK), 1e-10 relative, as the other splits."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda:0")


def _rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


# sizes: D1 n, D2ab sums of products, D2aa sums of n (n - 1) / 2 by symmetry
@pytest.mark.parametrize("amopi", [
    [1], [2],             # 1, 2, 4
    [3], [4], [5],        # 3, 9, 6, 16, 10, 25
    [4, 4],               # 32
    [8, 3],               # 31, 73, 24 + 24
    [11, 3],              # 33, 66, 130 (a padded one of 192)
    [9, 7],               # 63, 57, 130
    [8],                  # 28, 64
], ids=str)
@pytest.mark.parametrize("scale", [1.0, 1e-150, 1e145, 0.0], ids=str)
def test_split_at_kernel_edges(amopi, scale):
    import oracle_py as orc
    from v2rdm_casscf_amd import V2RDMSolver
    amopi = amopi + [0] * (8 - len(amopi)) if len(amopi) > 1 else amopi
    na = max(1, sum(amopi) // 2)
    L = orc.Layout(amopi, na, na, 1, "D")
    s = V2RDMSolver(amopi, na, na, 1, "D")
    rng = np.random.default_rng(17)
    if scale == 0.0:      # diagonal M: no rotation anywhere
        y, c = np.zeros(L.ncon), np.zeros(L.dimx)
        x0 = np.concatenate([np.diag(rng.normal(size=n)).ravel() for n in L.block_dims])
    else:
        y, c, x0 = (scale * rng.normal(size=k) for k in (L.ncon, L.dimx, L.dimx))
    x, z = _dev(x0), _dev(np.zeros(L.dimx))
    xr = x0
    for _ in range(2):    # the second call starts from the first one's eigenvectors
        xr, zr = L.update_xz(0.8, y, c, xr)
        s.update_xz(0.8, _dev(y), _dev(c), x, z)
        assert _rel(x.cpu().numpy(), xr) < 1e-10
        # z may vanish (mu x = M): its error is relative to M, as M's two parts are
        assert np.linalg.norm(z.cpu().numpy() - zr) < 1e-10 * np.hypot(np.linalg.norm(zr), 0.8 * np.linalg.norm(xr))
        y = y + 1e-3 * scale * rng.normal(size=L.ncon)
