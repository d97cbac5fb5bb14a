"""The work that a user of this framework has it do, as cases that can be timed.

Every case goes through the public entry points of V2RDMSolver and BatchSolver.
Five kinds of call make up that work:

  maps   A x and A^T y, one call each (the drop-in seams bpsdp_Au / bpsdp_ATu)
  cg     one solve of A A^T y = rhs, to a tolerance or an iteration cap
         (CGSolver::solve)
  split  converged per-block eigen splits (Update_xz), one after the other
  outer  some outer iterations of a solve that has settled, where a run spends
         nearly all of its thousands of iterations (compute_energy up to
         MAXITER, as a program calls it that looks in between)
  batch  the same for many problems in one batch (bond scans)

Active spaces are those of the repository's tests and benchmark, or generic.
All values are float64.  Linear solves are capped at CG_MAXITER = 12 or fewer
iterations, the setting for cheap inexact steps: later CG iterates lose their
orthogonality and amplify any change of rounding without bound, so that two
correct programs no longer agree on them.  For the same reason the outer cases
start near a solution that is known by construction: one tracking sweep far
from a diagonal matrix amplifies rounding just as much.
"""
import math

import numpy as np
import torch

from v2rdm_casscf_amd import V2RDMSolver
from v2rdm_casscf_amd.batch import BatchSolver

DEVICE = "cuda:0"
N2 = "2,0,1,1,0,2,1,1"
CHAINS = (8, 10, 12, 14, 16)


def _chain(n):
    """Orbitals per irrep of a hydrogen chain of n atoms in D2h."""
    return "%d,0,0,0,0,%d,0,0" % (n // 2, n // 2)


def listed():
    return [
        # one map pair on a valence active space: what a small drop-in call costs
        dict(name="maps_n2", kind="maps", amopi=N2, nalpha=5, nbeta=5, positivity="DQG"),
        # the same seams at the largest active space, where memory traffic counts
        dict(name="maps_h50", kind="maps", amopi=_chain(50), nalpha=25, nbeta=25, positivity="DQG"),
        # three-particle conditions: most rows are T2 rows, A^T scatters
        dict(name="maps_c10_t2", kind="maps", amopi="10", nalpha=5, nbeta=5, positivity="DQGT2"),
        # a linear solve inside a small external outer loop: latency and launches
        dict(name="cg_n2", kind="cg", amopi=N2, nalpha=5, nbeta=5, positivity="DQG",
             precond=0, tol=1e-4, maxiter=12),
        # an odd open-shell space without symmetry, with the Jacobi option
        dict(name="cg_c15_triplet_jacobi", kind="cg", amopi="15", nalpha=9, nbeta=7,
             positivity="DQG", precond=1, tol=1e-4, maxiter=12),
        # the linear solve that dominates large closed-shell runs
        dict(name="cg_h50", kind="cg", amopi=_chain(50), nalpha=25, nbeta=25, positivity="DQG",
             precond=0, tol=1e-4, maxiter=10),
        # the linear solve under the strongest conditions that are run in earnest
        dict(name="cg_c12_t2", kind="cg", amopi="12", nalpha=6, nbeta=6, positivity="DQGT2",
             precond=0, tol=1e-3, maxiter=12),
        # the projection of a mid-sized space, called from a program's own loop
        dict(name="split_c18", kind="split", amopi="18", nalpha=9, nbeta=9, positivity="DQG"),
        # outer iterations of the smallest space: its blocks are all 64 wide or less
        dict(name="outer_n2", kind="outer", amopi=N2, nalpha=5, nbeta=5, positivity="DQG",
             maxiter=12, steps=10),
        # outer iterations without symmetry: one 1152-wide block leads the split
        dict(name="outer_c24", kind="outer", amopi="24", nalpha=12, nbeta=12, positivity="DQG",
             maxiter=12, steps=3),
        # the headline: outer iterations of (50e,50o)
        dict(name="outer_h50", kind="outer", amopi=_chain(50), nalpha=25, nbeta=25,
             positivity="DQG", maxiter=12, steps=2),
        # a bond scan of 64 chains of 8 to 16 atoms in one batch
        dict(name="batch_64", kind="batch", count=64, sizes_seed=0, maxiter=12, steps=4),
    ]


def _spread(rng, orbitals, irreps):
    """orbitals dealt unevenly to the irreps of a group (some may stay empty)."""
    n = [0] * irreps
    for _ in range(orbitals):
        n[int(irreps * rng.random() ** 1.5)] += 1
    return ",".join(map(str, n))


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("maps", "cg", "cg", "split", "outer", "outer", "batch"))
    if kind == "batch":
        return dict(kind="batch", count=_log(rng, 2, 64), sizes_seed=rng.randrange(1000),
                    maxiter=rng.randrange(8, 13), steps=rng.randrange(2, 5))
    t2 = kind in ("maps", "cg") and rng.random() < 0.25
    irreps = rng.choice((1, 2, 4, 8))
    if t2:
        n = _log(rng, 5, 12)
    elif kind == "split":
        n = _log(rng, 6, 18)
    else:
        n = _log(rng, 6, (24, 32, 36, 40)[(1, 2, 4, 8).index(irreps)])
    ne = rng.randrange(2, n)
    open_shell = rng.choice((0, 0, 0, 1, 2)) if ne < n - 1 else 0
    case = dict(kind=kind, amopi=_spread(rng, n, irreps), nalpha=ne // 2 + 1 + open_shell,
                nbeta=ne // 2 + 1, positivity="DQGT2" if t2 else rng.choice(("DQG", "DQG", "DQG", "DQ", "DG")))
    if kind == "cg":
        case.update(precond=0 if t2 else rng.choice((0, 0, 0, 1)), tol=10.0 ** -rng.randrange(1, 5), maxiter=rng.randrange(6, 13))
    if kind == "outer":
        case.update(maxiter=rng.randrange(8, 13), steps=rng.randrange(2, 5))
    return case


def _solver(case, options=None):
    return V2RDMSolver([int(v) for v in case["amopi"].split(",")], case["nalpha"], case["nbeta"],
                       positivity=case["positivity"], device=DEVICE, options=options)


def _randn(gen, n):
    return torch.randn(n, dtype=torch.float64, device=DEVICE, generator=gen)


def _vectors(case, seed, dimx, ncon, dims):
    """The inputs of a maps, cg or split case."""
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed))
    if case["kind"] == "maps":
        return dict(x=_randn(gen, dimx), y=_randn(gen, ncon))
    if case["kind"] == "cg":
        # rhs = A u of a primal vector u, as A (c - z) - tau mu (A x - b) is
        return dict(u=_randn(gen, dimx), y0=0.1 * _randn(gen, ncon))
    # split: x positive semidefinite of low rank, c and y a fraction of it, and a
    # second y a step further
    x = torch.empty(dimx, dtype=torch.float64, device=DEVICE)
    o = 0
    for n in dims:
        if n:
            g = _randn(gen, n * max(1, n // 4)).reshape(n, -1) / math.sqrt(n)
            x[o:o + n * n] = (g @ g.T).reshape(-1)
            o += n * n
    y = 0.05 * _randn(gen, ncon)
    return dict(x0=x, c=0.1 * _randn(gen, dimx), y0=y, y1=y + 0.002 * _randn(gen, ncon), mu=0.7)


def _settled(s, parts, gen):
    """Puts a problem with a known solution into solver s and returns a start
    near it.  Per block x = V diag(l+) V^T and z = V diag(-l-) V^T with one V (a
    few reflections), c = A^T y + z and b = A x make (x, z, y) optimal at mu = 1;
    the start is the optimum of a problem whose b is 1e-4 away."""
    xs, zs = [], []
    for n in (n for dims in parts for n in dims if n):
        w = torch.rand(n, dtype=torch.float64, device=DEVICE, generator=gen) + 0.1
        w[torch.rand(n, dtype=torch.float64, device=DEVICE, generator=gen) > 0.4] *= -1.0
        for out, d in ((xs, w.clamp(min=0.0)), (zs, (-w).clamp(min=0.0))):
            out.append(torch.diag(d))
        for _ in range(4):
            v = _randn(gen, n)
            v /= torch.linalg.vector_norm(v)
            for m in (xs[-1], zs[-1]):
                u = m @ v
                m -= 2.0 * (torch.outer(u, v) + torch.outer(v, u)) - 4.0 * torch.dot(u, v) * torch.outer(v, v)
        xs[-1], zs[-1] = xs[-1].reshape(-1), zs[-1].reshape(-1)
    x, z = torch.cat(xs), torch.cat(zs)
    if isinstance(s, BatchSolver):
        au, atu, ncon = s.Au, s.ATu, s.ncon
    else:
        ncon = s.nconstraints
        au = lambda v: s.bpsdp_Au(torch.empty(ncon, dtype=torch.float64, device=DEVICE), v)  # noqa: E731
        atu = lambda v: s.bpsdp_ATu(torch.empty(s.dimx, dtype=torch.float64, device=DEVICE), v)  # noqa: E731
    y = 0.05 * _randn(gen, ncon)
    s.c, s.b = atu(y) + z, au(x + 1e-4 * _randn(gen, s.dimx))
    s.x, s.z, s.y = x.clone(), z.clone(), y.clone()
    return [x, z, y]


def prepare(case, seed):
    kind = case["kind"]
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed))
    if kind == "batch":
        sizes = np.random.default_rng(case["sizes_seed"]).choice(np.array(CHAINS), case["count"])
        bs = BatchSolver([dict(amopi=[int(v) for v in _chain(n).split(",")], nalpha=int(n) // 2,
                               nbeta=int(n) // 2) for n in sizes], device=DEVICE,
                         options=dict(MAXITER=case["steps"], CG_MAXITER=case["maxiter"]))
        parts = [_chain_space(n).dims for n in map(int, sizes)]
        return dict(kind=kind, s=bs, start=_settled(bs, parts, gen))
    if kind == "outer":
        s = _solver(case, dict(MAXITER=case["steps"], CG_MAXITER=case["maxiter"]))
        return dict(kind=kind, s=s, start=_settled(s, [s.dimensions], gen))
    s = _solver(case)
    st = dict(kind=kind, s=s, **_vectors(case, seed, s.dimx, s.nconstraints, s.dimensions))
    new = lambda n: torch.empty(n, dtype=torch.float64, device=DEVICE)  # noqa: E731
    if kind == "maps":
        st.update(ax=new(s.nconstraints), aty=new(s.dimx))
    elif kind == "cg":
        rhs = s.bpsdp_Au(new(s.nconstraints), st.pop("u"))
        st.update(rhs=rhs, y=new(s.nconstraints), tol=case["tol"] * float(torch.linalg.vector_norm(rhs)),
                  precond=case["precond"], maxiter=case["maxiter"])
    else:
        st.update(x=[new(s.dimx), new(s.dimx)], z=[new(s.dimx), new(s.dimx)])
    return st


def run(st):
    s, kind = st["s"], st["kind"]
    if kind == "maps":
        return [s.bpsdp_Au(st["ax"], st["x"]), s.bpsdp_ATu(st["aty"], st["y"])]
    if kind == "cg":
        st["y"].copy_(st["y0"])
        iters, res = s.cg_solve(st["rhs"], st["y"], st["tol"], st["maxiter"], precond=st["precond"])
        return [st["y"], iters, res]
    if kind == "split":
        for k, y in enumerate((st["y0"], st["y1"])):
            st["x"][k].copy_(st["x0"])
            s.update_xz(st["mu"], y, st["c"], st["x"][k], st["z"][k])
        return st["x"] + st["z"]
    for v, w in zip((s.x, s.z, s.y), st["start"]):
        v.copy_(w)
    if kind == "outer":
        r = s.compute_energy(guess=False)
        return dict(x=s.x, z=s.z, y=s.y, **{k: r[k] for k in ("energy_primal", "energy_dual", "ep", "ed", "mu", "oiter", "cg_iters")})
    out = s.compute_energy()
    return dict(x=s.x, z=s.z, y=s.y, energy=np.array([r["energy_primal"] for r in out]),
                ep=np.array([r["ep"] for r in out]), ed=np.array([r["ed"] for r in out]),
                oiter=np.array([r["oiter"] for r in out]), cg_iters=np.array([r["cg_iters"] for r in out]))


# ---------------------------------------------------------------------------
# Sizes, and the constraint matrix in plain numpy (singlet or M_s = S, spin and
# S_z constrained; D, Q and G conditions)
# ---------------------------------------------------------------------------
class _Space:
    """Geminal numbering, primal blocks and row count of an active space."""

    def __init__(self, amopi, nalpha, nbeta, positivity):
        self.amopi, self.na, self.nb = amopi, nalpha, nbeta
        self.singlet = nalpha == nbeta
        self.q2, self.g2, self.t2 = "Q" in positivity, "G" in positivity, "T2" in positivity
        self.H = H = len(amopi)
        self.sym = np.repeat(np.arange(H), amopi)
        self.off = np.concatenate([[0], np.cumsum(amopi)])
        a = self.amo = int(sum(amopi))
        self.gab, self.gaa = np.full((a, a), -1), np.full((a, a), -1)
        self.ab, self.aa = [], []
        for h in range(H):
            # second orbital outer, first inner; like-spin pairs keep first > second
            sec, fir = np.nonzero((self.sym[:, None] ^ self.sym[None, :]) == h)
            self.ab.append((fir, sec))
            self.gab[fir, sec] = np.arange(len(fir))
            m = fir > sec
            self.aa.append((fir[m], sec[m]))
            self.gaa[fir[m], sec[m]] = self.gaa[sec[m], fir[m]] = np.arange(int(m.sum()))
        self.g = [len(f) for f, _ in self.ab]
        self.ga = [len(f) for f, _ in self.aa]
        n, g, ga = amopi, self.g, self.ga
        blocks = [("d2ab", g), ("d2aa", ga), ("d2bb", ga), ("d200", g if self.singlet else [2 * v for v in g]),
                  ("d1a", n), ("d1b", n), ("q1a", n), ("q1b", n)]
        if self.q2:
            blocks += [("q2ab", g), ("q2aa", ga), ("q2bb", ga)]
        if self.g2:
            blocks += [("g2ab", g), ("g2ba", g), ("g2aa", [2 * v for v in g])]
        if self.t2:
            s3 = [[int(v) for v in np.bincount(x, minlength=H)] for x in self._triplets()]
            big = [p + q for p, q in zip(*s3)]
            blocks += [("t2aaa", big), ("t2bbb", big), ("t2aab", s3[0]), ("t2bba", s3[0])]
        self.at, self.dims, o = {}, [], 0
        for name, d in blocks:
            for h in range(H):
                self.at[name, h] = o
                self.dims.append(d[h])
                o += d[h] ** 2
        self.dimx = o
        n2, g2s, ga2 = sum(v * v for v in n), sum(v * v for v in g), sum(v * v for v in ga)
        self.ncon = 3 + 6 * n2 + 1 + (n2 + 3 * ga2 + g2s if self.singlet else 4 * g2s)
        self.ncon += (2 * g[0] + 6 * g2s if self.g2 else 0) + (g2s + 2 * ga2 if self.q2 else 0)
        if self.t2:
            self.ncon += 2 * sum(p * p for p in big) + 2 * sum(p * p for p in s3[0])

    def _triplets(self):
        """Irreps of the triplets i < j, k and of all i, j, k."""
        s3 = self.sym[:, None, None] ^ self.sym[None, :, None] ^ self.sym[None, None, :]
        return s3[np.triu_indices(self.amo, 1)].reshape(-1), s3.reshape(-1)

    def matrix(self):
        """(rows, columns, values) of A."""
        R, C, V, at = [], [], [], self.at
        row = 0

        def put(r, c, v):
            r, c, v = np.broadcast_arrays(r, c, np.asarray(v, dtype=np.float64))
            R.append(r.reshape(-1)), C.append(c.reshape(-1)), V.append(v.reshape(-1))

        def base(name):
            return np.array([at[name, h] for h in range(self.H)])

        amopi, off, sym, gab, gaa = np.array(self.amopi), self.off, self.sym, self.gab, self.gaa
        g, ga, a = np.array(self.g), np.array(self.ga), self.amo

        def d1(name, p, q):
            h = sym[p]
            return base(name)[h] + (p - off[h]) * amopi[h] + (q - off[h])

        def d2ab(p, q, r, s):
            h = sym[p] ^ sym[q]
            return base("d2ab")[h] + gab[p, q] * g[h] + gab[r, s]

        def d2aa(name, p, q, r, s):
            h = sym[p] ^ sym[q]
            return base(name)[h] + gaa[p, q] * ga[h] + gaa[r, s], np.where((p < q) == (r < s), 1.0, -1.0)

        p, q = (v.reshape(-1) for v in np.meshgrid(np.arange(a), np.arange(a), indexing="ij"))
        ne = p != q
        # traces
        put(0, d2ab(p, q, p, q), 1.0)
        for k, nm in ((1, "d2aa"), (2, "d2bb")):
            put(k, d2aa(nm, p[ne], q[ne], p[ne], q[ne])[0], 1.0)
        row = 3
        # D1 + Q1
        for dn, qn in (("d1a", "q1a"), ("d1b", "q1b")):
            for h, n in enumerate(self.amopi):
                i, j = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
                r = row + i * n + j
                put(r, at[dn, h] + j * n + i, 1.0)
                put(r, at[qn, h] + i * n + j, 1.0)
                row += n * n
        # contractions D2 -> D1
        for kind, (dn, cf) in enumerate((("d1a", self.nb), ("d1b", self.na), ("d1a", self.na - 1.0), ("d1b", self.nb - 1.0))):
            for h, n in enumerate(self.amopi):
                i, j = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
                r = row + i * n + j
                put(r, at[dn, h] + i * n + j, cf)
                if n:
                    i3, j3, k = np.broadcast_arrays((i + off[h])[..., None], (j + off[h])[..., None], np.arange(a))
                    r3 = np.broadcast_to(r[..., None], k.shape)
                    if kind < 2:
                        put(r3, d2ab(i3, k, j3, k) if kind == 0 else d2ab(k, i3, k, j3), -1.0)
                    else:
                        m = (i3 != k) & (j3 != k)
                        c, sg = d2aa("d2aa" if kind == 2 else "d2bb", i3[m], k[m], j3[m], k[m])
                        put(r3[m], c, -sg)
                row += n * n
        # S^2
        put(row, d2ab(p, q, q, p), 1.0)
        row += 1
        r2 = math.sqrt(2.0)
        pairs = []     # per irrep: bra p, q, ket r, s of the ab pairs, and their entry numbers
        for h in range(self.H):
            f, s = self.ab[h]
            e = np.arange(g[h] ** 2).reshape(g[h], g[h])
            pairs.append(tuple(np.broadcast_to(v, e.shape) for v in (f[:, None], s[:, None], f[None], s[None])) + (e,))
        like = []
        for h in range(self.H):
            f, s = self.aa[h]
            e = np.arange(ga[h] ** 2).reshape(ga[h], ga[h])
            like.append(tuple(np.broadcast_to(v, e.shape) for v in (f[:, None], s[:, None], f[None], s[None])) + (e,))
        if self.singlet:
            for h, n in enumerate(self.amopi):
                e = np.arange(n * n)
                put(row + e, at["d1a", h] + e, 1.0)
                put(row + e, at["d1b", h] + e, -1.0)
                row += n * n
            for h in range(self.H):
                e = np.arange(ga[h] ** 2)
                put(row + e, at["d2aa", h] + e, 1.0)
                put(row + e, at["d2bb", h] + e, -1.0)
                row += ga[h] ** 2
            for nm in ("d2aa", "d2bb"):
                for h in range(self.H):
                    i, j, k, l, e = like[h]
                    put(row + e, at[nm, h] + e, 1.0)
                    for c, v in ((d2ab(i, j, k, l), -0.5), (d2ab(j, i, k, l), 0.5), (d2ab(i, j, l, k), 0.5), (d2ab(j, i, l, k), -0.5)):
                        put(row + e, c, v)
                    row += ga[h] ** 2
        for h in range(self.H):
            i, j, k, l, e = pairs[h]
            w = 0.5 / (np.where(i == j, r2, 1.0) * np.where(k == l, r2, 1.0))
            cols = (d2ab(i, j, k, l), d2ab(j, i, k, l), d2ab(i, j, l, k), d2ab(j, i, l, k))
            G = int(g[h])
            if self.singlet:
                quads = (((0, 0), (-w, -w, -w, -w)),)
            else:
                wi, wk, half = 0.5 / np.where(i == j, r2, 1.0), 0.5 / np.where(k == l, r2, 1.0), 0.5
                quads = (((0, 0), (-w, -w, -w, -w)), ((0, 1), (-wi, -wi, wi, wi)), ((1, 0), (-wk, wk, -wk, wk)), ((1, 1), (-half, half, half, -half)))
                G *= 2
            ij, kl = e // max(1, int(g[h])), e % max(1, int(g[h]))
            for (qa, qb), vs in quads:
                x = (ij + qa * g[h]) * G + kl + qb * g[h]
                put(row + x, at["d200", h] + x, 1.0)
                for c, v in zip(cols, vs):
                    put(row + x, c, v)
            row += G * G
        if self.g2:
            d = np.arange(a)
            for o in range(2):
                kl, i = np.meshgrid(np.arange(g[0]), d, indexing="ij")
                ii = gab[i, i]
                put(row + kl, at["g2ba", 0] + (kl * g[0] + ii if o == 0 else ii * g[0] + kl), 1.0)
                row += int(g[0])
        if self.q2:
            for h in range(self.H):
                i, j, k, l, e = pairs[h]
                put(row + e, at["d2ab", h] + e, 1.0)
                put(row + e, at["q2ab", h] + e, -1.0)
                m = j == l
                put(row + e[m], d1("d1a", k[m], i[m]), -1.0)
                m = i == k
                put(row + e[m], d1("d1b", l[m], j[m]), -1.0)
                row += int(g[h]) ** 2
            for d2n, q2n, dn in (("d2aa", "q2aa", "d1a"), ("d2bb", "q2bb", "d1b")):
                for h in range(self.H):
                    i, j, k, l, e = like[h]
                    put(row + e, at[d2n, h] + e, 1.0)
                    put(row + e, at[q2n, h] + e, -1.0)
                    for m, x, y, v in ((j == l, k, i, -1.0), (j == k, l, i, 1.0), (i == l, k, j, 1.0), (i == k, l, j, -1.0)):
                        put(row + e[m], d1(dn, x[m], y[m]), v)
                    row += int(ga[h]) ** 2
        if self.g2:
            for o, (g2n, dn) in enumerate((("g2ab", "d1a"), ("g2ba", "d1b"))):
                for h in range(self.H):
                    i, j, k, l, e = pairs[h]
                    put(row + e, at[g2n, h] + e, -1.0)
                    m = j == l
                    put(row + e[m], d1(dn, i[m], k[m]), 1.0)
                    put(row + e, d2ab(i, l, k, j) if o == 0 else d2ab(l, i, j, k), -1.0)
                    row += int(g[h]) ** 2
            for h in range(self.H):
                i, j, k, l, e = pairs[h]
                G = int(g[h])
                ij, kl = e // max(1, G), e % max(1, G)
                for qa in range(2):
                    for qb in range(2):
                        x = (ij + qa * G) * 2 * G + kl + qb * G
                        put(row + x, at["g2aa", h] + x, -1.0)
                        if qa == qb:
                            m = j == l
                            put(row + x[m], d1("d1b" if qa else "d1a", i[m], k[m]), 1.0)
                            m = (i != l) & (k != j)
                            c, sg = d2aa("d2bb" if qa else "d2aa", i[m], l[m], k[m], j[m])
                            put(row + x[m], c, -sg)
                        else:
                            put(row + x, d2ab(l, i, k, j) if qa else d2ab(i, l, j, k), 1.0)
                row += 4 * G * G
        assert row == self.ncon
        return np.concatenate(R), np.concatenate(C), np.concatenate(V)


def _space(case):
    return _Space([int(v) for v in case["amopi"].split(",")], case["nalpha"], case["nbeta"], case["positivity"])


def _chain_space(n):
    return _Space([n // 2, 0, 0, 0, 0, n // 2, 0, 0], n // 2, n // 2, "DQG")


def work(case):
    """Bytes of inputs and outputs, and the operations of the method: one
    multiply and add per matrix element and product, a product with A and one
    with A^T per iteration of a linear solve, (16/3) n^3 per n x n eigen split."""
    if case["kind"] == "batch":
        sizes = np.random.default_rng(case["sizes_seed"]).choice(np.array(CHAINS), case["count"])
        spaces = [_chain_space(n) for n in map(int, sizes)]
    else:
        spaces = [_space(case)]
    steps, dimx, ncon = case.get("steps", 1), sum(s.dimx for s in spaces), sum(s.ncon for s in spaces)
    product, split = 2.0 * 4 * ncon, sum(16.0 / 3.0 * float(n) ** 3 for s in spaces for n in s.dims)
    if case["kind"] == "maps":
        return dict(bytes=16.0 * (dimx + ncon), flops=2 * product)
    if case["kind"] == "cg":
        return dict(bytes=24.0 * ncon, flops=2 * case["maxiter"] * product)
    if case["kind"] == "split":
        return dict(bytes=2 * 8.0 * (4 * dimx + ncon), flops=2 * split)
    return dict(bytes=8.0 * (5 * dimx + 3 * ncon), flops=steps * (2 * case["maxiter"] * product + split))


def exact(case, seed):
    """maps, cg and split up to about a million unknowns; the D, Q, G
    conditions only."""
    if case["kind"] not in ("maps", "cg", "split"):
        return None
    sp = _space(case)
    if sp.t2 or sp.dimx > 1_200_000:
        return None
    r, c, v = (torch.from_numpy(np.ascontiguousarray(t)).to(DEVICE) for t in sp.matrix())
    st = _vectors(case, seed, sp.dimx, sp.ncon, sp.dims)

    def au(x):
        return torch.zeros(sp.ncon, dtype=torch.float64, device=DEVICE).index_add_(0, r, v * x[c])

    def atu(y):
        return torch.zeros(sp.dimx, dtype=torch.float64, device=DEVICE).index_add_(0, c, v * y[r])

    if case["kind"] == "maps":
        return [au(st["x"]), atu(st["y"])]
    if case["kind"] == "cg":
        rhs, y = au(st["u"]), st["y0"].clone()
        tol = case["tol"] * float(torch.linalg.vector_norm(rhs))
        # squared row norms; a column that a row names twice counts once
        key, at = torch.unique(r * sp.dimx + c, return_inverse=True)
        val = torch.zeros(len(key), dtype=torch.float64, device=DEVICE).index_add_(0, at, v)
        n2 = torch.zeros(sp.ncon, dtype=torch.float64, device=DEVICE).index_add_(0, key // sp.dimx, val * val)
        minv = torch.where(n2 > 0, 1.0 / n2, torch.ones_like(n2)) if case["precond"] else torch.ones_like(n2)
        res = rhs - au(atu(y))
        p = minv * res
        rz, it = torch.dot(res, p), 0
        while it < case["maxiter"]:
            ap = au(atu(p))
            alpha = rz / torch.dot(p, ap)
            y += alpha * p
            res -= alpha * ap
            norm = float(torch.linalg.vector_norm(res))
            if norm < tol:
                break
            rz, old = torch.dot(res, minv * res), rz
            p = minv * res + rz / old * p
            it += 1
        return [y, it, norm]
    out = []
    for y in (st["y0"], st["y1"]):
        full = atu(y) - st["c"] + st["mu"] * st["x0"]
        x, z, o = torch.empty_like(full), torch.empty_like(full), 0
        for n in sp.dims:
            m = full[o:o + n * n].reshape(n, n).cpu()
            m = 0.5 * (m + m.T)
            w, u = torch.linalg.eigh(m)
            xb = (u * (w.clamp(min=0.0) / st["mu"])) @ u.T
            x[o:o + n * n] = xb.reshape(-1).to(DEVICE)
            z[o:o + n * n] = (st["mu"] * xb - m).reshape(-1).to(DEVICE)
            o += n * n
        out.append((x, z))
    return [out[0][0], out[1][0], out[0][1], out[1][1]]
