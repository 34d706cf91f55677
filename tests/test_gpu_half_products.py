"""Krylov products from half the blocks of S: block orders whose rows fill waves
and not, one and several objects a workgroup, objects that scatter nothing and
objects of very different sizes (whose pairs read the block of the larger)."""
import numpy as np
import pytest

from optimet_amd.problem import Cluster

pytestmark = pytest.mark.gpu

NM = 1e-9


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def lattice(P, nmax):
    """Weakly scattering spheres on a lattice, radii 2 to 60 nm, every fifth one of
    the background's permittivity."""
    rng = np.random.default_rng(P)
    m = int(np.ceil(P ** (1 / 3)))
    xyz = 400 * NM * np.array([(i, j, k) for i in range(m) for j in range(m) for k in range(m)][:P], float)
    eps = np.where(np.arange(P) % 5 == 4, 1.0, 2.25) + 0j
    return Cluster(xyz=xyz + 60 * NM * rng.random((P, 3)), radius=NM * np.where(np.arange(P) % 3 == 0, 2.0, 60.0) *
                   (0.8 + 0.2 * rng.random(P)), eps_r=eps, eps_r_sh=eps, nmax=nmax, wavelength=700 * NM, sh=False)


# N = 2 P nmax (nmax + 2) from 8192 on: n = 6, 30, 70, 126 (P > 64: eight objects a
# workgroup), 160, 240
@pytest.mark.parametrize("P,nmax", [(1366, 1), (275, 3), (118, 5), (66, 7), (52, 8), (35, 10)])
@pytest.mark.parametrize("kind", ["gmres64", "gmres32ir"])
def test_matches_the_factorisation(P, nmax, kind):
    """A residual of 1e-12 leaves the condition number, a few units, times it: 1e-10."""
    from optimet_amd import solver
    c = lattice(P, nmax)
    assert c.N >= 8192
    ref = solver.Solver(c, kind="lu64")
    ref.update()
    want = ref.solve()["x_sca"]
    s = solver.Solver(c, kind=kind, tol=1e-12)
    s.update()
    got = s.solve()["x_sca"]
    st = s.stats()
    assert st["residual"] <= 1e-12 and 0 < st["iterations"] < 60
    assert rel(got, want) < 1e-10
