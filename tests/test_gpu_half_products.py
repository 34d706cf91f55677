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


def test_tiny_size_parameters():
    """Size parameters of 2e-10, where the factors of degree 8 are about 1e-179 and
    their squares 0: every degree's coefficients, against the fixed point of x = Q
    - (S - 1) x on the host (the spheres couple weakly: a hundredth a step).  The
    high degrees come from their neighbours' fields alone, so a product that loses
    a row's blocks is wrong by its own size there; 1e-6 is far from that and from
    the rounding of a few Krylov steps."""
    from optimet_amd import solver
    P, nmax = 52, 8
    rng = np.random.default_rng(0)
    xyz = 400 * NM * np.array([(i, j, k) for i in range(4) for j in range(4) for k in range(4)][:P], float)
    eps = np.full(P, 2.25 + 0j)
    c = Cluster(xyz=xyz + 60 * NM * rng.random((P, 3)), radius=60 * NM * (0.8 + 0.2 * rng.random(P)), eps_r=eps,
                eps_r_sh=eps, nmax=nmax, wavelength=2 * np.pi * 60 * NM / 2e-10, sh=False)
    assert c.N >= 8192
    s = solver.Solver(c, kind="gmres64", tol=1e-14)
    s.update()
    S, Q = s.matrix(), s.vector("Q")
    want = Q
    for _ in range(12):
        want = Q - (S @ want - want)
    got = s.solve()["x_sca"]
    p = np.arange(2 * c.nf)
    deg = np.tile(np.sqrt(p % c.nf + 1.0).astype(int), P)
    pol = np.tile(p // c.nf, P)
    for n in range(1, nmax + 1):
        for q in (0, 1):
            k = (deg == n) & (pol == q)
            d = got[k] / np.abs(want[k]).max() - want[k] / np.abs(want[k]).max()
            assert np.abs(d).max() < 1e-6, (n, q, np.abs(d).max())


@pytest.mark.parametrize("P,nmax,kind,half", [(1366, 1, "gmres64", False), (512, 2, "gmres64", True),
                                              (275, 3, "gmres64", True), (66, 7, "gmres64", True)])
def test_orders_that_gain(P, nmax, kind, half):
    """Blocks of order 6 are read whole (their half takes four times as long), the
    others from half of them: by the bytes that the products count, 16 N^2 each or
    half of it in the Arnoldi steps.  The cycle's residuals are whole products: two
    of them beside 5 or more steps."""
    from optimet_amd import solver
    s = solver.Solver(lattice(P, nmax), kind=kind, tol=1e-12)
    s.update()
    s.ctx.set_profile(True)
    s.solve()
    st = s.stats()
    per = st["matvec_bytes"] / (16.0 * st["Np"] ** 2 * st["matvec_calls"])
    assert st["matvec_calls"] >= 7
    assert abs(per - 1.0) < 1e-12 if not half else 0.5 <= per < 0.7


def test_without_memory_for_the_scratch():
    """With the device's memory taken, all but 64 to 128 MB, the scratch of these
    products (300 MB) does not fit and they read the whole matrix: the solve goes
    through, with the solution of one that had the memory (1e-10, as above)."""
    from optimet_amd import solver
    from tests.test_zz_no_alloc import _Dev, _hip
    hip = _hip()
    c = lattice(1366, 2)
    a, b = solver.Solver(c, kind="gmres64", tol=1e-12), solver.Solver(c, kind="gmres64", tol=1e-12)
    a.update()
    want = a.solve()["x_sca"]
    b.update()
    b.vector("Q")
    held, size = [], 16 << 30
    try:
        while size >= 64 << 20:
            try:
                held.append(_Dev(hip, size))
            except AssertionError:
                size //= 2
        held.pop().free()
        got = b.solve()["x_sca"]
    finally:
        for d in held:
            d.free()
    assert rel(got, want) < 1e-10
    a.ctx.close()
    b.ctx.close()


def test_second_harmonic_operator():
    """V's inner products by the mixed Krylov read half of V's blocks, with the factors
    of the second harmonic: an outer step gains the six digits of an inner solve with
    the right operator, two to three steps to 1e-12, and one to two digits with the
    factors of S or another sign, five steps or more."""
    from optimet_amd import solver
    c = lattice(66, 7)
    c.sh = True
    c.eps_r, c.eps_r_sh = np.full(66, 2.25 + 0j), np.full(66, 3.0 + 0j)
    c.ksippp, c.ksiparppar, c.gamma = np.full(66, 1e-18 + 0j), np.full(66, 3e-19 + 0j), np.full(66, 1e-19 + 0j)
    assert c.N >= 8192
    ref = solver.Solver(c, kind="lu64")
    ref.update()
    want = ref.solve()
    s = solver.Solver(c, kind="gmres32ir", tol=1e-12)
    s.update()
    got = s.solve()
    st = s.stats()
    assert st["residual_sh"] <= 1e-12 and 0 < st["iterations_sh"] <= 3
    for k in ("x_sca", "x_sca_sh"):
        assert rel(got[k], want[k]) < 1e-10, k
    ref.ctx.close()
    s.ctx.close()
