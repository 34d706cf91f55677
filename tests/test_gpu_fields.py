"""Field maps at the sizes where their kernels change: one and a few points,
tiles of 64 points cut short, one to several objects per wave, the lowest and
the highest order, with and without the second harmonic."""
import numpy as np
import pytest

from optimet_amd.problem import drude_cluster

pytestmark = pytest.mark.gpu


def solved(P, nmax, sh, seed=3):
    from optimet_amd import solver
    c = drude_cluster(P, nmax, 700e-9, 60, 80, 700, 10, seed=seed, sh=sh)
    c.theta_k, c.phi_k = 0.4, 0.7
    s = solver.Solver(c, kind="lu64")
    s.update()
    return c, s, s.solve()


@pytest.mark.parametrize("P,nmax,npts,sh", [(1, 1, 1, True), (2, 2, 63, False), (3, 5, 64, True), (5, 4, 65, True),
                                            (9, 6, 200, False), (4, 10, 129, True)])
def test_fields_against_oracle(ora, P, nmax, npts, sh):
    """Against the oracle's fields at the device's own coefficients, 1e-10 of
    each field's largest component (the bar of the other field tests)."""
    c, s, out = solved(P, nmax, sh)
    rng = np.random.default_rng(npts)
    pts = rng.uniform(-100e-9, 800e-9, (npts, 3))
    # every third point inside a sphere
    for i in range(0, npts, 3):
        d = rng.standard_normal(3)
        pts[i] = c.xyz[i % P] + rng.uniform(0.3, 0.95) * c.radius[i % P] * d / np.linalg.norm(d)
    f = s.fields(pts)
    ref = ora.fields(c, ora.cg_tables(nmax), out, pts)
    for k in f:
        assert np.max(np.abs(f[k] - ref[k])) <= 1e-10 * np.max(np.abs(ref[k])), k


def test_fields_in_chunks():
    """More points than one chunk holds, the last chunk of another size: the
    same values as the points taken in two calls.  The sums over the objects
    may be split differently (a handful of terms), hence 1e-14."""
    c, s, _ = solved(9, 2, True)
    rng = np.random.default_rng(1)
    pts = rng.uniform(-100e-9, 800e-9, ((1 << 16) + 70, 3))
    f = s.fields(pts)
    a, b = s.fields(pts[:40000]), s.fields(pts[40000:])
    for k in f:
        ref = np.concatenate([a[k], b[k]])
        assert np.max(np.abs(f[k] - ref)) <= 1e-14 * np.max(np.abs(ref)), k
