"""The assembly at every harmonic order (each has a workgroup shape of its
own) and the batched one: S, V, Q and the local incident fields against the
oracle at 1e-12, the bar of the other assembly tests."""
import numpy as np
import pytest

from optimet_amd.problem import drude_cluster

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("nmax", range(1, 11))
def test_assembly_at_every_order(ora, nmax):
    """Three spheres, one of them centred at the origin (its coupling to the
    incident wave is the identity), a lossy background, oblique incidence."""
    from optimet_amd import solver
    c = drude_cluster(3, nmax, 700e-9, 40, 60, 500, 10, seed=20 + nmax)
    c.xyz = c.xyz - c.xyz[1]
    c.theta_k, c.phi_k, c.bg_eps_r = 0.5, -0.3, 1.5 + 0.02j
    s = solver.Solver(c, kind="lu64")
    s.update()
    assert rel(s.vector("Q"), ora.source_vector(c)) < 1e-12
    assert rel(s.vector("inc"), np.concatenate([ora.inc_local(c, j) for j in range(3)])) < 1e-12
    assert rel(s.matrix(), ora.scattering_matrix(c)) < 1e-12
    assert rel(s.matrix(sh=True), ora.scattering_matrix(c, sh=True)) < 1e-12


def test_update_returns_before_the_device():
    """A second update of the same context with other inputs, and reads of
    another context in between, see their own assembly."""
    from optimet_amd import solver
    a = drude_cluster(12, 5, 700e-9, 40, 60, 700, 10, seed=1)
    b = drude_cluster(12, 5, 650e-9, 40, 60, 700, 10, seed=2)
    sa, sb = solver.Solver(a, kind="lu64"), solver.Solver(b, kind="lu64")
    sa.update()
    sb.update()
    Sa, Sb = sa.matrix(), sb.matrix()
    sa.set_cluster(b)
    sa.update()
    sb.set_cluster(a)
    sb.update()
    assert np.array_equal(sa.matrix(), Sb) and np.array_equal(sb.matrix(), Sa)
