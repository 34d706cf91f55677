"""The device-driven GMRES over the shapes where its kernels change: a block's
rows not full, exactly full and one system of a single block; cycles of one
step, of a few and longer than the solve; budgets that end inside a cycle."""
import numpy as np
import pytest

from optimet_amd.problem import Cluster, drude_cluster, random_cluster

pytestmark = pytest.mark.gpu

NM = 1e-9


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def glass(P, nmax):
    """Weakly scattering spheres: a condition number of a few units."""
    xyz, radii, _ = random_cluster(P, 40 * NM, 80 * NM, 1200 * NM, 10 * NM, 5 + P)
    return Cluster(xyz=xyz, radius=radii, eps_r=np.full(P, 2.25 + 0j), eps_r_sh=np.full(P, 2.25 + 0j), nmax=nmax,
                   wavelength=700 * NM, sh=False)


# N = 2 P nmax (nmax + 2): 6, 256, 350, 510, 1152
@pytest.mark.parametrize("P,nmax", [(1, 1), (16, 2), (5, 5), (17, 3), (12, 6)])
@pytest.mark.parametrize("restart", [1, 3, 256])
def test_cycles(P, nmax, restart):
    """A residual of 1e-12 leaves at most the condition number times it: 1e-10."""
    from optimet_amd import solver
    c = glass(P, nmax)
    ref = solver.Solver(c, kind="lu64")
    ref.update()
    want = ref.solve()["x_sca"]
    s = solver.Solver(c, kind="gmres64", tol=1e-12, maxit=200, restart=restart)
    s.update()
    got = s.solve()["x_sca"]
    st = s.stats()
    assert st["residual"] <= 1e-12 and 0 < st["iterations"] <= 200
    assert rel(got, want) < 1e-10
    # again on the same state, from what the first solve left in the workspaces
    assert np.array_equal(s.solve()["x_sca"], got) and s.stats()["iterations"] == st["iterations"]


@pytest.mark.parametrize("maxit", [1, 2, 5])
def test_budget(maxit):
    """The budget counts steps, inside a cycle and across cycles: either that
    many were taken or the tolerance was met before."""
    from optimet_amd import solver
    for restart in (2, 40):
        s = solver.Solver(glass(12, 6), kind="gmres64", tol=1e-14, maxit=maxit, restart=restart)
        s.update()
        try:
            s.solve()
        except solver.OmxError as e:
            assert "converge" in str(e)
        assert s.stats()["iterations"] <= maxit


def test_a_batch_counts_its_systems_steps_alone():
    """Systems that leave a batch at the FP64 floor, by a correction too small to
    change them, take no further steps while the others go on: each one's count is
    that of the same system alone, to a few cycles of two steps that rounding at
    the floor shifts (8; those that went on took the slowest one's 56 instead of
    about 30)."""
    from optimet_amd import solver
    c = drude_cluster(14, 8, 700 * NM, 40, 80, 1000, 10, seed=91)
    lams = np.linspace(450, 850, 8) * NM

    def its(l):
        s = solver.Solver(c, kind="auto", tol=1e-18, restart=2, maxit=2000)
        s.ctx.set_autotune(False)
        s.ctx.set_auto_budget(1000)
        out = s.sweep(l, batch=len(l), outputs=("x_sca",))["iterations"][:, 0]
        s.ctx.close()
        return out

    together, alone = its(lams), np.concatenate([its([l]) for l in lams])
    assert (np.abs(together - alone) <= 8).all(), (together, alone)


def test_a_profiled_sweep_times_itself():
    """The sweep's time holds its products, and is not shorter than half of the same
    sweep's without the products' events."""
    from optimet_amd import solver
    c = drude_cluster(6, 5, 700 * NM, 40, 80, 700, 10, seed=3)
    s = solver.Solver(c, kind="lu32ir")
    s.ctx.set_profile(True)
    s.sweep(np.linspace(450, 850, 8) * NM, batch=4)
    st = s.stats()
    s.ctx.close()
    assert st["matvec_calls"] > 4 and st["t_matvec_ms"] > 0
    wall = st["t_solve_ms"]
    s = solver.Solver(c, kind="lu32ir")
    s.sweep(np.linspace(450, 850, 8) * NM, batch=4)  # the same sweep without the events
    plain = s.stats()["t_solve_ms"]
    s.ctx.close()
    assert wall > st["t_matvec_ms"] and wall > 0.5 * plain
