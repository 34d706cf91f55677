"""The compression and the compressed product at every block order n = 2 nmax
(nmax + 2): rows in one to four registers of a wave, 16-lane groups full and not."""
import numpy as np
import pytest

from optimet_amd.problem import Cluster, drude_cluster, random_cluster

pytestmark = pytest.mark.gpu

NM = 1e-9


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("nmax", range(1, 11))
def test_orders(nmax):
    """A cross approximation of r terms reproduces r rows and r columns of its
    block (to the rounding of r updates, 1e-10 of the block); the solution is the
    compressed operator's, expanded on the host, at the GMRES tolerance times a
    condition number of a few units (1e-11)."""
    from optimet_amd import solver
    P = 9
    xyz, radii, _ = random_cluster(P, 30 * NM, 60 * NM, 2500 * NM, 150 * NM, 3)
    c = Cluster(xyz=xyz, radius=radii, eps_r=np.full(P, 2.25 + 0j), eps_r_sh=np.full(P, 2.25 + 0j), nmax=nmax,
                wavelength=700 * NM, sh=False)
    n = c.N // P
    d = solver.Solver(c, kind="lu64")
    d.update()
    S = d.matrix()
    s = solver.Solver(c, kind="aca", tol=1e-13)
    s.update()
    ranks, info = s.aca_info()
    assert info["compressed_blocks"] > 0
    A = np.eye(c.N, dtype=complex)
    for i in range(P):
        for j in range(P):
            if i == j:
                continue
            U, V = s.aca_block(i, j)
            B = U if V is None else U @ V
            A[i * n:(i + 1) * n, j * n:(j + 1) * n] = B
            E = np.abs(B - S[i * n:(i + 1) * n, j * n:(j + 1) * n])
            small = 1e-10 * np.abs(S[i * n:(i + 1) * n, j * n:(j + 1) * n]).max()
            r = min(n, n if V is None else U.shape[1])
            assert (E.max(axis=1) <= small).sum() >= r and (E.max(axis=0) <= small).sum() >= r, (i, j, r)
    x = s.solve()["x_sca"]
    assert rel(x, np.linalg.solve(A, s.vector("Q"))) < 1e-11


def test_memory_follows_the_cluster():
    """A context that compressed a large cluster holds no more for a small one than
    a fresh context, except the vectors of the larger order (basis of 240 steps and
    partial sums, about 440 of them): the pools and the staging are kept for
    clusters of the same shape only.  Another kind of solver gives them back."""
    from optimet_amd import solver

    def cluster(P):
        return drude_cluster(P, 5, 800 * NM, 30, 60, 2500, 10, seed=1, sh=False)

    small, large = cluster(60), cluster(200)
    fresh = solver.Solver(small, kind="aca")
    fresh.update()
    want = fresh.solve()["x_sca"]
    bound = fresh.ctx.mem_info()[2] + 16 * large.N * 441
    fresh.ctx.close()
    s = solver.Solver(large, kind="aca")
    s.update()
    s.solve()
    s.set_cluster(small)
    for _ in range(2):
        s.update()
        assert np.array_equal(s.solve()["x_sca"], want)
        assert s.ctx.mem_info()[2] <= bound
    s.ctx.set_solver("lu64")
    s.update()
    d = solver.Solver(small, kind="lu64")
    d.update()
    assert s.ctx.mem_info()[2] <= d.ctx.mem_info()[2] + 16 * large.N * 441
    s.ctx.close()
    d.ctx.close()
