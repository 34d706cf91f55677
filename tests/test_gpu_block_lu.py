"""The block-pivoting LU: pivots from anywhere in a panel's 64 rows, one panel,
pairs and a last panel alone, in both precisions; zero pivots reported."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.fixture(scope="module")
def ctx():
    from optimet_amd import solver
    return solver.Context()


def blocked(rng, N):
    """Dominant entries in every block's rows in a random order, so that block
    pivoting finds them all; well conditioned."""
    A = rng.standard_normal((N, N)) + 1j * rng.standard_normal((N, N))
    for k in range(0, N, 64):
        n = min(64, N - k)
        A[k + rng.permutation(n), k + np.arange(n)] += 6 * np.sqrt(N) * np.exp(2j * np.pi * rng.random(n))
    return A


@pytest.mark.parametrize("N", [1, 17, 64, 65, 128, 129, 192, 250, 321, 640, 1100])
@pytest.mark.parametrize("kind", ["lu64", "lu32ir"])
def test_block_pivoting_sizes(ctx, N, kind):
    """Against numpy: refined solutions of matrices of small condition, 1e-12."""
    rng = np.random.default_rng(N)
    A, b = blocked(rng, N), rng.standard_normal(N) + 1j * rng.standard_normal(N)
    x = ctx.dense_solve(A, b, kind)
    assert ctx.stats()["pivot_fallbacks"] == 0
    assert rel(x, np.linalg.solve(A, b)) < 1e-12


@pytest.mark.parametrize("col", [0, 63, 64, 100, 191])
def test_zero_pivot_is_reported(ctx, col):
    """A column of zeros: singular in both pivot modes, with its number."""
    from optimet_amd.solver import OmxError
    rng = np.random.default_rng(col)
    A = blocked(rng, 192)
    A[:, col] = 0
    with pytest.raises(OmxError, match=f"column {col}"):
        ctx.dense_solve(A, rng.standard_normal(192) + 0j, "lu64")
