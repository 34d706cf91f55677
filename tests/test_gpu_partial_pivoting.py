"""The partial-pivoting LU over the sizes where its tournament changes: one
workgroup, one level of merges, several, incomplete last sets; rows whose
pivots come from far below the panel, in both precisions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.fixture(scope="module")
def ctx():
    from optimet_amd import solver
    return solver.Context()


def graded(rng, N):
    """Rows in an order that puts the large ones last, so that every panel's
    pivots come from the end of the column; well conditioned after pivoting."""
    A = rng.standard_normal((N, N)) + 1j * rng.standard_normal((N, N))
    A[np.arange(N), N - 1 - np.arange(N)] += 4 * np.sqrt(N)
    return A


@pytest.mark.parametrize("N", [1, 63, 64, 65, 128, 192, 193, 257, 576, 577, 640, 1000])
@pytest.mark.parametrize("kind", ["lu64", "lu32ir"])
def test_partial_pivoting_sizes(ctx, N, kind):
    """Against numpy: N eps times the growth of these matrices, 1e-11."""
    rng = np.random.default_rng(N)
    A, b = graded(rng, N), rng.standard_normal(N) + 1j * rng.standard_normal(N)
    ctx.set_pivoting("partial")
    try:
        x = ctx.dense_solve(A, b, kind)
    finally:
        ctx.set_pivoting("block")
    assert rel(x, np.linalg.solve(A, b)) < 1e-11


@pytest.mark.parametrize("scale", [1e-170, 1e-60, 1e60, 1e140])
def test_partial_pivoting_scales(ctx, scale):
    """Entries far outside the single-precision range: the pivots still order."""
    rng = np.random.default_rng(7)
    A, b = graded(rng, 200) * scale, rng.standard_normal(200) + 1j * rng.standard_normal(200)
    ctx.set_pivoting("partial")
    try:
        if scale < 1e-160:  # squares of the pivots underflow: reported singular, as before
            from optimet_amd.solver import OmxError
            with pytest.raises(OmxError):
                ctx.dense_solve(A, b, "lu64")
            return
        x = ctx.dense_solve(A, b, "lu64")
    finally:
        ctx.set_pivoting("block")
    assert rel(x, np.linalg.solve(A, b)) < 1e-11


def test_singular_column_is_reported(ctx):
    from optimet_amd.solver import OmxError
    rng = np.random.default_rng(3)
    A = graded(rng, 300)
    A[:, 150] = 0.0
    ctx.set_pivoting("partial")
    try:
        with pytest.raises(OmxError) as e:
            ctx.dense_solve(A, np.ones(300, complex), "lu64")
    finally:
        ctx.set_pivoting("block")
    assert e.value.code == -4 and "column 150" in str(e.value)


@pytest.mark.parametrize("kind", ["lu64", "lu32ir"])
def test_negative_zeros_do_not_order_first(ctx, kind):
    """Columns whose entries below the pivot are zeros of either sign."""
    rng = np.random.default_rng(5)
    N = 300
    A = np.triu(rng.standard_normal((N, N)) + 1j * rng.standard_normal((N, N))) + 30 * np.eye(N)
    A = np.where(A == 0, -0.0 - 0.0j, A)
    b = rng.standard_normal(N) + 1j * rng.standard_normal(N)
    ctx.set_pivoting("partial")
    try:
        x = ctx.dense_solve(A, b, kind)
    finally:
        ctx.set_pivoting("block")
    assert rel(x, np.linalg.solve(A, b)) < 1e-11


@pytest.mark.parametrize("N", [64, 130, 192])
def test_pivots_are_the_largest_of_their_columns(ctx, N):
    """Up to 192 rows the panel's rows meet in one workgroup, so every pivot is the
    column's largest in modulus: no multiplier above 1, to the rounding of the
    panel's products with the inverse of its triangle (u times a condition number
    of 1e4: 1e-11).  The moduli of the first column differ by 1e-8 at most."""
    from tests.test_zz_no_alloc import _Dev, _hip
    hip = _hip()
    rng = np.random.default_rng(N)
    Np = -(-N // 64) * 64
    A = np.exp(2j * np.pi * rng.random((N, N))) * (1 + 1e-8 * rng.random((N, N)))
    b = rng.standard_normal(N) + 1j * rng.standard_normal(N)
    cols = np.zeros((Np, Np), complex)  # row c is column c of A
    cols[:N, :N] = A.T
    dA, db, dx = _Dev(hip, cols.nbytes), _Dev(hip, b.nbytes), _Dev(hip, b.nbytes)
    try:
        dA.put(cols)
        db.put(b)
        ctx.dense_solve_noalloc(N, dA.p.value, Np, db.p.value, dx.p.value)
        L = np.tril(dA.get((Np, Np), np.complex128).T, -1)
        x = dx.get(N, np.complex128)
    finally:
        for d in (dA, db, dx):
            d.free()
    assert np.abs(L).max() <= 1 + 1e-11, np.abs(L).max() - 1
    assert rel(x, np.linalg.solve(A, b)) < 1e-11
