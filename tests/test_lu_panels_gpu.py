"""The panels of the blocked LU at the orders where they hand over: one wave
(64 rows), two, four and eight waves (128, 256, 512 rows) and ragged last
panels of one to 31 columns, against LAPACK, with equal pivots (distinct
magnitudes), with ties, which go to the lower row as IDAMAX has them, and
with a zero column.

Both factorisations are backward stable with the same pivots, so the
factors agree to n eps times the growth, far below 1e-10 here."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 31, 33, 63, 64, 65, 95, 127, 129, 160, 255, 257, 289, 511, 515])
def test_small_orders_match_lapack(n):
    from scipy.linalg import lu_factor

    from volcanor_amd import vlm
    ctx = vlm.Context(0)
    A = np.random.default_rng(n).standard_normal((n, n))
    LU, piv = ctx.lu_factor(A)
    LUl, pivl = lu_factor(A)
    np.testing.assert_array_equal(piv, pivl)
    assert np.max(np.abs(LU - LUl)) <= 1e-10 * np.max(np.abs(LUl))
    # every candidate of a column equal in magnitude: the first row wins
    S = np.where(np.random.default_rng(n + 1).random((n, n)) < 0.5, -1.0, 1.0)
    S += np.diag(np.arange(n) * 1e-3)
    LU, piv = ctx.lu_factor(S)
    LUl, pivl = lu_factor(S)
    assert piv[0] == np.argmax(np.abs(S[:, 0])) == pivl[0]
    P = np.arange(n)
    for k in range(n):
        P[[k, piv[k]]] = P[[piv[k], k]]
    L, U = np.tril(LU, -1) + np.eye(n), np.triu(LU)
    assert np.max(np.abs(L @ U - S[P])) <= 1e-10 * np.max(np.abs(U))
    ctx.close()


@pytest.mark.parametrize("n,col", [(20, 19), (64, 40), (100, 80), (200, 10), (300, 290)])
def test_zero_column_is_reported(n, col):
    from volcanor_amd import vlm
    A = np.random.default_rng(n).standard_normal((n, n))
    A[:, col] = 0.0
    ctx = vlm.Context(0)
    with pytest.raises(vlm.VLMError, match="singular"):
        ctx.lu_factor(A)
    ctx.close()
