"""LU of matrices that hold NaNs and infinities, on every panel kernel of the
orders up to 256: a column's candidates are its numbers, a column without any
pivots on its diagonal, and the factors hold NaN and infinities exactly where
the column-by-column algorithm has them (finished rows are not touched).
Finite entries agree as those of finite matrices do."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _lu_reference(A):
    A, piv = A.copy(), []
    n = len(A)
    with np.errstate(all="ignore"):
        for k in range(n):
            c = np.abs(A[k:, k])
            p = k if np.all(np.isnan(c)) else k + int(np.nanargmax(c))
            piv.append(p)
            A[[k, p]] = A[[p, k]]
            A[k + 1:, k] *= 1.0 / A[k, k]
            A[k + 1:, k + 1:] -= np.outer(A[k + 1:, k], A[k, k + 1:])
    return A, np.array(piv)


def _check(A):
    from volcanor_amd import vlm
    ctx = vlm.Context(0)
    LU, piv = ctx.lu_factor(A)
    ctx.close()
    ref, pref = _lu_reference(A)
    np.testing.assert_array_equal(piv, pref)
    np.testing.assert_array_equal(np.isnan(LU), np.isnan(ref))
    np.testing.assert_array_equal(np.isposinf(LU), np.isposinf(ref))
    np.testing.assert_array_equal(np.isneginf(LU), np.isneginf(ref))
    f = np.isfinite(ref)
    if f.any():
        assert np.max(np.abs(LU[f] - ref[f])) <= 1e-10 * max(1.0, np.max(np.abs(ref[f])))


@pytest.mark.parametrize("n", [1, 20, 64, 65, 100, 129, 200, 256])
@pytest.mark.parametrize("where", ["entry", "column", "all"])
def test_nan(n, where):
    A = np.random.default_rng(n).standard_normal((n, n))
    if where == "entry":
        A[n // 2, n // 3] = np.nan
    elif where == "column":
        A[:, 2 * n // 5] = np.nan
    else:
        A[:] = np.nan
    _check(A)


@pytest.mark.parametrize("n", [20, 64, 65, 100, 129, 200, 256])
@pytest.mark.parametrize("row,col", [(0.5, 0.3), (0.1, 0.97), (0.9, 0.6)])
def test_infinity(n, row, col):
    A = np.random.default_rng(n).standard_normal((n, n))
    A[int(row * n), int(col * n)] = -np.inf
    _check(A)


def test_nan_above_the_order_is_reported():
    from volcanor_amd import vlm
    ctx = vlm.Context(0)
    with pytest.raises(vlm.VLMError, match="singular"):
        ctx.lu_factor(np.full((300, 300), np.nan))
    ctx.close()
