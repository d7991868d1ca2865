"""Triangular solves with infinite and NaN values on every path (one and two
rows per lane, blocks of 64 rows): entries that the column-by-column
substitution leaves finite stay finite, and infinities and NaNs stand where it
has them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _substitution(LU, b):
    y = b.copy()
    n = len(y)
    with np.errstate(all="ignore"):
        for j in range(n):
            y[j + 1:] -= LU[j + 1:, j] * y[j]
        for j in range(n - 1, -1, -1):
            y[j] /= LU[j, j]
            y[:j] -= LU[:j, j] * y[j]
    return y


@pytest.mark.parametrize("n", [40, 90, 97, 128, 130, 200, 449])
@pytest.mark.parametrize("row", [0.0, 0.01, 0.4, 0.7])
def test_zero_on_the_diagonal(n, row):
    """U with a zero pivot: the rows below it are finite."""
    from volcanor_amd import vlm
    rng = np.random.default_rng(n)
    LU = np.asfortranarray(0.5 * rng.standard_normal((n, n)) / np.sqrt(n) + 2.0 * np.eye(n))
    k = int(row * n)
    LU[k, k] = 0.0
    # above it, one sign, so that the infinities do not all cancel to NaN
    LU[:k, k] = np.abs(LU[:k, k])
    b = rng.standard_normal(n)
    ctx = vlm.Context(0)
    x, _ = ctx.lu_solve_refine(LU, LU, np.arange(n, dtype=np.int32), b, max_iter=0)
    ctx.close()
    ref = _substitution(LU, b)
    assert np.isinf(ref[k]) and np.all(np.isfinite(ref[k + 1:]))
    np.testing.assert_array_equal(np.isnan(x), np.isnan(ref))
    np.testing.assert_array_equal(np.isposinf(x), np.isposinf(ref))
    np.testing.assert_array_equal(np.isneginf(x), np.isneginf(ref))
    np.testing.assert_allclose(x[k + 1:], ref[k + 1:], rtol=1e-10, atol=1e-12)


@pytest.mark.parametrize("n", [40, 90, 97, 130])
def test_a_residual_of_nans_ends_the_refinement(n):
    from volcanor_amd import vlm
    rng = np.random.default_rng(n)
    A = np.asfortranarray(0.5 * rng.standard_normal((n, n)) / np.sqrt(n) + 2.0 * np.eye(n))
    b = rng.standard_normal(n)
    b[0] = np.nan
    ctx = vlm.Context(0)
    LU, piv = ctx.lu_factor(A)
    x, it = ctx.lu_solve_refine(A, LU, piv, b, max_iter=3)
    ctx.close()
    assert np.all(np.isnan(x)) and it == 0
