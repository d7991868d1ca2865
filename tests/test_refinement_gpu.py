"""The refinement steps of the circulation solve, on the one-wave solve (one and
two rows per lane) and the blocked one, with the factors of a matrix that
differs from A by 1%: every correction then counts, as the error is 3 to 7% of
x without any and falls to a twentieth to a fiftieth with each.

After k corrections the solution agrees with NumPy's refinement with the same
factors to the rounding of the steps, 4 n eps cond(A), four orders or more below the
third correction; the number of corrections is NumPy's for tolerances halfway
(in decades) between two residuals."""
import numpy as np
import pytest
from scipy.linalg import lu_factor, lu_solve

pytestmark = pytest.mark.gpu


def _system(n):
    rng = np.random.default_rng(n)
    A = (np.eye(n) + 0.3 * rng.standard_normal((n, n)) / np.sqrt(n))[rng.permutation(n)]
    lu, piv = lu_factor(A * (1.0 + 1e-2 * rng.standard_normal((n, n))))
    return np.asfortranarray(A), np.asfortranarray(lu), piv.astype(np.int32), rng.standard_normal(n)


def _refinements(A, lu, piv, b, count):
    """x after 0, 1, .. count corrections and the residuals before each."""
    xs, rs = [lu_solve((lu, piv), b)], []
    for _ in range(count):
        r = b - A @ xs[-1]
        rs.append(np.max(np.abs(r)) / np.max(np.abs(b)))
        xs.append(xs[-1] + lu_solve((lu, piv), r))
    return xs, rs


@pytest.mark.parametrize("n", [40, 64, 65, 90, 96, 97, 129, 449, 1025])
def test_each_correction(n):
    from volcanor_amd import vlm
    A, lu, piv, b = _system(n)
    assert np.any(piv != np.arange(n))
    xs, rs = _refinements(A, lu, piv, b, 4)
    true = np.linalg.solve(A, b)
    tol = 4 * n * 2.2e-16 * np.linalg.cond(A) * np.max(np.abs(true))
    err = [np.max(np.abs(x - true)) for x in xs]
    assert err[0] > 1e-4 and err[2] > 10 * tol
    ctx = vlm.Context(0)
    for k in range(4):
        x, it = ctx.lu_solve_refine(A, lu, piv, b, max_iter=k, tol=0.0)
        assert it == k
        assert np.max(np.abs(x - xs[k])) <= tol
    # stops at the tolerance, before max_iter
    for k in range(1, 4):
        x, it = ctx.lu_solve_refine(A, lu, piv, b, max_iter=6, tol=np.sqrt(rs[k - 1] * rs[k]))
        assert it == k
        assert np.max(np.abs(x - xs[k])) <= tol
    x, it = ctx.lu_solve_refine(A, lu, piv, b, max_iter=12, tol=0.0)
    ctx.close()
    assert it == 12 and np.max(np.abs(x - true)) <= tol
    assert np.max(np.abs(b - A @ x)) <= n * 2.2e-16 * np.max(np.abs(A) @ np.abs(x))
