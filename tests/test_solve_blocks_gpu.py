"""The blocked substitutions (one workgroup per 64 rows and sweep) at the
edges of their blocks, against LAPACK: orders around multiples of 64, one
block more than the one-wave solve, several corrections, and a matrix with a
diagonal whose reciprocals leave the normal range.

The tolerance is that of a backward stable solve: n eps cond(A), with
cond below 1e5 on these diagonally shifted matrices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(n, seed):
    rng = np.random.default_rng(seed)
    A = rng.standard_normal((n, n)) + np.diag(rng.choice([-1.0, 1.0], n) * np.sqrt(n))
    return np.asfortranarray(A), rng.standard_normal(n)


@pytest.mark.parametrize("n", [97, 127, 128, 129, 191, 449, 1025])
@pytest.mark.parametrize("max_iter", [0, 3])
def test_blocked_solve_matches_lapack(n, max_iter):
    from volcanor_amd import vlm
    A, b = _system(n, n)
    ctx = vlm.Context(0)
    LU, piv = ctx.lu_factor(A)
    for k in range(3):   # the same work buffers again
        rhs = b * (k + 1)
        x, it = ctx.lu_solve_refine(A, LU, piv, rhs, max_iter=max_iter, tol=1e-15)
        ref = np.linalg.solve(A, rhs)
        assert np.max(np.abs(x - ref)) <= n * 2.2e-16 * 1e5 * np.max(np.abs(ref))
        assert 0 <= it <= max_iter
    # a tolerance the first solve meets stops the corrections
    x, it = ctx.lu_solve_refine(A, LU, piv, b, max_iter=5, tol=1e-3)
    assert it == 0
    ctx.close()


def test_blocked_solve_scaled_diagonal():
    from volcanor_amd import vlm
    n = 130
    A = np.asfortranarray(np.diag(np.full(n, 1e-305)) + np.diag(np.full(n - 1, 1e-306), 1))
    LU, piv = A.copy(order="F"), np.arange(n, dtype=np.int32)
    ctx = vlm.Context(0)
    x, _ = ctx.lu_solve_refine(A, LU, piv, np.full(n, 1e-300), max_iter=0)
    ref = np.zeros(n)
    ref[-1] = 1e5
    for i in range(n - 2, -1, -1):
        ref[i] = (1e-300 - 1e-306 * ref[i + 1]) / 1e-305
    assert np.max(np.abs(x - ref)) <= 1e-12 * np.max(np.abs(ref))
    with pytest.raises(vlm.VLMError, match="pivot out of range"):
        ctx.lu_solve_refine(A, LU, np.full(n, n, dtype=np.int32), np.ones(n))
    ctx.close()
