"""The one-wave solve at the edges of its column blocks (8, 64, 96) with rows
that the pivoting moves, with diagonals whose reciprocal leaves the normal
range (scaled by 1e305 and 1e-305: the division path), and with ties, against
LAPACK's solution.  Refined on the FP64 residual, both agree to a few
condition numbers of eps: matrices here have condition below 1e3, so 1e-11."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1.0, 1e305, 1e-305])
@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 63, 64, 65, 72, 73, 95, 96])
def test_wave_solve_matches_lapack(n, scale):
    from volcanor_amd import vlm
    ctx = vlm.Context(0)
    rng = np.random.default_rng(n)
    # a well-conditioned matrix whose rows are out of order
    A = (np.eye(n) + 0.3 * rng.standard_normal((n, n)) / np.sqrt(n))[rng.permutation(n)]
    x = rng.standard_normal(n)
    b = A @ x
    LU, piv = ctx.lu_factor(A)
    got, it = ctx.lu_solve_refine(A, LU, piv, b, max_iter=3)
    assert np.max(np.abs(got - x)) <= 1e-11 * np.max(np.abs(x))
    if scale != 1.0:
        # U times a power of ten near the end of the range, L as it was: the
        # solve without refinement scales by its inverse
        U = np.triu(LU) * scale
        S = np.asfortranarray(np.tril(LU, -1) + U)
        base, _ = ctx.lu_solve_refine(A, LU, piv, b, max_iter=0)
        got, _ = ctx.lu_solve_refine(A, S, piv, b, max_iter=0)
        assert np.max(np.abs(got * scale - base)) <= 1e-11 * np.max(np.abs(x))
