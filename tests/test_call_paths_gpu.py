"""One-call evaluations whose inputs the kernels read in pinned memory, on
both sides of the size (4 MiB) at which they are copied first and of the
kernels' block sizes, against the same sums over device-resident sets: the
records, chunks and kernels are the same, so the bits are.  Copies that go in
two and three pieces carry a matrix through the factorisation."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nfil,m", [(1, 1), (255, 191), (256, 192), (257, 1030), (31, 257),
                                    (65400, 30), (65600, 3), (20, 90000)])
def test_one_call_equals_resident_sets(nfil, m):
    from volcanor_amd import vlm
    ctx = vlm.Context(0)
    rng = np.random.default_rng(nfil + m)
    a, b, p, v0 = (rng.normal(size=(k, 3)) for k in (nfil, nfil, m, m))
    g, rc = rng.normal(size=nfil), rng.uniform(0.01, 0.1, nfil)
    fs, (ps, _) = ctx.fset_create(a, b, g, rc), ctx.pset_create(p)
    ctx.fset_vind(fs, ps)
    want = ctx.pset_velocity(ps, m)
    assert np.array_equal(ctx.filament_vind(a, b, g, rc, p), want)
    assert np.array_equal(ctx.filament_vind(a, b, g, rc, p, v=v0), v0 + want)


def test_no_filaments():
    from volcanor_amd import vlm
    ctx = vlm.Context(0)
    p, e = np.ones((70, 3)), np.zeros((0, 3))
    v = np.arange(210.0).reshape(70, 3)
    assert np.array_equal(ctx.filament_vind(e, e, np.zeros(0), np.zeros(0), p), np.zeros_like(p))
    assert np.array_equal(ctx.filament_vind(e, e, np.zeros(0), np.zeros(0), p, v=v), v)


@pytest.mark.parametrize("n", [512, 520, 740])
def test_matrices_in_pieces(n):
    from scipy.linalg import lu_factor

    from volcanor_amd import vlm
    ctx = vlm.Context(0)
    rng = np.random.default_rng(n)
    A, x = rng.standard_normal((n, n)), rng.standard_normal(n)
    LU, piv = ctx.lu_factor(A)
    ref, pref = lu_factor(A)
    assert np.array_equal(piv, pref)
    assert np.max(np.abs(LU - ref)) <= 1e-9 * np.max(np.abs(ref))
    got, _ = ctx.lu_solve_refine(A, LU, piv, A @ x)
    assert np.max(np.abs(A @ got - A @ x)) <= 1e-11 * n


@pytest.mark.parametrize("n,m", [(1, 2049), (31, 2049), (32, 2112), (33, 2113), (1000, 2111),
                                 (4687, 640), (4688, 640),        # 3e6 pairs, either kernel
                                 (40000, 400), (40001, 400), (7500, 401),
                                 (83333, 192), (83334, 192), (20000, 51), (250000, 64),
                                 (250001, 64), (123000, 130)])
def test_kernels_at_the_rule_match_oracle(n, m):
    """Both sides of the few-pairs rule and the edges of groups and waves just
    above it; the tolerance of the grouped kernels' own tests."""
    from oracle import oracle as orc
    from tests.test_bs_groups_gpu import _chain
    from volcanor_amd import vlm
    ctx = vlm.Context(0)
    a, b, g, rc, p = _chain(n, m, n + m)
    w = orc.filament_sum(a, b, g, rc, p)
    v = ctx.filament_vind(a, b, g, rc, p)
    assert np.max(np.abs(v - w)) <= 1e-11 * np.max(np.abs(w))
    fs, (ps, mm) = ctx.fset_create(a, b, g, rc), ctx.pset_create(p)
    ctx.fset_vind(fs, ps)
    assert np.array_equal(ctx.pset_velocity(ps, mm), v)
