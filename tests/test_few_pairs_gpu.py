"""Launches of few pairs (segments on lanes) and grouped ones on both sides of
the lines between them, 6e7 pairs up to 256 targets and 3e7 below 2048, and where short lists are
split (at most 512 blocks, 16 chunks, 2 segments per lane), against the FP64
oracle; a list alone sums like the same list among others, to the bit."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.test_bs_groups_gpu import _chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(2047, 14655), (2047, 14656), (2048, 10), (400, 75000), (400, 75001),
                                 (192, 312500), (192, 312501), (257, 116731), (257, 116732), (1000, 50), (600, 6666),
                                 (128, 8192), (129, 8191), (2047, 511), (300, 13333)])
def test_both_sides_match_oracle(m, n):
    from volcanor_amd import vlm
    ctx = vlm.Context(0)
    a, b, g, rc, p = _chain(n, m, n + m)
    w = orc.filament_sum(a, b, g, rc, p, threads=8)
    fs, (ps, mm) = ctx.fset_create(a, b, g, rc), ctx.pset_create(p)
    ctx.fset_vind(fs, ps)
    v = ctx.pset_velocity(ps, mm)
    ctx.close()
    assert np.max(np.abs(v - w)) <= 1e-11 * np.max(np.abs(w))


@pytest.mark.parametrize("ns,rows,m", [(30, 2, 40), (30, 100, 200), (30, 300, 90), (30, 300, 600)])
def test_one_list_alone_and_among_others(ns, rows, m):
    """The wing's list (empty circulation) adds nothing to the wake's."""
    from tests import wake_harness as H
    from volcanor_amd import vlm
    case = H.Case(nb=2, nc=1, ns=ns, nNwake=rows, nFwake=0)
    ctx = vlm.Context(0)
    ir = H.setup(ctx, case)[0]
    rng = np.random.default_rng(rows)
    nodes = rng.standard_normal((2, rows, ns + 1, 3))
    ctx.rotor_set_wake(ir, dict(nodes=nodes, le=rng.standard_normal((2, ns + 1, 3)),
                                gam=rng.standard_normal((2, rows, ns)),
                                rc4=np.full((2, rows, ns, 4), 0.1), far_fc=np.zeros((2, 0, 2, 3)),
                                far_gam=np.zeros((2, 0)), far_rc=np.zeros((2, 0))), 1, 1)
    ctx.rotor_set_wing(ir, rng.standard_normal((2, ns, 1, 4, 3)), np.full((2, ns, 1, 4), 0.1),
                       np.zeros((2, ns, 1)))
    p = rng.standard_normal((m, 3))
    alone = ctx.rotor_induced_velocity(ir, vlm.SET_WAKE, p)
    one = ctx.induced_velocity_terms([(ir, vlm.SET_WAKE, 0)], p)
    among = ctx.induced_velocity_terms([(ir, vlm.SET_WING, 0), (ir, vlm.SET_WAKE, 0)], p)
    ctx.close()
    assert np.array_equal(alone, one) and np.array_equal(alone, among)
