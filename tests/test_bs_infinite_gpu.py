"""A segment of infinite or NaN circulation among finite ones: infinities and
NaNs stand where the oracle has them, in launches of few pairs and grouped
ones, far and near."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.test_bs_groups_gpu import _chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("n,m", [(40, 300), (33, 3300), (1000, 3300)])
@pytest.mark.parametrize("away", [0.0, 9.0])
def test_circulation_without_a_number(n, m, value, away):
    from volcanor_amd import vlm
    a, b, g, rc, p = _chain(n, m, n)
    p = p[m // 3:] + away          # no end points of segments
    g[n // 2] = value
    with np.errstate(all="ignore"):
        w = orc.filament_sum(a, b, g, rc, p)
    ctx = vlm.Context(0)
    v = ctx.filament_vind(a, b, g, rc, p)
    ctx.close()
    np.testing.assert_array_equal(np.isnan(v), np.isnan(w))
    np.testing.assert_array_equal(np.isposinf(v), np.isposinf(w))
    np.testing.assert_array_equal(np.isneginf(v), np.isneginf(w))
