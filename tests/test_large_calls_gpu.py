"""Calls with many points: they pass through the pinned arena in pieces (87296
points each), and what they need on the device is given back."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as orc
from tests.test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [87295, 87297, 174593, 300001])
def test_points_in_pieces(m):
    from volcanor_amd import vlm
    rng = np.random.default_rng(m)
    a, b, p, v0 = (rng.normal(size=(k, 3)) for k in (4, 4, m, m))
    g, rc = rng.normal(size=4), np.full(4, 0.1)
    w = orc.filament_sum(a, b, g, rc, p, threads=8)
    tol = 1e-12 * np.max(np.abs(w))
    ctx = vlm.Context(0)
    assert np.max(np.abs(ctx.filament_vind(a, b, g, rc, p) - w)) <= tol
    v = ctx.filament_vind(a, b, g, rc, p, v=v0)
    assert np.max(np.abs(v - (v0 + w))) <= tol + 1e-15 * np.max(np.abs(v0))
    fs, (ps, n) = ctx.fset_create(a, b, g, rc), ctx.pset_create(p)
    ctx.fset_vind(fs, ps)
    assert np.max(np.abs(ctx.pset_velocity(ps, n) - w)) <= tol
    ctx.close()


def test_device_memory_is_given_back():
    from volcanor_amd import vlm
    hip = _Hip().lib

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    a, b = np.zeros((1, 3)), np.ones((1, 3))
    g, rc = np.ones(1), np.full(1, 0.1)
    ctx = vlm.Context(0)
    ctx.filament_vind(a, b, g, rc, np.full((100, 3), 2.0))
    free0 = free()
    m = 15000000                   # 360 MB of points, results and partial sums each
    v = ctx.filament_vind(a, b, g, rc, np.tile(np.arange(3.0), (m, 1)))
    assert np.all(v == v[0])
    assert free0 - free() <= 24 * m + (64 << 20)   # the partial sums
    ctx.close()
