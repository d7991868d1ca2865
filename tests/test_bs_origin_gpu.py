"""Targets at the exact origin, far from every segment: the records that pad
a list's last group must give nothing there, whatever the list's length.
Tolerance of the grouped kernels (a pair's d1 j1 - d2 j2 cancels by about
|r| / |r0|, at most 1e3 here)."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.test_bs_groups_gpu import _chain
from tests.test_zz_no_alloc import _Hip, _noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 32, 33, 1000])
def test_origin_target_is_finite(n):
    from volcanor_amd import vlm
    a, b, g, rc, _ = _chain(n, 1, n)
    off = np.array([9.0, -8.0, 7.0])
    a, b = a + off, b + off
    # an odd grid around the origin: its centre is at 0 exactly
    x = np.linspace(-0.5, 0.5, 13)
    p = np.stack(np.meshgrid(x, x, x, indexing="ij"), -1).reshape(-1, 3)
    assert len(p) > 2048 and np.any(np.all(p == 0.0, axis=1))
    w = orc.filament_sum(a, b, g, rc, p)
    ctx, hip = vlm.Context(0), _Hip()
    fs, (ps, m) = ctx.fset_create(a, b, g, rc), ctx.pset_create(p)
    ctx.fset_vind(fs, ps)
    got = [ctx.filament_vind(a, b, g, rc, p), ctx.pset_velocity(ps, m),
           _noalloc(ctx, hip, a, b, g, rc, p)]
    hip.free()
    ctx.close()
    for v in got:
        assert np.all(np.isfinite(v)) and np.max(np.abs(v - w)) <= 1e-11 * np.max(np.abs(w))
