"""The grouped Biot-Savart kernels (groups of 32 segments with a far radius,
waves of 64 or 128 targets) at the edges of groups, tiles and chunks and of
the few-target and mixed-precision dispatch, against the FP64 oracle.

Tolerances, from the arithmetic: a pair's d1 j1 - d2 j2 cancels by about
|r| / |r0| (at most 1e3 here), so FP64 sums agree to 1e3 eps64 = 2e-13 of
the largest velocity, times 50 for sums whose terms cancel; FP32 pairs to
1e3 eps32 = 6e-5 of it in the worst pair, below 2e-5 of the RMS summed."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _chain(n, m, seed, zero_core=False):
    """n connected segments of a jittered helix, points around it, a third of
    them end points of its segments."""
    rng = np.random.default_rng(seed)
    th = np.linspace(0.0, 0.05 * n, n + 1)
    x = np.stack([np.cos(th), np.sin(th), 0.02 * th], axis=1)
    x += 1e-3 * rng.standard_normal(x.shape)
    g, rc = rng.standard_normal(n), np.full(n, 0.02)
    if zero_core:
        rc[n // 2] = 0.0
    p = rng.uniform(-1.5, 1.5, size=(m, 3))
    k = m // 3
    p[:k] = x[rng.integers(0, n + 1, size=k)]
    return x[:-1], x[1:], g, rc, p


@pytest.mark.parametrize("zero_core", [False, True])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 1000])
@pytest.mark.parametrize("m", [191, 192, 257, 1030])
def test_fp64_groups_match_oracle(n, m, zero_core):
    from volcanor_amd import vlm
    ctx = vlm.Context(0)
    a, b, g, rc, p = _chain(n, m, n + m, zero_core)
    v, w = ctx.filament_vind(a, b, g, rc, p), orc.filament_sum(a, b, g, rc, p)
    assert np.max(np.abs(v - w)) <= 1e-11 * np.max(np.abs(w))
    # the same list resident on the device, every format of it
    fs = ctx.fset_create(a, b, g, rc)
    for k in (m, min(m, 40)):
        ps, mm = ctx.pset_create(p[:k])
        ctx.fset_vind(fs, ps)
        assert np.max(np.abs(ctx.pset_velocity(ps, mm) - w[:k])) <= 1e-11 * np.max(np.abs(w))
    ctx.close()


@pytest.mark.parametrize("n,m", [(33, 1024), (1000, 1151), (4099, 1153), (20011, 2048)])
def test_mixed_groups_match_oracle(n, m):
    from volcanor_amd import vlm
    ctx = vlm.Context(0)
    ctx.set_precision(vlm.MIXED)
    a, b, g, rc, p = _chain(n, m, n + m, zero_core=n == 1000)
    v, w = ctx.filament_vind(a, b, g, rc, p), orc.filament_sum(a, b, g, rc, p)
    rms = np.sqrt(np.mean(np.sum(w * w, axis=1)))
    assert np.max(np.abs(v - w)) <= 2e-5 * max(rms, 0.1 * np.max(np.abs(w)))
    ctx.close()
