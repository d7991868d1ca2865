"""Small cores: targets far from a straight chain and close to its axis,
where |r1 x r2|^2 is small against (|r0| |r1|)^2 and only the core bounds the
denominator, on both sides of the distances (2^10 and 2^24 core radii) at
which the far pairs change their form, against the FP64 oracle.

Tolerance: d1 / |r1| - d2 / |r2| carries a rounding error of about 3 eps |r0|;
times |c| / sqrt(q^2 + |c|^4), at most 1 / (sqrt(2) rc |r0|), a unit pair is
off by up to 2 eps / rc.  Twice that per pair, and in FP64 the same again for
the oracle, whose formula has the same difference."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _axis_case(n, r0, rc, dist, angle, m, seed):
    """n collinear segments of length r0 about the origin, m targets at
    distances and angles off their axis spread over the given decades."""
    rng = np.random.default_rng(seed)
    u = rng.standard_normal(3)
    u /= np.linalg.norm(u)
    w = np.cross(u, rng.standard_normal((m, 3)))
    w /= np.linalg.norm(w, axis=1)[:, None]
    th = 10.0 ** rng.uniform(*angle, size=m)
    d = 10.0 ** rng.uniform(*dist, size=m) * rng.choice([-1.0, 1.0], size=m)
    x = (np.arange(n + 1) - 0.5 * n)[:, None] * r0 * u
    p = d[:, None] * (np.cos(th)[:, None] * u + np.sin(th)[:, None] * w)
    return x[:-1], x[1:], rng.choice([-1.0, 1.0], size=n), np.full(n, rc), p


@pytest.mark.parametrize("n", [1, 32, 70])
@pytest.mark.parametrize("rc", [1e-2, 1e-3, 1e-4, 1e-5, 1e-6])
def test_mixed_small_cores_off_the_axis(n, rc):
    from volcanor_amd import vlm
    a, b, g, r, p = _axis_case(n, 0.01, rc, (0.0, 0.6), (-5.0, -2.0), 20000, n)
    ctx = vlm.Context(0)
    ctx.set_precision(vlm.MIXED)
    v, w = ctx.filament_vind(a, b, g, r, p), orc.filament_sum(a, b, g, r, p)
    ctx.close()
    assert np.max(np.linalg.norm(v - w, axis=1)) <= n * 4 * 2.0**-24 / rc / (4 * np.pi)


@pytest.mark.parametrize("n,dist", [(1, (0.6, 0.75)), (32, (1.4, 1.6))])
@pytest.mark.parametrize("rc", [1.1e-9, 5e-9, 1e-6])
def test_fp64_small_cores_off_the_axis(n, dist, rc):
    from volcanor_amd import vlm
    a, b, g, r, p = _axis_case(n, 1.0, rc, dist, (-11.0, -1.0), 100000, n)
    ctx = vlm.Context(0)
    v, w = ctx.filament_vind(a, b, g, r, p), orc.filament_sum(a, b, g, r, p)
    ctx.close()
    assert np.max(np.linalg.norm(v - w, axis=1)) <= n * 8 * 2.0**-53 / rc / (4 * np.pi)


@pytest.mark.parametrize("shuffle", [False, True])
def test_mixed_tiles_of_near_and_far_targets(shuffle):
    """Every pair of halves of a 128-target tile: beside the chain, within
    2^10 core radii of it and past them; and (shuffled) every target order.
    Near pairs obey the same bound."""
    from volcanor_amd import vlm
    rng = np.random.default_rng(11)
    n, rc = 40, 1e-3
    a, b, g, r, p = _axis_case(n, 0.01, rc, (0.0, 0.0), (-3.0, 0.4), 18 * 64 + 30, 7)
    radii = {"near": (-2.0, -0.9), "far": (-0.3, -0.1), "past": (0.3, 0.6)}
    pairs = [x for q in radii for s in radii for x in (q, s)] + ["near"]
    scale = np.concatenate([10.0 ** rng.uniform(*radii[q], size=64) for q in pairs])[:len(p)]
    p = p * scale[:, None]
    if shuffle:
        p = p[rng.permutation(len(p))]
    ctx = vlm.Context(0)
    ctx.set_precision(vlm.MIXED)
    v, w = ctx.filament_vind(a, b, g, r, p), orc.filament_sum(a, b, g, r, p)
    ctx.close()
    assert np.max(np.linalg.norm(v - w, axis=1)) <= n * 4 * 2.0**-24 / rc / (4 * np.pi)
