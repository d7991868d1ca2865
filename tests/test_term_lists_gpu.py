"""Ordered term sums whose source lists share their launches: term counts on
both sides of the lists per launch (16), with sets that have no segments yet
(an unborn far wake) among them.  A list must contribute the bits that it
contributes alone, so the single-term calls are the reference and the
comparison is exact; one case is held to the oracle besides."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests import wake_harness as H

pytestmark = pytest.mark.gpu

CASE = dict(nb=2, nc=2, ns=5, nNwake=4, nFwake=3, nt=9, scheme=0, omega=30.0, vel=(0, 0, 1.0))


@pytest.mark.parametrize("steps", [1, 8])
@pytest.mark.parametrize("nterms", [1, 15, 16, 17, 35])
def test_shared_launches_equal_single_terms(nterms, steps):
    from volcanor_amd import vlm
    dev = vlm.Context(0)
    case = H.Case(**CASE)
    ir = H.setup(dev, case)
    for it in range(1, steps + 1):
        H.step(dev, case, ir, it)
    rng = np.random.default_rng(nterms)
    sets = [vlm.SET_WAKE, vlm.SET_WING, vlm.SET_WING_BOUND]
    terms = [(ir[0], sets[k % 3], bool(rng.random() < 0.4)) for k in range(nterms)]
    for m in (1, 4, 65, 191):
        p = rng.normal(size=(m, 3))
        for v0 in (None, rng.normal(size=(m, 3))):
            seq = np.zeros_like(p) if v0 is None else v0.copy()
            for i, s, neg in terms:
                seq = dev.rotor_induced_velocity(i, s, p, v=-seq if neg else seq)
            got = dev.induced_velocity_terms(terms, p, v=v0)
            assert np.array_equal(got, seq), (m, v0 is None)


def test_shared_launches_match_oracle():
    from volcanor_amd import vlm
    dev, ref = vlm.Context(0), orc.System()
    case = H.Case(**CASE)
    ia, ib = H.setup(dev, case), H.setup(ref, case)
    for it in range(1, 7):
        H.step(dev, case, ia, it)
        H.step(ref, case, ib, it)
    p = np.random.default_rng(3).normal(size=(50, 3))
    got = dev.induced_velocity_terms([(ia[0], s, s == 0) for s in (2, 1, 0)] * 7, p)
    want, scale = np.zeros_like(p), np.zeros_like(p)
    for s in (2, 1, 0) * 7:
        u = ref.rotor_induced_velocity(ib[0], s, p)
        want = (-want if s == 0 else want) + u
        scale += np.abs(u)
    assert np.all(np.abs(got - want) <= 1e-11 * np.max(scale))
