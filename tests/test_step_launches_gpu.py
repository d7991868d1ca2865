"""The kernels that a step runs once per rotor where it ran several: the far
shift with rollup and near shift (more far filaments than one block of 256
lanes, no far wake, two near rows), the dissipation, and the wake download in
pieces (larger than one piece), against NumPy restatements of the copies and
the oracle's arithmetic (1e-13: a handful of roundings)."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _pair(nb, ns, nN, nF, seed, rollup=None):
    from volcanor_amd import vlm
    rng = np.random.default_rng(seed)
    w = dict(nodes=rng.normal(size=(nb, nN, ns + 1, 3)), le=rng.normal(size=(nb, ns + 1, 3)),
             gam=rng.uniform(0.5, 1.5, (nb, nN, ns)), rc4=rng.uniform(0.01, 0.1, (nb, nN, ns, 4)),
             far_fc=rng.normal(size=(nb, nF, 2, 3)), far_gam=rng.normal(size=(nb, nF)),
             far_rc=rng.uniform(0.01, 0.1, (nb, nF)))
    out = []
    for s in (vlm.Context(0), orc.System()):
        r = s.rotor_create(nb, 1, ns, nN, nF, nbConvect=nb, rollupStart=(rollup or (1, ns))[0],
                           rollupEnd=(rollup or (1, ns))[1], rollupMin=1, spanwiseCore=0.02,
                           streamwiseCoreVec=np.full(ns + 1, 0.02))
        s.rotor_set_wake(r, w, 1, 1)
        out.append((s, r))
    return w, out


@pytest.mark.parametrize("nb,ns,nN,nF", [(1, 1, 2, 1), (2, 3, 2, 255), (2, 3, 4, 256),
                                         (1, 300, 3, 257), (3, 5, 6, 600), (2, 4, 5, 0)])
def test_end_of_step_and_dissipation(nb, ns, nN, nF):
    w, pair = _pair(nb, ns, nN, nF, nF, rollup=(1 + ns // 4, ns))
    got = []
    for s, r in pair:
        s.rotor_begin_step(r, nN + nF + 1)
        s.rotor_dissipate_wake(r, 0.01, 1.8e-5, 50.0, 0.1)
        s.rotor_rollup(r)
        got.append(s.rotor_get_wake(r, (nb, ns, nN, nF)))
    for k in got[0]:
        a, b = got[0][k], got[1][k]
        assert a.shape == b.shape
        if a.size:
            assert np.max(np.abs(a - b)) <= 1e-13 * (1.0 + np.max(np.abs(b))), k


def test_wake_download_in_pieces():
    nb, ns, nN, nF = 2, 60, 1500, 7   # 0.9 M doubles
    w, ((dev, r), _) = _pair(nb, ns, nN, nF, 1)
    dims = (nb, ns, nN, nF)
    got = dev.rotor_get_wake(r, dims)
    for k in got:
        assert np.array_equal(got[k], w[k]), k
    dev.rotor_begin_step(r, nN + nF + 1)
    dev.rotor_rollup(r)                # the head moves: rows wrap around
    got = dev.rotor_get_wake(r, dims)
    assert np.array_equal(got["nodes"][:, 1:], w["nodes"][:, :-1])
    assert np.array_equal(got["nodes"][:, 0], w["nodes"][:, 0])
    assert np.array_equal(got["gam"][:, 1:], w["gam"][:, :-1])
    assert np.array_equal(got["rc4"][:, 1:], w["rc4"][:, :-1])
    assert np.array_equal(got["le"], w["le"])
