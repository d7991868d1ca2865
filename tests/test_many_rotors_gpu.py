"""The launches that serve all rotors of a step, with more rotors than one
launch describes (12 wake updates, 12 target sets, 20 source sets), an image
in the middle of the order, ragged sizes, a rotor without a far wake and an
axisymmetric one, for each scheme that the oracle has, step by step against the oracle."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests import wake_harness as H
from tests.test_wake_gpu import compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", [0, 1, 2, 3])
def test_sixteen_rotors_match_oracle(scheme):
    from volcanor_amd import vlm
    surfaces = []
    for k in range(16):
        d = dict(nb=1 + k % 2, nc=1, ns=2 + k % 3, nNwake=3 + k % 4, nFwake=k % 4, rollup=(1, 2),
                 span=0.5, root=0.1, hub=(1.1 * k, 0.0, 0.3 * (k % 5)), omega=20.0)
        if k == 9:
            d.update(nb=2, axisym=True)
        surfaces.append(d)
    surfaces[13] = dict(surfaces[6], image=(6, 3))
    case = H.Case(scheme=scheme, nt=7, dt=0.01, vel=(0.0, 0.0, 1.0), surfaces=surfaces)
    dev, ref = vlm.Context(0), orc.System()
    ia, ib = H.setup(dev, case), H.setup(ref, case)
    for it in range(1, case.nt + 1):
        H.step(dev, case, ia, it)
        H.step(ref, case, ib, it)
        compare(H.snapshot(dev, case, ia), H.snapshot(ref, case, ib), case)


def test_initial_wake_velocity_adds_to_the_windows():
    """Two equal states, one of them stepped with an initial wake velocity:
    pass 1 differs by + u along the shaft on the active near rows and - u on
    the active far filaments (one rounding of each sum), nowhere else."""
    from volcanor_amd import vlm
    case = H.Case(nb=2, nc=1, ns=4, nNwake=4, nFwake=6, scheme=0, omega=20.0, dt=0.01,
                  vel=(0.0, 0.0, 1.0))
    vel = []
    for u in (0.0, 0.7):
        dev = vlm.Context(0)
        ir = H.setup(dev, case)
        for it in range(1, 8):
            if it == 7:
                dev.rotor_set_init_wake_vel(ir[0], u, 99)
            H.step(dev, case, ir, it)
        vel.append(dev.rotor_get_velocity(ir[0], 0, case.dims))
        rn, rf = dev.rotor_cursors(ir[0])
    (n0, f0), (n1, f1) = vel
    wn, wf = np.zeros_like(n0), np.zeros_like(f0)
    wn[:, rn - 1:, :, 2] = 0.7
    wf[:, rf - 1:, 2] = -0.7
    assert 1 < rf <= case.nFwake
    assert np.max(np.abs(n1 - n0 - wn)) <= 1e-14 * (1 + np.max(np.abs(n0)))
    assert np.max(np.abs(f1 - f0 - wf)) <= 1e-14 * (1 + np.max(np.abs(f0)))
