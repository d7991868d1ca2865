"""Which launches the kernel timing counts: every one of the grouped kernels
with its time and pairs, those of few pairs only in the total."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,mixed,timed", [
    (300, 100001, False, True), (300, 2000, False, False), (640, 46876, False, True),
    (640, 46875, False, False), (1200, 2000, False, False), (1200, 2000, True, True),
    (2049, 10, False, True), (20, 200000, False, False), (700, 100000, True, True)])
def test_timed_launches(m, n, mixed, timed):
    from volcanor_amd import vlm
    rng = np.random.default_rng(1)
    a, b = rng.uniform(-2, 2, size=(2, n, 3))
    ctx = vlm.Context(0)
    ctx.set_precision(vlm.MIXED if mixed else vlm.FP64)
    fs = ctx.fset_create(a, b, rng.normal(size=n), np.full(n, 0.02))
    ps, _ = ctx.pset_create(rng.uniform(-2, 2, size=(m, 3)))
    ctx.profile_enable(True)
    ctx.profile_reset()
    for _ in range(2):
        ctx.fset_vind(fs, ps)
    ms, count, pairs = ctx.profile_get()
    assert (count, pairs, ms > 0) == ((2, 2 * m * n, True) if timed else (0, 0, False))
    assert ctx.profile_get_all() == (2 * m * n, 2)
    ctx.close()
