"""The predictor's kernels at the edges of their tiles (16 samples), of the
workgroups of a training launch (512 tiles, then several tiles each) and of
the batches read in pinned memory (4 MiB: about 21800 samples), against the
FP64 oracle.  Tolerances: a layer sums 64 FP32 products (relative 64 eps32 =
8e-6 at worst), a gradient m of them with random rounding, 1e-5 of the
largest entry."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 15, 16, 17, 255, 2048, 8191, 8193, 21700, 23000])
def test_tiles_match_fp64_oracle(m):
    from volcanor_amd import vlm
    ctx = vlm.Context(0)
    rng = np.random.default_rng(m)
    p = (rng.normal(size=ctx.mlp_num_params()) * 0.15).astype(np.float32)
    x = rng.normal(size=(m, 45)).astype(np.float32)
    t = rng.normal(size=(m, 3)).astype(np.float32)
    ctx.mlp_set_params(p)
    y = ctx.mlp_forward(x)
    yo = orc.mlp_forward(p.astype(np.float64), x.astype(np.float64))
    assert np.max(np.abs(y - yo)) <= 3e-5 * np.max(np.abs(yo))
    loss, g = ctx.mlp_loss_grad(x, t)
    lo, go = orc.mlp_loss_grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64))
    assert loss == pytest.approx(lo, rel=1e-5)
    assert np.max(np.abs(g - go)) <= 1e-5 * np.max(np.abs(go))
    # repeated: the same bits, whatever order the workgroups ran in
    assert np.array_equal(ctx.mlp_loss_grad(x, t)[1], g)
