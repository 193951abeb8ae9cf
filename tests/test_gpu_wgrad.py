"""Weight and bias gradients of the network (csrc/fia_unet.hip conv3_wgrad_kernel) on boxes whose
levels do not divide into its 4 x 4 x 16 voxel tiles, layer by layer against the numpy oracle run
with the same BF16 rounding points.  Bars: those of test_gpu_unet.py, relative L2 <= 3e-2 and
cosine >= 0.999 of the whole gradient, 1e-1 per layer (few voxels decide the deepest levels).
"""
import numpy as np
import pytest

import unet
from test_gpu_unet import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(8, 8, 8), (8, 24, 40), (40, 8, 16), (16, 16, 72)])
def test_weight_gradient_matches_oracle(fia, ctx, shape):
    print("case wgrad", shape, flush=True)
    rng = np.random.default_rng(31)
    rhs = rng.normal(size=shape)
    p = unet.init_params(seed=8)
    net = fia.UNet(ctx, seed=1)
    try:
        net.set_params(p)
        _, _, g = net.loss_grad(rhs, None, loss="energy")
        _, _, again = net.loss_grad(rhs, None, loss="energy")
    finally:
        net.close()
    assert np.array_equal(g, again)
    pd = p.astype(np.float64)
    y, cache = unet.forward(pd, rhs, None, bf=True)
    _, dy = unet.loss(y, cache, unet.fluid_flags(None, shape), "energy")
    ref = unet.backward(pd, cache, dy)
    assert rel_l2(g, ref) <= 3e-2
    assert np.dot(g, ref) / (np.linalg.norm(g) * np.linalg.norm(ref)) >= 0.999
    for i, (ow, ob) in enumerate(unet.offsets()[0]):
        cout = unet.CONVS[i][1]
        assert rel_l2(g[ow:ob], ref[ow:ob]) <= 1e-1, ("weights", i)
        assert rel_l2(g[ob:ob + cout], ref[ob:ob + cout]) <= 1e-1, ("bias", i)
