"""Weight and bias gradients of the network layer by layer (csrc/fia_unet.hip conv3_wgrad_kernel) where
nothing else rounds: a network of a few weights of +-1/2 and 1 per output channel, on a right-hand side
of +-1 over a power of two of voxels, where every value before a rounding is exact in FP32 (checked here
on the oracle's FP64 values), so that the GPU and the oracle round the same values
to BF16 and the layers' gradients differ by the FP32 sums over the voxels alone.

Bar: relative L2 <= 1e-5 per layer.  A sum of n terms in FP32 strays by some sqrt(n) roundings of 2^-24 of
a term's size, and is itself some sqrt(n) terms large: some 1e-7; the bar leaves a factor of 100.
"""
import numpy as np
import pytest

import unet
from test_gpu_unet import rel_l2

pytestmark = pytest.mark.gpu


def _exact_params(seed):
    """Two weights of +-1/2 or 1 per output channel, biases of 1/2 or 1 (they keep ReLU open)."""
    rng = np.random.default_rng(seed)
    offs, oo, n = unet.offsets()
    p = np.zeros(n, dtype=np.float32)
    for (cin, cout, _, real), (ow, ob) in zip(unet.CONVS, offs):
        W = np.zeros((27, cout, cin))
        for co in range(cout):
            for ci in rng.choice(real, size=2, replace=False):
                W[rng.integers(27), co, ci] = rng.choice([1.0, 0.5, -0.5])
        p[ow:ow + W.size] = W.reshape(-1)
        p[ob:ob + cout] = rng.choice([0.5, 1.0], size=cout)
    p[oo:oo + 16] = rng.choice([0.5, -0.5, 0.25], size=16)
    p[oo + 16] = 0.5
    return p


@pytest.mark.parametrize("shape", [(16, 16, 16), (8, 32, 64), (64, 8, 16)])
def test_layer_gradients_match_oracle(fia, ctx, monkeypatch, shape):
    print("case wgrad layers", shape, flush=True)
    rhs = np.random.default_rng(37).choice([-1.0, 1.0], size=shape)
    p = _exact_params(9)
    net = fia.UNet(ctx, seed=1)
    try:
        net.set_params(p)
        _, _, g = net.loss_grad(rhs, None, loss="energy")
    finally:
        net.close()

    # everything that the oracle rounds, to BF16 or to FP32, is an FP32 value before
    plain = {name: getattr(unet, name) for name in ("bf16", "f32")}

    def checked(name):
        def rounded(x):
            assert np.array_equal(plain["f32"](x), np.asarray(x, dtype=np.float64)), name
            return plain[name](x)
        return rounded

    for name in plain:
        monkeypatch.setattr(unet, name, checked(name))
    pd = p.astype(np.float64)
    y, cache = unet.forward(pd, rhs, None, bf=True)
    assert cache["scale"] == 1.0
    _, dy = unet.loss(y, cache, unet.fluid_flags(None, shape), "energy")
    ref = unet.backward(pd, cache, dy)
    errs = []
    for i, (ow, ob) in enumerate(unet.offsets()[0]):
        cout = unet.CONVS[i][1]
        assert np.count_nonzero(ref[ow:ob]) > 0 and np.count_nonzero(ref[ob:ob + cout]) > 0
        errs.append((rel_l2(g[ow:ob], ref[ow:ob]), rel_l2(g[ob:ob + cout], ref[ob:ob + cout])))
    print("relative L2 by layer (weights/bias): " + " ".join("%.1e/%.1e" % e for e in errs), flush=True)
    for i, (w, b) in enumerate(errs):
        assert w <= 1e-5 and b <= 1e-5, i
