"""U-Net gradients where the gradient kernels can go wrong: dims that leave
partial 2 x 4 x 32 tiles at every level, one-voxel dims at the lowest level,
channel counts that leave a half-filled or a second 32-channel block, and data
gradients of more than 96 channels (two pieces).  Same oracle and bounds as
the other gradient tests: 5e-2 relative L2 per layer (BF16 rounding points that
land one step away), 1e-3 for the loss."""
import numpy as np
import pytest

from test_gpu_unet import dev, layer_slices
from test_oracle_unet import random_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,dims", [(8, (4, 4, 4)), (16, (4, 12, 36)), (24, (12, 4, 68)), (24, (8, 20, 28))])
def test_gradients_at_tile_edges(orc, xr, ctx, torch_dev, C, dims):
    net = xr.UNet(ctx, C, seed=1)
    p = random_params(orc, C, 60 + C)
    net.set_params(p)
    rng = np.random.default_rng(200 + C)
    x = rng.uniform(0.0, 0.05, dims).astype(np.float32)
    t = np.maximum(x + rng.normal(0, 0.005, dims), 0).astype(np.float32)
    s = float(x.mean())
    print("C", C, "dims", dims, flush=True)
    loss = net.loss_grad(dev(x, torch_dev), dev(t, torch_dev), dims, scale=s)
    g = net.grads()
    want_loss, want = orc.unet_loss_grad(p, C, x, t, s, emulate_bf16=True)
    assert abs(loss - want_loss) <= 1e-3 * want_loss
    for name, sl in layer_slices(C):
        w, gg = want[sl], g[sl]
        if name == "W0":  # only input channel 0 carries data
            w = w.reshape(C, 27, 8)[:, :, 0].reshape(-1)
            gg = gg.reshape(C, 27, 8)[:, :, 0].reshape(-1)
        err = np.linalg.norm(gg - w) / max(np.linalg.norm(w), 1e-30)
        print("  ", name, "rel err", err, flush=True)
        assert err <= 5e-2, name
    net.close()
