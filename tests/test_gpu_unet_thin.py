"""U-Net on volumes of few layers, whose convolutions take tiles of 8 and 4 layers
by 2 and 4 columns: whole and partial tiles at every level, narrow and wide
layers (one and two voxel tiles per wave); the oracle and bounds of the other
network tests."""
import pytest

import test_gpu_unet as unet
import test_gpu_unet_gradient_shapes as gradients

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,dims", [(8, (8, 40, 8)), (24, (12, 36, 8)), (32, (8, 20, 8)), (16, (4, 68, 4)), (32, (8, 36, 4)),
                                    (24, (20, 12, 12)), (8, (8, 8, 16))])
def test_forward(orc, xr, ctx, torch_dev, C, dims):
    unet.test_forward_matches_oracle(orc, xr, ctx, torch_dev, C, dims)


@pytest.mark.parametrize("C,dims", [(8, (8, 20, 8)), (24, (12, 20, 8)), (24, (8, 36, 4)), (16, (12, 12, 12))])
def test_gradients(orc, xr, ctx, torch_dev, C, dims):
    gradients.test_gradients_at_tile_edges(orc, xr, ctx, torch_dev, C, dims)
