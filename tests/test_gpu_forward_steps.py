"""Steps of the untilted forward's column loop, as test_gpu_forward_shapes.py
checks them (bits of other work splits, the FP64 oracle): directional volumes of
one to three chunks of 64 layers, whole and partial, the basis count equal to
and below a compiled one; plain volumes of two to seven chunks, whole and
partial, which a column takes in one step."""
import pytest

import test_gpu_forward_shapes as shapes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,U,V,K", [(64, 100, 96, 13), (64, 100, 50, 3), (64, 90, 90, 8), (127, 180, 180, 4),
                                     (128, 180, 190, 3), (128, 180, 120, 10), (129, 190, 190, 16), (192, 280, 280, 3)])
def test_directional_steps(orc, xr, ctx, torch_dev, N, U, V, K):
    shapes.test_forward_depths(orc, xr, ctx, torch_dev, N, U, V, K)


@pytest.mark.parametrize("N,U,V", [(128, 180, 190), (150, 210, 220), (192, 260, 200), (320, 400, 440), (330, 420, 300),
                                   (384, 500, 500), (430, 300, 600)])
def test_plain_steps(orc, xr, ctx, torch_dev, N, U, V):
    shapes.test_forward_depths(orc, xr, ctx, torch_dev, N, U, V, 0)
