"""Steps of the untilted forward's column loop, as test_gpu_forward_shapes.py
checks them (bits of other work splits, the FP64 oracle): directional volumes of
one to three chunks of 64 layers, whole and partial, the basis count equal to
and below a compiled one."""
import pytest

import test_gpu_forward_shapes as shapes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,U,V,K", [(64, 100, 96, 13), (64, 100, 50, 3), (64, 90, 90, 8), (127, 180, 180, 4),
                                     (128, 180, 190, 3), (128, 180, 120, 10), (129, 190, 190, 16), (192, 280, 280, 3)])
def test_directional_steps(orc, xr, ctx, torch_dev, N, U, V, K):
    shapes.test_forward_depths(orc, xr, ctx, torch_dev, N, U, V, K)
