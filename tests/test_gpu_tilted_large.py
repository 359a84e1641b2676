"""Tilted forward projection of a volume of more than 2^32 voxels (17 GB) with
the lanes along x or y: a launch of one view reads the volume strided, one of
two views reads a copy whose lane axis is contiguous.  The images are exact
fixed-point sums, so both give the same bits."""
import numpy as np
import pytest

from test_gpu_parity import rot_x, rot_y

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("axis", ["x", "y"])
def test_strided_reads_pass_32_bits(xr, ctx, torch_dev, axis):
    import torch

    N, U, P = 1632, 400, 2
    assert N ** 3 > 2 ** 32
    R = rot_x(90.0) if axis == "y" else rot_y(90.0)
    geom = xr.make_geometry(600.0, 300.0, 0.8, N, U, P, vox_size=0.08)
    plan = ctx.plan(geom, xr.Scan(cond_R=R.reshape(-1)))
    g = torch.Generator(device=torch_dev).manual_seed(7)
    vol = torch.rand(N ** 3, device=torch_dev, generator=g)
    both, apart = torch.zeros(P * U * U, device=torch_dev), torch.zeros(P * U * U, device=torch_dev)
    plan.project(vol, both, [0, 1], out_mode=xr.OUT_RAW)
    for c in (0, 1):
        plan.project(vol, apart, [c], out_mode=xr.OUT_RAW)
    ctx.synchronize()
    plan.close()
    assert float(both.sum()) > 0
    assert torch.equal(both, apart)
