"""Tilted forward projections at the edges of their lane packing: the lane axis
along x, y and z, volume edges around 64 and odd, detectors that cut the
volume: the raw splat against the FP64 oracle (1e-5 relative L2 as everywhere).  The images
are fixed-point sums over exact per-voxel tests, so a launch over many views
(which copies the volume for lanes along x or y) and one launch per view
(which reads it strided) give the same bits."""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_parity import Setup, XTT_BASIS13, columns, rot_x, rot_y

pytestmark = pytest.mark.gpu

TILTS = {"x45": rot_x(45.0), "x60": rot_x(60.0), "y70": rot_y(70.0), "x90": rot_x(90.0), "y35x35": rot_y(35.0) @ rot_x(35.0)}


@pytest.mark.parametrize("tilt", list(TILTS))
@pytest.mark.parametrize("N,U,V,K", [(33, 50, 44, 0), (65, 80, 96, 0), (20, 40, 30, 13), (24, 40, 36, 3)])
def test_tilted_forward(orc, xr, ctx, torch_dev, tilt, N, U, V, K):
    import torch

    R = np.concatenate([np.eye(3).reshape(-1), TILTS[tilt].reshape(-1)])
    st = Setup(orc, xr, N=N, U=U, V=V, P=12, vs=0.6, cond_R=R, basis=XTT_BASIS13[:K] if K else None)
    rng = np.random.default_rng(5)
    xtt, ch = K > 0, max(K, 1)
    vol = (rng.random((ch, N, N, N)) * 0.02).astype(np.float32)
    # a plain volume per condition, or K coefficients shared by both
    vcol = columns(ctx, vol if xtt else np.concatenate([vol, vol]), N, ch if xtt else 2, torch_dev)
    plan = ctx.plan(st.geom, st.scan)
    codes = np.arange(2 * st.P, dtype=np.int32)
    proj = torch.zeros(2 * st.P * V * U, device=torch_dev)
    plan.project(vcol, proj, codes, out_mode=xr.OUT_RAW, xtt=xtt)
    apart = torch.zeros_like(proj)
    for c in codes:
        plan.project(vcol, apart, [c], out_mode=xr.OUT_RAW, xtt=xtt)
    assert torch.equal(proj, apart)
    got = proj.cpu().numpy().reshape(2, st.P, V, U)
    src = vol if xtt else vol[0]
    for v in (0, 3, 7):
        want, _ = st.case.forward_view(src, v, cond=1, xtt=xtt, normalise=False)
        # a voxel within rounding of the acceptance window (0.55 < u < U - 0.55)
        # may fall on either side of it in FP32 and FP64; it touches only the
        # detector's two outermost rows and columns
        assert rel_l2(got[1, v, 2:-2, 2:-2], want[2:-2, 2:-2]) <= 1e-5
    plan.close()
