"""Tilted backprojections at the limits of their arithmetic."""
import numpy as np
import pytest

from test_gpu_parity import Setup, rot_x, rot_y, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [rot_x(30.0), rot_y(70.0)], ids=["x30", "y70"])
@pytest.mark.parametrize("U", [40, 26])  # tiles inside the window; a detector that cuts the volume
def test_infinite_texels_stay_infinite(orc, xr, ctx, torch_dev, R, U):
    """A detector pixel without a count is infinite after -log.  A voxel whose
    sample takes a share of it becomes infinite and no other does: the four
    weighted terms of the oracle, 0.55 < u, v < U - 0.55."""
    import torch

    st = Setup(orc, xr, N=22, U=U, P=8, vs=0.5, cond_R=R)
    rng = np.random.default_rng(3)
    img = rng.random((st.P, st.V, st.U)).astype(np.float32) + 0.5
    for v in range(st.P):
        img[v, rng.integers(0, st.V, 6), rng.integers(0, st.U, 6)] = np.inf
    plan = ctx.plan(st.geom, st.scan)
    n3 = st.N ** 3
    tmp, fac = torch.zeros(n3, device=torch_dev), torch.zeros(n3, device=torch_dev)
    views = [1, 4, 6]
    plan.backproject(to_dev(img, torch_dev), plan.codes(views), tmp, fac)
    tref, fref = torch.empty_like(tmp), torch.empty_like(fac)
    ctx.from_columns(tmp, tref, st.N, 1)
    ctx.from_columns(fac, fref, st.N, 1)
    want_t, want_f = np.zeros(n3), np.zeros(n3)
    for v in views:
        st.case.backward_view(img[v], v, want_t, want_f)
    got, same = tref.cpu().numpy(), fref.cpu().numpy() == want_f
    plan.close()
    # a voxel within rounding of the acceptance window may fall on either side
    assert np.count_nonzero(~same) <= 1e-4 * n3
    assert np.isinf(want_t).sum() > 20 and not np.isnan(want_t).any()
    assert not np.isnan(got).any()
    # a sample within FP32 rounding of a texel's edge takes a share of it in one precision alone
    assert np.count_nonzero(np.isinf(got[same]) != np.isinf(want_t[same])) <= 2


@pytest.mark.parametrize("R", [rot_y(45.0), rot_x(90.0)], ids=["y45", "x90"])
def test_xtt_weights_are_not_negative(xr, ctx, torch_dev, R):
    """|B x S|^2 vanishes where the ray runs along the scattering direction S;
    rounding must not leave a weight below zero there: the denominator of the
    MLEM quotient is a sum of weights.  S along the view's central ray and next
    to it, and a grating vector that is not normal to it."""
    import torch

    N, U, P = 65, 100, 16
    rng = np.random.default_rng(1)
    geom = xr.make_geometry(600.0, 300.0, 0.8, N, U, P, vox_size=0.5)
    n3 = N ** 3
    img = torch.ones(P * U * U, device=torch_dev)
    vol, proj = torch.ones(3 * n3, device=torch_dev), torch.zeros(P * U * U, device=torch_dev)
    for view in range(1, P, 2):
        th = 2.0 * np.pi * view / P
        d = R @ np.array([-np.sin(th), np.cos(th), 0.0])  # condition rotation and view angle on the y axis
        e = np.cross(d, rng.normal(size=3))
        basis = np.stack([d, d + 1e-4 * e, d - 2e-4 * e]).astype(np.float32)
        plan = ctx.plan(geom, xr.Scan(cond_R=R.reshape(-1), basis=basis, grating=np.array([0.6, 0.7, 0.5])))
        tmp, fac = torch.zeros(3 * n3, device=torch_dev), torch.zeros(3 * n3, device=torch_dev)
        plan.backproject(img, plan.codes([view]), tmp, fac, xtt=True)
        plan.project(vol, proj, plan.codes([view]), out_mode=xr.OUT_RAW, xtt=True)
        ctx.synchronize()
        plan.close()
        assert float(fac.max()) > 0.0
        assert float(fac.min()) >= 0.0 and float(tmp.min()) >= 0.0 and float(proj.min()) >= 0.0
