"""Backprojection kernels that the default tile choice reaches: the small-volume
kernel (eight views per barrier), z depths of 1 to 5 chunks, footprints wider
than the fixed staging width, view counts at the edges of the groups of 2 and
8 and the batches of 16, tilted tiles inside and across the detector's edge.
Each voxel sums its views in order whatever the shape, so every shape gives
the bits of the explicitly set ones; tilted tiles are compared with the FP64
oracle (1e-5 relative L2, counts exact up to window rounding, as in the parity
tests)."""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_parity import Setup, XTT_BASIS13, columns, grating, rot_x, rot_y, to_dev

pytestmark = pytest.mark.gpu

# N, U, V, voxel size: one chunk (small kernel), 2, 3 and 5 chunks; a detector
# that cuts the volume; more than 1.4 pixels per voxel (wide footprints)
SHAPES = {"n24": (24, 40, 36, 0.5), "n64": (64, 96, 96, 0.4), "n66": (66, 100, 90, 0.4), "n150_cut": (150, 180, 130, 0.4),
          "n300": (300, 460, 420, 0.4), "n64_wide": (64, 200, 180, 0.8), "n140_wide": (140, 460, 400, 0.8)}


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("kind", ["raw", "mlem", "art", "fdk"])
def test_default_shape_matches_set_shapes(xr, ctx, torch_dev, shape, kind):
    import torch

    N, U, V, vs = SHAPES[shape]
    P = 36
    geom = xr.make_geometry(600.0, 300.0, 0.8, N, U, P, vox_size=vs, n_det_v=V)
    plan = ctx.plan(geom, xr.Scan(), convention=xr.CONV_FDK if kind == "fdk" else xr.CONV_IR)
    g = torch.Generator(device=torch_dev).manual_seed(3)
    img = torch.rand(P * U * V, device=torch_dev, generator=g) + 0.5
    start = torch.rand(N ** 3, device=torch_dev, generator=g)

    def once(codes):
        v, f = start.clone(), torch.zeros_like(start)
        if kind == "raw":
            plan.backproject(img, codes, v, f)
        elif kind == "fdk":
            plan.fdk_backproject(img, codes, v, overwrite=False)
        else:
            plan.backproject_update(img, codes, v, method=xr.METHOD_MLEM if kind == "mlem" else xr.METHOD_ART, lam=0.1,
                                    subset_size=len(codes))
        ctx.synchronize()
        return v, f

    for nv in (1, 2, 3, 7, 8, 9, 16, 17, 33, 36):
        codes = plan.codes(np.arange(nv) * 5 % P)
        plan.set_tiles()
        v, f = once(codes)
        plan.set_tiles(bwd_zpl=1, bwd_gx=4)
        w, h = once(codes)
        assert torch.equal(v, w) and torch.equal(f, h), (shape, kind, nv)
    plan.close()


@pytest.mark.parametrize("xtt_k", [0, 3, 13])
@pytest.mark.parametrize("tilt", ["x30", "y60", "x90"])
def test_tilted_backward(orc, xr, ctx, torch_dev, tilt, xtt_k):
    import torch

    R = {"x30": rot_x(30.0), "y60": rot_y(60.0), "x90": rot_x(90.0)}[tilt]
    N = 70 if xtt_k == 0 else 36
    st = Setup(orc, xr, N=N, U=N + 20, V=N + 6, P=20, vs=0.5, cond_R=R, basis=XTT_BASIS13[:xtt_k] if xtt_k else None,
               grating=grating([30]) if xtt_k else None)
    rng = np.random.default_rng(11)
    img = rng.random((1, st.P, st.V, st.U)).astype(np.float32)
    plan = ctx.plan(st.geom, st.scan)
    K, n3 = max(xtt_k, 1), N ** 3
    views = list(range(0, 20, 3))
    tmp, fac = torch.zeros(K * n3, device=torch_dev), torch.zeros(K * n3, device=torch_dev)
    plan.backproject(to_dev(img, torch_dev), plan.codes(views), tmp, fac, xtt=xtt_k > 0)
    tref, fref = torch.empty_like(tmp), torch.empty_like(fac)
    ctx.from_columns(tmp, tref, N, K)
    ctx.from_columns(fac, fref, N, K)
    want_t, want_f = np.zeros(K * n3), np.zeros(K * n3)
    for v in views:
        st.case.backward_view(img[0, v], v, want_t, want_f, **({"cond": 0, "xtt": True} if xtt_k else {}))
    got_t, got_f = tref.cpu().numpy(), fref.cpu().numpy()
    # a voxel within rounding of the acceptance window may fall on either side
    same = np.abs(got_f - want_f) <= 1e-4 * np.abs(want_f).max() if xtt_k else got_f == want_f
    assert np.count_nonzero(~same) <= 1e-4 * same.size
    assert rel_l2(got_t[same], want_t[same]) <= 1e-5
    if xtt_k:
        assert rel_l2(got_f[same], want_f[same]) <= 1e-5
    plan.close()
