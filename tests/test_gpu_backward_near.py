"""Backprojections near the source and on fine detectors, where a tile's
footprint changes several times over the volume: the default depth is chosen by
a typical one, fixed or any width, and the largest are read directly.  Every
voxel sums its views in order, so each shape gives the bits of the others."""
import numpy as np
import pytest

from test_gpu_parity import XTT_BASIS13, grating

pytestmark = pytest.mark.gpu

# N, voxel (mm), source to object (mm): footprints of the fixed width near the centre and wider at the edge; wide
# everywhere; so wide that one chunk is the most; directional ones with one voxel of the fixed width, and with two
CASES = {"fixed_and_wide": (260, 0.4, 200.0), "wide": (150, 0.6, 200.0), "widest": (100, 1.0, 200.0), "far": (140, 0.5, 1000.0)}


@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("K", [0, 3, 8, 13])
def test_default_depth_matches_set_ones(xr, ctx, torch_dev, case, K):
    import torch

    N, vs, sod = CASES[case]
    if K and N > 200:
        N = 140
    P, U, V = 18, int(2.6 * N * vs / 0.8), int(2.2 * N * vs / 0.8)
    geom = xr.make_geometry(2.0 * sod, sod, 0.8, N, U, P, vox_size=vs, n_det_v=V)
    plan = ctx.plan(geom, xr.Scan(basis=XTT_BASIS13[:K], grating=grating([30])) if K else xr.Scan())
    g = torch.Generator(device=torch_dev).manual_seed(6)
    img = torch.rand(P * U * V, device=torch_dev, generator=g) + 0.5
    start = torch.rand(max(K, 1) * N ** 3, device=torch_dev, generator=g)
    codes = plan.codes(range(P))

    def all_kinds():
        out = []
        for m in (xr.METHOD_MLEM, xr.METHOD_ART):
            v = start.clone()
            plan.backproject_update(img, codes, v, method=m, lam=0.1, subset_size=P, xtt=K > 0)
            out.append(v)
        t, f = start.clone(), torch.zeros_like(start)
        plan.backproject(img, codes, t, f, xtt=K > 0)
        ctx.synchronize()
        return out + [t, f]

    want = all_kinds()
    for zpl, gx in ((1, 2), (2, 4)) if K else ((1, 4), (2, 4), (4, 2)):
        plan.set_tiles(bwd_zpl=zpl, bwd_gx=gx)
        for a, b in zip(all_kinds(), want):
            assert torch.equal(a, b), (zpl, gx)
    plan.close()


@pytest.mark.parametrize("K", [3, 8, 13, 16])
@pytest.mark.parametrize("N", [66, 130])
def test_directional_two_voxels_match_one(xr, ctx, torch_dev, K, N):
    """More than 64 layers: two voxels per lane where the accumulators fit, the
    second chunk partial."""
    import torch

    rng = np.random.default_rng(2)
    basis = np.concatenate([XTT_BASIS13, rng.normal(size=(3, 3))])[:K]
    P, U, V = 10, (3 * N) // 2, (5 * N) // 4
    geom = xr.make_geometry(600.0, 300.0, 0.8, N, U, P, vox_size=0.4, n_det_v=V)
    plan = ctx.plan(geom, xr.Scan(basis=basis, grating=grating([60])))
    g = torch.Generator(device=torch_dev).manual_seed(5)
    img = torch.rand(P * U * V, device=torch_dev, generator=g) + 0.5
    start = torch.rand(K * N ** 3, device=torch_dev, generator=g)
    codes = plan.codes(range(P))

    def all_kinds():
        out = []
        for m in (xr.METHOD_MLEM, xr.METHOD_ART):
            v = start.clone()
            plan.backproject_update(img, codes, v, method=m, lam=0.1, subset_size=P, xtt=True)
            out.append(v)
        t, f = start.clone(), torch.zeros_like(start)
        plan.backproject(img, codes, t, f, xtt=True)
        ctx.synchronize()
        return out + [t, f]

    want = all_kinds()
    plan.set_tiles(bwd_zpl=1, bwd_gx=2)
    for a, b in zip(all_kinds(), want):
        assert torch.equal(a, b)
    plan.close()


@pytest.mark.parametrize("tilt", [25.0, 65.0])
def test_tilted_directional_two_voxels(orc, xr, ctx, torch_dev, tilt):
    """Tilted, K = 3, more than 64 layers: two voxels per lane whose footprint
    fits, against the FP64 oracle (1e-5 relative L2)."""
    import torch

    from conftest import rel_l2
    from test_gpu_parity import Setup, rot_x, to_dev

    N, K = 70, 3
    st = Setup(orc, xr, N=N, U=100, V=96, P=8, vs=0.25, cond_R=rot_x(tilt), basis=XTT_BASIS13[3:6], grating=grating([30]))
    rng = np.random.default_rng(4)
    img = rng.random((1, st.P, st.V, st.U)).astype(np.float32)
    plan = ctx.plan(st.geom, st.scan)
    n3, views = N ** 3, [0, 3, 5]
    tmp, fac = torch.zeros(K * n3, device=torch_dev), torch.zeros(K * n3, device=torch_dev)
    plan.backproject(to_dev(img, torch_dev), plan.codes(views), tmp, fac, xtt=True)
    tref, fref = torch.empty_like(tmp), torch.empty_like(fac)
    ctx.from_columns(tmp, tref, N, K)
    ctx.from_columns(fac, fref, N, K)
    plan.close()
    want_t, want_f = np.zeros(K * n3), np.zeros(K * n3)
    for v in views:
        st.case.backward_view(img[0, v], v, want_t, want_f, cond=0, xtt=True)
    got_t, got_f = tref.cpu().numpy(), fref.cpu().numpy()
    same = np.abs(got_f - want_f) <= 1e-4 * np.abs(want_f).max()
    assert np.count_nonzero(~same) <= 1e-4 * same.size
    assert rel_l2(got_t[same], want_t[same]) <= 1e-5
    assert rel_l2(got_f[same], want_f[same]) <= 1e-5
