"""The default backprojection shape among those that can be set: reported and set
again, or found fastest by the autotuner, it is the default still (64^3 has a
kernel of its own, twice as fast as the shapes that can be named), and every
shape gives the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def fastest(torch, ctx, fn, runs=7):
    best = 1e30
    for _ in range(runs):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        ctx.synchronize()
        a.record()
        for _ in range(4):
            fn()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b))
    return best


def test_default_shape_survives_tuning(xr, torch_dev):
    import torch

    N, U, P = 64, 96, 90
    ctx = xr.Context(0)
    geom = xr.make_geometry(600.0, 300.0, 0.8, N, U, P, vox_size=0.4)
    plan = ctx.plan(geom, xr.Scan())
    g = torch.Generator(device=torch_dev).manual_seed(1)
    vol = torch.rand(N ** 3, device=torch_dev, generator=g) + 0.5
    img = torch.rand(P * U * U, device=torch_dev, generator=g) + 0.5
    work = vol.clone()
    codes = plan.codes(range(P))
    step = lambda: plan.backproject_update(img, codes, work)
    base = fastest(torch, ctx, step)
    reported = plan.tiles()
    plan.set_tiles(bwd_zpl=reported[0], bwd_gx=reported[1])
    assert fastest(torch, ctx, step) <= 1.4 * base
    plan.set_tiles()
    best, _ = plan.autotune(vol, img)
    assert fastest(torch, ctx, step) <= 1.4 * base
    plan.set_tiles(bwd_zpl=best[0], bwd_gx=best[1], fwd_rows=best[2])
    assert fastest(torch, ctx, step) <= 1.4 * base
    plan.close()
    ctx.close()


@pytest.mark.parametrize("N,U,V", [(24, 40, 36), (64, 96, 96), (64, 60, 40), (96, 140, 120), (160, 200, 210)])
def test_default_matches_other_shapes(xr, ctx, torch_dev, N, U, V):
    import torch

    P = 25
    geom = xr.make_geometry(600.0, 300.0, 0.8, N, U, P, vox_size=0.4, n_det_v=V)
    g = torch.Generator(device=torch_dev).manual_seed(3)
    img = torch.rand(P * U * V, device=torch_dev, generator=g) + 0.5
    start = torch.rand(N ** 3, device=torch_dev, generator=g)
    plan, fdk = ctx.plan(geom, xr.Scan()), ctx.plan(geom, xr.Scan(), convention=xr.CONV_FDK)
    codes = plan.codes(np.arange(P))

    def all_kinds(zpl, gx):
        out = [start.clone() for _ in range(4)] + [torch.zeros_like(start)]
        for p in (plan, fdk):
            p.set_tiles(bwd_zpl=zpl, bwd_gx=gx)
        plan.backproject_update(img, codes, out[0], method=xr.METHOD_MLEM)
        plan.backproject_update(img, codes, out[1], method=xr.METHOD_ART, lam=0.1, subset_size=P)
        plan.backproject(img, codes, out[2], out[4])
        fdk.fdk_backproject(img, codes, out[3], overwrite=False)
        ctx.synchronize()
        return out

    want = all_kinds(0, 0)
    for zpl, gx in ((1, 2), (2, 8), (4, 16), (1, 4), (2, 4), (4, 4)):
        for a, b in zip(all_kinds(zpl, gx), want):
            assert torch.equal(a, b), (zpl, gx)
    plan.close()
    fdk.close()
