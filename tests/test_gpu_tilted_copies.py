"""Which tilted forward launches copy the volume: those whose views have lanes
along x or y and read it often enough.  A plan that also holds such a condition
copies nothing for the views of its others, and what is copied is what the
launched views project (exact fixed-point sums: the images of one launch per
view, which never copies)."""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_parity import Setup, XTT_BASIS13, columns, grating, rot_x, rot_y

pytestmark = pytest.mark.gpu

N, U, P = 160, 200, 12
TILTS = [np.eye(3), rot_x(90.0), rot_y(80.0), rot_x(20.0)]  # lanes along z, y, x, z


@pytest.mark.parametrize("K", [0, 3])
def test_copies_follow_the_views(xr, ctx, torch_dev, K):
    import torch

    geom = xr.make_geometry(600.0, 300.0, 0.8, N, U, P, vox_size=0.4)
    kw = dict(basis=XTT_BASIS13[:K], grating=grating([0, 30, 60, 90])) if K else {}
    plan = ctx.plan(geom, xr.Scan(cond_R=np.concatenate([R.reshape(-1) for R in TILTS]), **kw))
    g = torch.Generator(device=torch_dev).manual_seed(4)
    vol = torch.rand((K or len(TILTS)) * N ** 3, device=torch_dev, generator=g)
    total = len(TILTS) * P * U * U
    apart = torch.zeros(total, device=torch_dev)
    for c in range(len(TILTS) * P):
        plan.project(vol, apart, [c], out_mode=xr.OUT_RAW, xtt=K > 0)

    out = torch.zeros(total, device=torch_dev)
    torch.equal(out[:U * U], apart[:U * U])

    def project(views):
        out.zero_()
        plan.project(vol, out, np.array(views, np.int32), out_mode=xr.OUT_RAW, xtt=K > 0)
        ctx.synchronize()
        for c in views:
            at = slice(c * U * U, (c + 1) * U * U)
            assert torch.equal(out[at], apart[at]), (views, c)

    free = torch.cuda.mem_get_info()[0]
    project(range(P))                                    # the untilted condition
    project(range(3 * P, 4 * P))                         # 20 degrees: lanes along z
    project([0, P + 1, 3 * P])                           # one view with lanes along y
    assert torch.cuda.mem_get_info()[0] >= free - N ** 3  # no copy (N^3 floats) was made
    project(range(P, 2 * P))
    project(range(2 * P, 3 * P))
    project([0, 1, P, P + 1, P + 2, P + 3, 3 * P])
    project([P, P + 5, 2 * P, 2 * P + 1, 2 * P + 2, 2 * P + 3])
    project(range(len(TILTS) * P))
    plan.close()


@pytest.mark.parametrize("N,U,V,K", [(20, 34, 30, 0), (65, 90, 100, 0), (150, 190, 240, 0), (270, 200, 180, 0), (64, 90, 80, 3),
                                     (130, 190, 150, 4)])
def test_untilted_views_of_a_mixed_plan(orc, xr, ctx, torch_dev, N, U, V, K):
    """They are splat by whole columns: against the FP64 oracle (1e-5 relative L2,
    without the two outermost rows and columns, as the tilted ones)."""
    import torch

    R = np.concatenate([np.eye(3).reshape(-1), rot_x(50.0).reshape(-1)])
    st = Setup(orc, xr, N=N, U=U, V=V, P=9, vs=0.4, cond_R=R, basis=XTT_BASIS13[:K] if K else None)
    xtt, ch = K > 0, max(K, 1)
    rng = np.random.default_rng(N)
    vol = (rng.random((ch, N, N, N), dtype=np.float32) * 0.02).astype(np.float32)
    vcol = columns(ctx, vol if xtt else np.concatenate([vol, vol]), N, ch if xtt else 2, torch_dev)
    plan = ctx.plan(st.geom, st.scan)
    proj = torch.zeros(2 * st.P * V * U, device=torch_dev)
    plan.project(vcol, proj, np.arange(2 * st.P), out_mode=xr.OUT_RAW, xtt=xtt)
    got = proj.cpu().numpy().reshape(2, st.P, V, U)
    plan.close()
    for c, v in ((0, 1), (0, 5), (1, 5)):
        want, _ = st.case.forward_view(vol if xtt else vol[0], v, cond=c, xtt=xtt, normalise=False)
        assert rel_l2(got[c, v, 2:-2, 2:-2], want[2:-2, 2:-2]) <= 1e-5
