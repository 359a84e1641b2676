"""Orientation-aware XTT backprojection at volume edges that are no multiple of
the 2 x 4 column tile: the waves past the volume have no orientation of their
own to read.  Detectors wide enough that the edge tiles lie inside the
acceptance window, and one that cuts the volume; one and two z chunks; against
the FP64 oracle (1e-5 relative L2, as the parity tests)."""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_orth import BASIS3
from test_gpu_parity import Setup, columns, grating, rot_x, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tilt", [0.0, 20.0, 75.0])
@pytest.mark.parametrize("N,U", [(21, 64), (22, 64), (23, 64), (25, 30), (66, 140), (67, 140)])
def test_orth_backward_matches_oracle(orc, xr, ctx, torch_dev, N, U, tilt):
    import torch

    cond_R = np.concatenate([np.eye(3).reshape(-1), rot_x(tilt).reshape(-1)])
    st = Setup(orc, xr, N=N, U=U, P=10, vs=0.5, cond_R=cond_R, basis=BASIS3, grating=grating([0, 60]))
    K, N3 = 3, N ** 3
    rng = np.random.default_rng(N)
    coef = np.stack([rng.uniform(-np.pi, np.pi, (N, N, N)), rng.uniform(-1.0, 1.0, (N, N, N))]).astype(np.float32)
    img = rng.random((2, st.P, st.V, st.U)).astype(np.float32)
    views = [0, 3, 7]
    codes = np.concatenate([np.array(views) + c * st.P for c in range(2)])
    plan = ctx.plan(st.geom, st.scan)
    ccol = columns(ctx, coef, N, 2, torch_dev)
    plan.set_orientation(ccol)
    tmp, fac = torch.zeros(K * N3, device=torch_dev), torch.zeros(K * N3, device=torch_dev)
    plan.backproject(to_dev(img, torch_dev), codes, tmp, fac, xtt=True)
    tref, fref = torch.empty_like(tmp), torch.empty_like(fac)
    ctx.from_columns(tmp, tref, N, K)
    ctx.from_columns(fac, fref, N, K)
    want_t, want_f = np.zeros(K * N3), np.zeros(K * N3)
    for c in range(2):
        for v in views:
            st.case.backward_view_orth(img[c, v], coef, v, want_t, want_f, cond=c)
    got_t, got_f = tref.cpu().numpy(), fref.cpu().numpy()
    # a voxel within rounding of the acceptance window may fall on either side
    same = np.abs(got_f - want_f) <= 1e-4 * np.abs(want_f).max()
    assert np.count_nonzero(~same) <= 1e-4 * same.size
    assert rel_l2(got_t[same], want_t[same]) <= 1e-5
    assert rel_l2(got_f[same], want_f[same]) <= 1e-5
    plan.close()
