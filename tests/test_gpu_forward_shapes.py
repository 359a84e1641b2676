"""Untilted forward kernels by the volume's depth: one, two, four and eight
chunks of 64 layers per column and step, partial last chunks, depths beyond
eight chunks, a detector that cuts the volume and one whose rows are split.
The images are exact fixed-point sums, so an explicit split into row chunks or
sub-bands (which takes the tested paths) gives the same bits; a few views are
compared with the FP64 oracle (raw splat, 1e-5 relative L2; pixels that a voxel
within rounding of the acceptance window can touch, the two outermost rows and
columns, are left out)."""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_parity import Setup, XTT_BASIS13, columns

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,U,V,K", [(1, 8, 8, 0), (40, 60, 60, 0), (64, 96, 90, 0), (65, 98, 98, 0), (130, 200, 120, 0),
                                     (200, 290, 300, 0), (257, 300, 380, 0), (577, 160, 840, 0), (33, 50, 50, 3),
                                     (96, 140, 150, 5), (130, 190, 200, 13), (70, 100, 60, 16)])
def test_forward_depths(orc, xr, ctx, torch_dev, N, U, V, K):
    import torch

    rng = np.random.default_rng(N)
    basis = None
    if K:
        basis = np.concatenate([XTT_BASIS13, rng.normal(size=(3, 3))])[:K]
        basis /= np.linalg.norm(basis, axis=1, keepdims=True)
    st = Setup(orc, xr, N=N, U=U, V=V, P=7, vs=0.4, basis=basis)
    xtt, ch = K > 0, max(K, 1)
    vol = (rng.random((ch, N, N, N), dtype=np.float32) * 0.02).astype(np.float32)
    plan = ctx.plan(st.geom, st.scan)
    vcol = columns(ctx, vol, N, ch, torch_dev)
    views = [0, 2, 5]
    out = []
    for rows, scan, split in ((0, 0, 0), (0, 1, 1), (0, 0, 4), (V // 2 + 1, 0, 2)):
        plan.set_tiles(fwd_rows=rows, fwd_scan=scan, fwd_split=split)
        p = torch.zeros(st.P * V * U, device=torch_dev)
        plan.project(vcol, p, views, out_mode=xr.OUT_RAW, xtt=xtt)
        out.append(p)
    for p in out[1:]:
        assert torch.equal(p, out[0])
    got = out[0].cpu().numpy().reshape(st.P, V, U)
    if N <= 260:
        src = vol if xtt else vol[0]
        want, _ = st.case.forward_view(src, 2, xtt=xtt, normalise=False)
        inner = (slice(2, -2), slice(2, -2))
        assert rel_l2(got[2][inner], want[inner]) <= 1e-5
    plan.close()
