"""Batched problems tilted by more than 45 degrees, whose forward lanes run along
x, y or (without the volume copies of a standalone launch, where strided reads
would not pay) z: each equals its own solve bit for bit, the forward sums being
exact and the backprojection's per voxel in order."""
import numpy as np
import pytest

from test_gpu_parity import XTT_BASIS13, grating, rot_x, rot_y

pytestmark = pytest.mark.gpu


def geometry(xr, N, P):
    return xr.make_geometry(600.0, 300.0, 0.8, N, (3 * N) // 2, P, vox_size=0.5)


@pytest.mark.parametrize("flags", ["eager", "graph"])
def test_plain_batch_equals_standalone(xr, ctx, flags):
    specs = [(40, 24, 1, rot_x(60.0)), (64, 240, 1, rot_y(75.0)), (33, 20, 2, None), (48, 30, 3, rot_x(90.0))]
    geoms = [geometry(xr, N, P) for N, P, _, _ in specs]
    scans = [xr.Scan(cond_R=None if R is None else R.reshape(-1)) for _, _, _, R in specs]
    rng = np.random.default_rng(8)
    sinos = [rng.random(g.n_proj * g.n_det_u * g.n_det_v).astype(np.float32) + 0.5 for g in geoms]
    init = [np.full(g.n_vox ** 3, 0.01, np.float32) for g in geoms]
    want = []
    for g, s, y, (_, _, b, _), v0 in zip(geoms, scans, sinos, specs, init):
        v = [v0.copy()]
        ctx.ir_reconstruct(g, s, [y.copy()], v, 2, b)
        want.append(v[0])
    got = [v.copy() for v in init]
    ctx.batch_reconstruct(geoms, [y.copy() for y in sinos], got, 2, batch=[s[2] for s in specs], scans=scans,
                          flags=xr.BATCH_GRAPH if flags == "graph" else 0)
    for i, (a, b) in enumerate(zip(got, want)):
        assert np.array_equal(a, b), specs[i][:3]


@pytest.mark.parametrize("K", [3, 13])
def test_xtt_batch_equals_standalone(xr, ctx, K):
    specs = [(32, 12, rot_x(65.0)), (21, 10, rot_y(90.0))]
    geoms = [geometry(xr, N, P) for N, P, _ in specs]
    scans = [xr.Scan(cond_R=np.concatenate([np.eye(3).reshape(-1), R.reshape(-1)]), basis=XTT_BASIS13[:K],
                     grating=grating([0, 60])) for _, _, R in specs]
    rng = np.random.default_rng(9)
    sinos = [rng.random((2, g.n_proj * g.n_det_u * g.n_det_v)).astype(np.float32) + 0.5 for g in geoms]
    got = [np.full(K * g.n_vox ** 3, 0.01, np.float32) for g in geoms]
    ctx.batch_reconstruct(geoms, [y.reshape(-1).copy() for y in sinos], got, 2, scans=scans)
    for i, (g, s, y) in enumerate(zip(geoms, scans, sinos)):
        n3 = g.n_vox ** 3
        vol = [np.full(n3, 0.01, np.float32) for _ in range(K)]
        md = [np.zeros(n3, np.float32) for _ in range(3)]
        ctx.xtt_reconstruct(g, s, [c.copy() for c in y], vol, md, 2, 1)
        assert np.array_equal(got[i], np.concatenate(vol)), specs[i][:2]
