"""Principal orientation where its closed form is delicate: double and triple
eigenvalues at either end (the angle's ends), rank one, every basis count, odd
voxel counts, small and large coefficients.  Checked against FP64 eigenvalues of
the same matrix.  Bounds: a double root is known to about 1e-8 of the trace in
FP64, FP32 results are rounded three times (quotient of sums): 4 * 2^-24 + 1e-7
on the normalised eigenvalues; the direction's residual |C e - l0 e|, with three
rounded components, 1e-6 of the trace."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 2, 3, 7, 13, 16])
@pytest.mark.parametrize("scale", [1.0, 1e-9, 1e6])
def test_eigen_pairs(xr, ctx, torch_dev, K, scale):
    import torch

    rng = np.random.default_rng(10 * K)
    basis = rng.normal(size=(K, 3))
    basis[:3] = np.eye(3)[:K]  # axes first: equal coefficients give double and triple roots
    basis = (basis / np.linalg.norm(basis, axis=1, keepdims=True)).astype(np.float32)
    n = 1021
    mu = rng.uniform(0.1, 1.0, (K, n))
    mu[:, :40] = 0.0
    for i in range(40):  # few non-zero coefficients, equal ones among them
        mu[rng.integers(K, size=3), i] = [1.0, 1.0, [1.0, 0.5, 2.0][i % 3]]
    mu[3:, 40:80] *= 1e-7  # nearly diagonal, nearly equal
    mu[:3, 40:80] = np.where(np.arange(40) % 2, 1.0, [[1.0], [1.0], [0.25]][:K])
    mu = (mu * scale).astype(np.float32)
    md = torch.empty(3 * n, device=torch_dev)
    ev = torch.empty(3 * n, device=torch_dev)
    ctx.pca(torch.from_numpy(mu.reshape(-1)).to(torch_dev), basis, n, n, md, ev)
    torch.cuda.synchronize()
    md = md.cpu().numpy().reshape(3, n).astype(np.float64)
    ev = ev.cpu().numpy().reshape(3, n).astype(np.float64)
    w = mu.astype(np.float64)[:, :, None] * basis.astype(np.float64)[:, None, :]
    C = np.einsum("kni,knj->nij", w, w) / K
    tr = np.trace(C, axis1=1, axis2=2)
    want = np.linalg.eigvalsh(C / tr[:, None, None])
    assert np.abs(ev.T - want).max() <= 4 * 2.0**-24 + 1e-7
    mean = mu.astype(np.float64).mean(axis=0)
    e = (md / mean).T
    assert np.abs(np.linalg.norm(e, axis=1) - 1).max() <= 1e-6
    assert (md[2] >= 0).all()
    res = np.einsum("nij,nj->ni", C / tr[:, None, None], e) - want[:, :1] * e
    assert np.abs(res).max() <= 1e-6
