"""The FDK row filter's three block widths (128, 256 and 512 columns, chosen by
the row length and the number of rows).  The order of each sum is the same in
all, so one call on all views (wide blocks) must give the bits of calls on a few
views (128 columns; pinned to the oracle elsewhere), in both the linear and the
circular form; one view is also compared with the oracle."""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_parity import Setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("U,V,P,kind", [(500, 121, 280, 0), (512, 121, 280, 2), (225, 121, 280, 1), (680, 91, 210, 1),
                                        (513, 64, 230, 2), (31, 77, 430, 0)])
def test_widths_agree(orc, xr, ctx, torch_dev, U, V, P, kind):
    import torch

    st = Setup(orc, xr, N=8, U=U, V=V, P=P, vs=0.5)
    plan = ctx.plan(st.geom, st.scan, convention=xr.CONV_FDK)
    gen = torch.Generator(device=torch_dev).manual_seed(U)
    sino = torch.rand(P * V * U, device=torch_dev, generator=gen)
    whole = torch.full_like(sino, -1.0)
    parts = torch.full_like(sino, -2.0)
    plan.fdk_filter(sino, whole, np.arange(P, dtype=np.int32), filter=kind)
    for lo in range(0, P, 20):
        plan.fdk_filter(sino, parts, np.arange(lo, min(lo + 20, P), dtype=np.int32), filter=kind)
    torch.cuda.synchronize()
    assert torch.equal(whole, parts)
    want = st.case.fdk_filter_view(sino.reshape(P, V, U)[P - 1].cpu().numpy(), kind=kind)
    got = whole.reshape(P, V, U)[P - 1].cpu().numpy()
    # FP32 rounding of up to 680 terms of one sign pattern: 1e-5, as the other filter tests
    assert rel_l2(got, want.reshape(V, U)) <= 1e-5
    plan.close()
