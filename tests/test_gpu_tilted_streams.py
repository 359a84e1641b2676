"""Tilted forward projections whose volume copies belong to the plan, on several
streams in turn: each launch overwrites the copies, so it has to come after the
last one that reads them, whatever stream that ran on.  Also the launches that
make no copy: the entry that allocates nothing, and an allocation that fails.
All give the images of one stream (exact fixed-point sums)."""
import ctypes

import numpy as np
import pytest

from test_gpu_parity import rot_x

pytestmark = pytest.mark.gpu

N, U, P = 128, 192, 24


@pytest.fixture()
def case(xr, torch_dev):
    import torch

    c = xr.Context(0)
    geom = xr.make_geometry(600.0, 300.0, 0.8, N, U, P, vox_size=0.4)
    plan = c.plan(geom, xr.Scan(cond_R=rot_x(70.0).reshape(-1)))
    g = torch.Generator(device=torch_dev).manual_seed(2)
    vols = [torch.rand(N ** 3, device=torch_dev, generator=g) for _ in range(6)]
    want = []
    for v in vols:
        p = torch.zeros(P * U * U, device=torch_dev)
        plan.project(v, p, np.arange(P), out_mode=xr.OUT_RAW)
        c.synchronize()
        want.append(p)
    yield c, geom, plan, vols, want
    plan.close()
    c.close()


def test_two_streams_in_turn(xr, torch_dev, case):
    import torch

    c, _, plan, vols, want = case
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [torch.zeros(P * U * U, device=torch_dev) for _ in vols]
    torch.cuda.synchronize()
    for i, v in enumerate(vols):
        # the context's scratch belongs to one call at a time: the next stream waits for this one
        streams[i % 2].wait_stream(streams[1 - i % 2])
        c.set_stream(streams[i % 2].cuda_stream)
        plan.project(v, outs[i], np.arange(P), out_mode=xr.OUT_RAW)
    torch.cuda.synchronize()
    c.set_stream(0)
    for o, w in zip(outs, want):
        assert torch.equal(o, w)


def test_stream_handle_used_again(xr, torch_dev, case):
    """A stream destroyed and another created in its place may have the same handle."""
    import torch

    c, _, plan, vols, want = case
    hip = ctypes.CDLL("libamdhip64.so")
    outs = [torch.zeros(P * U * U, device=torch_dev) for _ in vols]
    torch.cuda.synchronize()
    for v, o in zip(vols, outs):
        s = ctypes.c_void_p()
        assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0  # non-blocking, default priority
        c.set_stream(s.value)
        plan.project(v, o, np.arange(P), out_mode=xr.OUT_RAW)
        assert hip.hipStreamSynchronize(s) == 0
        c.set_stream(0)
        assert hip.hipStreamDestroy(s) == 0
    for o, w in zip(outs, want):
        assert torch.equal(o, w)


def test_without_copies(xr, torch_dev, case):
    import torch

    c, geom, plan, vols, want = case
    fresh = c.plan(geom, xr.Scan(cond_R=rot_x(70.0).reshape(-1)))
    out = torch.zeros(P * U * U, device=torch_dev)
    fresh.project(vols[0], out, [0], out_mode=xr.OUT_RAW)  # one view: the tables, no copy
    xr.test_fail_allocations(0)
    try:
        fresh.project(vols[0], out, np.arange(P), out_mode=xr.OUT_RAW)
    finally:
        xr.test_fail_allocations(-1)
    c.synchronize()
    assert torch.equal(out, want[0])
    out.zero_()
    fresh.project_noalloc(vols[1], out, np.arange(P), out_mode=xr.OUT_RAW)
    c.synchronize()
    assert torch.equal(out, want[1])
    for i in (2, 3):  # with a copy again
        fresh.project(vols[i], out, np.arange(P), out_mode=xr.OUT_RAW)
        c.synchronize()
        assert torch.equal(out, want[i])
    fresh.close()
