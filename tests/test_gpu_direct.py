"""Direct gridding and degridding of small calls (croc_convgrid /
croc_convdegrid below the limits of csrc/direct.hip) against the binned
tile kernels (plans): the same fixed-point sums and the same order of
summation per lane, so equality is bit for bit, and errors leave the outputs
and the next call alone."""
import numpy
import pytest
import torch

import crocodile_amd.synthesis as G
from crocodile_amd import _lib
from test_oracle import random_case

pytestmark = pytest.mark.gpu


def make(gpu, seed, N, S, Q, nv, planes, separable):
    rng = numpy.random.default_rng(seed)
    tables, p, v = random_case(rng, N, S, Q, nv, planes, separable)
    bank = G.KernelBank.from_tables(tables, separable)
    uvw = torch.as_tensor(p, device=gpu).contiguous()
    vis = torch.as_tensor(v, device=gpu).to(torch.complex64)
    vp = torch.as_tensor(rng.integers(0, planes, nv).astype(numpy.int32), device=gpu)
    grid = torch.as_tensor(rng.standard_normal((N, N)) + 1j * rng.standard_normal((N, N)),
                           device=gpu).to(torch.complex64)
    return bank, uvw, vis, vp, grid


@pytest.mark.parametrize('separable', [False, True])
@pytest.mark.parametrize('N,S,Q,nv,planes', [
    (64, 1, 1, 1, 1), (65, 5, 3, 63, 2), (128, 8, 4, 64, 3), (255, 16, 8, 65, 1),
    (512, 16, 2, 12287, 2), (512, 16, 2, 12289, 2),
    (512, 16, 2, 2560, 2), (512, 16, 2, 2561, 2),     # both sides of gridding's limit
    (300, 3, 2, 5120, 2), (300, 3, 2, 5121, 2),
    (300, 33, 2, 900, 2), (400, 64, 1, 300, 1), (300, 64, 1, 16385, 1),
    (300, 64, 1, 8192, 1), (300, 64, 1, 8193, 1),     # and of degridding's
    (300, 64, 8, 16384, 2), (300, 64, 8, 16385, 2)])  # and with a bank of 4 MiB
def test_direct_equals_tiles(gpu, N, S, Q, nv, planes, separable):
    print('direct N=%d S=%d nv=%d sep=%s' % (N, S, nv, separable), flush=True)
    bank, uvw, vis, vp, grid = make(gpu, N + S, N, S, Q, nv, planes, separable)
    mode = _lib.PLANE_INDEX
    plan = G.GridPlan(bank, N, uvw, 1.0, mode, vp)
    a, b = grid.clone(), grid.clone()
    G.grid_device(bank, a, uvw, 1.0, vis, mode, vp)
    plan.grid(b, vis)
    assert torch.equal(a, b)
    x, y = torch.empty_like(vis), torch.empty_like(vis)
    G.degrid_device(bank, grid, uvw, 1.0, x, mode, vp)
    plan.degrid(grid, y)
    assert torch.equal(x, y)


@pytest.mark.parametrize('separable', [False, True])
@pytest.mark.parametrize('S', [1, 2, 3, 4, 7, 8, 15])
def test_direct_concentrated(gpu, S, separable):
    """As many visibilities as the path takes, all within a few cells: many
    atomic sums on each cell, few useful lanes at the small supports."""
    nv = 40960 // max(S, 8)
    print('direct concentrated S=%d nv=%d sep=%s' % (S, nv, separable), flush=True)
    bank, uvw, vis, vp, grid = make(gpu, S, 64, S, 2, nv, 2, separable)
    uvw[:, :2] *= 0.02
    mode = _lib.PLANE_INDEX
    plan = G.GridPlan(bank, 64, uvw, 1.0, mode, vp)
    a, b = grid.clone(), grid.clone()
    G.grid_device(bank, a, uvw, 1.0, vis, mode, vp)
    plan.grid(b, vis)
    assert torch.equal(a, b)
    x, y = torch.empty_like(vis), torch.empty_like(vis)
    G.degrid_device(bank, grid, uvw, 1.0, x, mode, vp)
    plan.degrid(grid, y)
    assert torch.equal(x, y)


def test_direct_errors_leave_outputs_and_next_call(gpu):
    bank, uvw, vis, vp, grid = make(gpu, 7, 128, 8, 4, 700, 2, False)
    mode = _lib.PLANE_INDEX
    ref, out = grid.clone(), torch.empty_like(vis)
    G.grid_device(bank, ref, uvw, 1.0, vis, mode, vp)
    G.degrid_device(bank, grid, uvw, 1.0, out, mode, vp)
    for what, exc in (('domain', AssertionError), ('bounds', ValueError), ('plane', ValueError)):
        u, q = uvw.clone(), vp.clone()
        if what == 'plane':
            q[350] = 2
        else:
            u[350, 0] = 0.7 if what == 'domain' else 0.499
        g, o = grid.clone(), torch.full_like(vis, 3.0)
        with pytest.raises(exc):
            G.grid_device(bank, g, u, 1.0, vis, mode, q)
        with pytest.raises(exc):
            G.degrid_device(bank, grid, u, 1.0, o, mode, q)
        torch.cuda.synchronize()
        assert torch.equal(g, grid) and bool((o == 3.0).all())
        g = grid.clone()
        G.grid_device(bank, g, uvw, 1.0, vis, mode, vp)
        G.degrid_device(bank, grid, uvw, 1.0, o, mode, vp)
        assert torch.equal(g, ref) and torch.equal(o, out)
