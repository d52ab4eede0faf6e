"""AW-towers imaging on the device (crocodile_amd.synthesis.aw_towers_imaging)
against the FP64 oracle (oracle/awtowers_ref.py, awtowers.ipynb cells 17,
19, 22), which test_oracle_awtowers.py pins against the A-corrected direct
Fourier image.  The device pre-grids in complex64 with FP32 atomics and
transforms in complex64 FFTs: the bound is 2e-6 of the grid's largest
value."""
import numpy
import pytest
import torch

import crocodile_amd.synthesis as G
from oracle import awtowers_ref as AWT
from oracle import synthesis_ref as R
from test_oracle_awtowers import compare, scenario

pytestmark = pytest.mark.gpu

TOL = 2e-6


def both(sc, wstep, dl=0.0, dm=0.0, **kw):
    wk = R.w_kernel_function(sc['l'], sc['m'], wstep)
    args = (sc['theta'], sc['lam'], sc['uvw'], sc['src'], sc['vis'], wstep, sc['S'],
            sc['margin'], sc['aa_gcf'], sc['aa_sub'], sc['aa_sub2'], sc['aimage'], wk)
    ref = AWT.aw_towers_imaging(*args, dl=dl, dm=dm)
    got = G.aw_towers_imaging(*args, dl=dl, dm=dm, **kw)
    return got, ref


def rel(got, ref):
    return numpy.abs(got - ref).max() / numpy.abs(ref).max()


@pytest.mark.parametrize('S,margin,wstep,budget', [(64, 16, 2.0, 4 << 30),
                                                    (64, 15, 5.0, 4 << 30),
                                                    (64, 16, 2.0, 37 * 128 * 128 * 8),
                                                    (32, 6, 3.0, 4 << 30)])
def test_matches_oracle(gpu, S, margin, wstep, budget):
    """Even and odd chunk widths; groups split into batches of 37 (batches
    that cut through chunks)."""
    print('case awtowers S=%d margin=%d wstep=%g budget=%d' % (S, margin, wstep, budget),
          flush=True)
    sc = scenario(S=S, margin=margin)
    got, ref = both(sc, wstep, max_stack_bytes=budget)
    assert got.shape == ref.shape and got.dtype == numpy.complex128
    assert rel(got, ref) < TOL, rel(got, ref)


def test_shifted_field_matches_oracle(gpu):
    print('case awtowers dl dm', flush=True)
    sc = scenario(seed=2)
    got, ref = both(sc, 2.0, dl=0.02, dm=-0.015)
    assert rel(got, ref) < TOL, rel(got, ref)


def test_physics_on_device(gpu):
    """The device grid's image against the A-corrected DFT image: scale 4
    and residual < 1 %."""
    sc = scenario(seed=4, nant=8, ndump=30)
    wk = R.w_kernel_function(sc['l'], sc['m'], 2.0)
    g = G.aw_towers_imaging(sc['theta'], sc['lam'], sc['uvw'], sc['src'], sc['vis'], 2.0,
                            sc['S'], sc['margin'], sc['aa_gcf'], sc['aa_sub'], sc['aa_sub2'],
                            sc['aimage'], wk)
    c, res = compare(sc, R.ifft(g) / numpy.outer(sc['aa'], sc['aa']))
    assert abs(c - 4) < 0.01 and res < 0.01, (c, res)


def test_torch_in_torch_out(gpu):
    sc = scenario(seed=1)
    wk = R.w_kernel_function(sc['l'], sc['m'], 2.0)
    ref = AWT.aw_towers_imaging(sc['theta'], sc['lam'], sc['uvw'], sc['src'], sc['vis'], 2.0,
                                sc['S'], sc['margin'], sc['aa_gcf'], sc['aa_sub'],
                                sc['aa_sub2'], sc['aimage'], wk)
    d = lambda a: torch.as_tensor(a, device='cuda')  # noqa: E731
    got = G.aw_towers_imaging(sc['theta'], sc['lam'], d(sc['uvw']), d(sc['src']), d(sc['vis']),
                              2.0, sc['S'], sc['margin'], d(sc['aa_gcf']), sc['aa_sub'],
                              sc['aa_sub2'], d(sc['aimage']), d(wk))
    assert isinstance(got, torch.Tensor) and got.is_cuda
    assert rel(got.cpu().numpy(), ref) < TOL


def test_errors(gpu):
    sc = scenario()
    wk = R.w_kernel_function(sc['l'], sc['m'], 2.0)
    args = [sc['theta'], sc['lam'], sc['uvw'], sc['src'], sc['vis'], 2.0, sc['S'],
            sc['margin'], sc['aa_gcf'], sc['aa_sub'], sc['aa_sub2'], sc['aimage'], wk]
    bad = list(args)
    bad[3] = sc['src'] + 10
    with pytest.raises(IndexError):
        G.aw_towers_imaging(*bad)
    bad = list(args)
    bad[6] = 63          # odd sub-grid
    with pytest.raises(ValueError):
        G.aw_towers_imaging(*bad)
    empty = G.aw_towers_imaging(sc['theta'], sc['lam'], numpy.zeros((0, 3)),
                                numpy.zeros((0, 2), dtype=int), numpy.zeros(0), *args[5:])
    assert empty.shape == (sc['N'], sc['N']) and not empty.any()


@pytest.mark.parametrize('form', ['column', 'flat', 'empty'])
def test_src_without_pairs(gpu, form):
    """One antenna index per visibility, or none, is refused before the
    device reads pairs."""
    sc = scenario()
    nv = len(sc['uvw'])
    src = {'column': numpy.zeros((nv, 1), int), 'flat': numpy.zeros(nv, int),
           'empty': numpy.zeros((nv, 0), int)}[form]
    wk = R.w_kernel_function(sc['l'], sc['m'], 2.0)
    with pytest.raises((IndexError, RuntimeError)):
        G.aw_towers_imaging(sc['theta'], sc['lam'], sc['uvw'], src, sc['vis'], 2.0, sc['S'],
                            sc['margin'], sc['aa_gcf'], sc['aa_sub'], sc['aa_sub2'],
                            sc['aimage'], wk)


@pytest.mark.parametrize('direct', [True, False])
@pytest.mark.parametrize('S,margin,K,budget', [(32, 6, 6, 4 << 30),    # one pixel tile
                                               (34, 8, 5, 4 << 30),    # ragged tiles, odd support
                                               (64, 16, 7, 1),         # one segment per chunk
                                               (96, 30, 8, 4 << 30)])
def test_direct_and_transformed_groups(gpu, monkeypatch, direct, S, margin, K, budget):
    """Group images summed directly (croc_awt_direct) and through pre-grids:
    both against the oracle, for supports and sub-grids off the tile size and
    chunks of one and of several segments."""
    monkeypatch.setattr(G, 'AWT_DIRECT_CELLS', 0 if direct else 1 << 40)
    print('case awtowers direct=%s S=%d K=%d' % (direct, S, K), flush=True)
    sc = scenario(seed=5, S=S, margin=margin)
    wk = R.w_kernel_function(sc['l'], sc['m'], 2.0)
    gcf = R.kernel_oversample(sc['aa'], 64, K)
    args = (sc['theta'], sc['lam'], sc['uvw'], sc['src'], sc['vis'], 2.0, S, margin, gcf,
            sc['aa_sub'], sc['aa_sub2'], sc['aimage'], wk)
    got = G.aw_towers_imaging(*args, max_stack_bytes=budget)
    ref = AWT.aw_towers_imaging(*args)
    assert rel(got, ref) < TOL, rel(got, ref)


@pytest.mark.parametrize('S,margin,run,budget', [(32, 6, 40_000, 4 << 30),  # one tile, many parts
                                                 (34, 8, 1000, 4 << 30),    # ragged tiles
                                                 (64, 16, 40_000, 1)])      # no room for parts
def test_direct_sum_of_a_long_run(gpu, monkeypatch, S, margin, run, budget):
    """One antenna pair's long dense run among groups of a few visibilities,
    summed directly: its equal terms make the worst of a plain FP32 sum (1e-4
    after 4e4), where sums of at most 47 stay within 47 / 2 roundings of 2^-24
    = 1.4e-6, inside the bound of this file."""
    monkeypatch.setattr(G, 'AWT_DIRECT_CELLS', 0)
    print('case awtowers run S=%d n=%d' % (S, run), flush=True)
    sc = scenario(seed=6, S=S, margin=margin)
    uvw = numpy.concatenate([sc['uvw'][:40], numpy.repeat(sc['uvw'][40:41], run, 0),
                             sc['uvw'][40:]])
    src = numpy.concatenate([sc['src'][:40], numpy.repeat(sc['src'][40:41], run, 0),
                             sc['src'][40:]])
    vis = numpy.concatenate([sc['vis'][:40], numpy.full(run, 1.1 + 0.7j), sc['vis'][40:]])
    vis = vis.astype(numpy.complex64)
    wk = R.w_kernel_function(sc['l'], sc['m'], 2.0)
    args = (sc['theta'], sc['lam'], uvw, src, vis, 2.0, S, margin, sc['aa_gcf'], sc['aa_sub'],
            sc['aa_sub2'], sc['aimage'], wk)
    got = G.aw_towers_imaging(*args, max_stack_bytes=budget)
    # the oracle on one visibility standing for the run
    one = numpy.concatenate([vis[:40], [numpy.complex128(vis[40]) * run], vis[40 + run:]])
    keep = numpy.r_[0:41, 40 + run:len(uvw)]
    ref = AWT.aw_towers_imaging(sc['theta'], sc['lam'], uvw[keep], src[keep],
                                one.astype(complex), *args[5:])
    assert rel(got, ref) < TOL, rel(got, ref)


@pytest.mark.parametrize('nv,spread', [(1, 1), (65_536, 65_536), (65_537, 65_537),
                                       (140_000, 131_073), (300_000, 900)])
def test_groups(gpu, nv, spread):
    """croc_awt_groups against NumPy: group and chunk tables that come to the
    host in one piece and in several, with chunks across the cuts."""
    import ctypes
    from crocodile_amd import _lib
    print('case awt groups nv=%d' % nv, flush=True)
    rng = numpy.random.default_rng(nv)
    theta, wstep, chunk, nant = 0.1, 3.0, 20, 700
    which = rng.permutation(numpy.arange(nv) % spread)   # `spread` groups
    chunks = which % 11
    uvw = numpy.stack([(chunks % 4 - 1.3) * chunk / theta, (chunks // 4 + 0.2) * chunk / theta,
                       (which // 11 % 5) * wstep + rng.uniform(-1, 1, nv)], 1)
    src = numpy.stack([which // 55 % nant, which // 55 // nant], 1)
    d = lambda n, t: torch.zeros(n, dtype=t, device=gpu)  # noqa: E731
    order, vstart, gid, gwp, ga1, ga2 = (d(nv + 1, torch.int32) for _ in range(6))
    rel = d((nv, 3), torch.float64)
    vstart_h, cstart = numpy.zeros(nv + 1, numpy.int32), numpy.zeros(nv + 1, numpy.int64)
    cub, cvb = numpy.zeros((2, nv), numpy.int32)
    ng, nc = ctypes.c_int64(), ctypes.c_int64()
    host = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    ud, sd = torch.as_tensor(uvw, device=gpu), torch.as_tensor(src, device=gpu)
    _lib.check(_lib.load().croc_awt_groups(
        _lib.ctx(), _lib.ptr(ud), nv, 3, theta, wstep, chunk, _lib.ptr(sd), nant,
        *(_lib.ptr(t) for t in (order, vstart, gid, rel, gwp, ga1, ga2)), ctypes.byref(ng),
        ctypes.byref(nc), host(vstart_h), host(cstart), host(cub), host(cvb)))
    G_, C = ng.value, nc.value
    ub, vb = (numpy.floor(uvw[:, k] * theta / chunk + 0.5).astype(int) for k in (0, 1))
    wp = numpy.around(uvw[:, 2] / wstep).astype(int)
    perm = numpy.lexsort((src[:, 1], src[:, 0], wp, vb, ub))   # stable
    key = numpy.stack([ub, vb, wp, src[:, 0], src[:, 1]], 1)[perm]
    new = numpy.r_[True, (key[1:] != key[:-1]).any(1)]
    starts = numpy.flatnonzero(new)
    assert G_ == len(starts) == spread
    eq = numpy.testing.assert_array_equal
    eq(order[:nv].cpu().numpy(), perm)
    eq(vstart[:G_ + 1].cpu().numpy(), numpy.r_[starts, nv])
    eq(vstart_h[:G_ + 1], numpy.r_[starts, nv])
    eq(gid[:nv].cpu().numpy(), numpy.cumsum(new) - 1)
    for got, col in ((gwp, 2), (ga1, 3), (ga2, 4)):
        eq(got[:G_].cpu().numpy(), key[starts, col])
    cnew = numpy.r_[True, (key[starts][1:, :2] != key[starts][:-1, :2]).any(1)]
    assert C == cnew.sum()
    eq(cstart[:C + 1], numpy.r_[numpy.flatnonzero(cnew), G_])
    eq(numpy.stack([cub[:C], cvb[:C]], 1), key[starts][cnew, :2])
