"""w at exact half steps: the plane is that of numpy.around(w / wstep), the
same in every part of a call.  A product with the rounded reciprocal of wstep
(what torch makes of tensor / number on the device) differs at the steps taken
here."""
import numpy
import pytest
import torch

import crocodile_amd.synthesis as G
from crocodile_amd import _lib
from crocodile_amd.autograd import WProjectionOperator
from oracle import awtowers_ref as AWT
from oracle import synthesis_ref as R
from oracle import wstacking_ref as WS
from test_gpu_core import assert_close
from test_oracle_awtowers import scenario

pytestmark = pytest.mark.gpu


def ties(wstep, wmax):
    """The half steps up to wmax that the reciprocal puts on another plane."""
    k = numpy.arange(-int(wmax / wstep) - 1, int(wmax / wstep) + 1)
    w = (k + 0.5) * wstep
    w = w[numpy.abs(w) <= wmax]
    return w[numpy.around(w / wstep) != numpy.around(w * (1.0 / wstep))]


def case(seed, wstep, wmax, nv=3000, spread=None):
    """Visibilities with the ties up to wmax, the rest of w in +-spread."""
    rng = numpy.random.default_rng(seed)
    w = rng.uniform(-1, 1, nv) * (wmax if spread is None else spread)
    t = ties(wstep, wmax)
    assert len(t) > 1
    w[:nv // 5] = rng.choice(t, nv // 5)
    r, ph = 150.0 * numpy.sqrt(rng.uniform(0, 1, nv)), rng.uniform(0, 2 * numpy.pi, nv)
    uvw = numpy.stack([r * numpy.cos(ph), r * numpy.sin(ph), w], 1)
    return uvw, rng.standard_normal(nv) + 1j * rng.standard_normal(nv)


@pytest.mark.parametrize('stride', [3, 5])
@pytest.mark.parametrize('wstep', [49.0, 75.0, 99.0, 0.1, 9.8, -49.0])
def test_bins(gpu, wstep, stride):
    uvw = numpy.zeros((100_003, stride))
    uvw[:, 2] = (numpy.arange(len(uvw)) - 50_000 + 0.5) * abs(wstep)
    uvw[::7, 2] += 0.3 * abs(wstep)
    got = G._w_bins(torch.as_tensor(uvw, device=gpu), wstep)
    assert got.dtype == torch.int64
    numpy.testing.assert_array_equal(got.cpu().numpy(), numpy.around(uvw[:, 2] / wstep))


# ties inside the range of planes, and on its first and last plane
@pytest.mark.parametrize('wstep,wmax,spread', [(49.0, 200.0, None), (4.9, 120.0, None),
                                               (49.0, 100.0, 70.0)])
def test_w_stacking(gpu, wstep, wmax, spread):
    """Both forms against the oracle, within the complex64 bound of their own
    tests (2e-6 of the largest value)."""
    print('case w-stacking ties wstep=%g' % wstep, flush=True)
    N, theta, npk = 256, 0.5, 8
    uvw, vis = case(7, wstep, wmax, spread=spread)
    ref = WS.w_stacking_subgrid_imaging(theta, N / theta, uvw, None, vis, wstep, npk)
    got = G.w_stacking_subgrid_imaging(theta, N / theta, uvw, None, vis, wstep, npk)
    assert numpy.abs(got - ref).max() < 2e-6 * numpy.abs(ref).max()
    ref = WS.w_stacking_imaging(theta, N / theta, uvw, None, vis, wstep)
    got = G.w_stacking_imaging(theta, N / theta, uvw, None, vis, wstep)
    assert numpy.abs(got - ref).max() < 2e-6 * numpy.abs(ref).max()


def test_negative_step(gpu):
    """w-planes counted downwards: the sub-grid w-stacking form and AW-towers
    take a negative wstep, as their notebooks' arithmetic does."""
    print('case negative wstep', flush=True)
    N, theta, npk = 256, 0.5, 8
    uvw, vis = case(9, 49.0, 200.0)
    ref = WS.w_stacking_subgrid_imaging(theta, N / theta, uvw, None, vis, -25.0, npk)
    got = G.w_stacking_subgrid_imaging(theta, N / theta, uvw, None, vis, -25.0, npk)
    assert numpy.abs(got - ref).max() < 2e-6 * numpy.abs(ref).max()
    sc = scenario(seed=3)
    wk = R.w_kernel_function(sc['l'], sc['m'], -2.0)
    args = (sc['theta'], sc['lam'], sc['uvw'], sc['src'], sc['vis'], -2.0, sc['S'],
            sc['margin'], sc['aa_gcf'], sc['aa_sub'], sc['aa_sub2'], sc['aimage'], wk)
    ref = AWT.aw_towers_imaging(*args)
    got = G.aw_towers_imaging(*args)
    assert numpy.abs(got - ref).max() < 2e-6 * numpy.abs(ref).max()


def test_w_cache_and_operator(gpu):
    """Ties on the first and last plane of a kernel bank."""
    print('case w_cache ties', flush=True)
    theta, lam, wstep = 0.1, 1000.0, 49.0
    uvw, vis = case(8, wstep, 100.0, nv=600, spread=70.0)
    kw = dict(NpixFF=16, NpixKern=8, Qpx=2)
    ref = R.w_cache_imaging(theta, lam, uvw, None, vis, wstep=wstep, **kw)
    assert_close(G.w_cache_imaging(theta, lam, uvw, None, vis, wstep=wstep, **kw), ref,
                 what='w_cache_imaging')
    op = WProjectionOperator(theta, lam, uvw, wstep, 16, 8, 2)
    assert op.wbin0 == numpy.around(uvw[:, 2] / wstep).min()
    img = torch.ones((100, 100), device=gpu)
    guv = G.fft(img.to(torch.complex64)).cpu().numpy().astype(complex)
    want = R.w_cache_predict(theta, lam, uvw, None, guv, wstep=wstep, invert=False, **kw) / 16 ** 2
    assert_close(op.apply(img).cpu().numpy(), want, what='operator')
