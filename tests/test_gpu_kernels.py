"""AW kernels by FFT convolution with shared spectra, and the persistent
kernel cache (crocodile_amd.kernels), against the oracle's aw_kernel_fn
(scipy.signal.convolve2d, as crocodile/synthesis.py:701-734) and the direct
w-kernel generator."""
import numpy
import pytest
import scipy.signal
import torch
from numpy.testing import assert_allclose

import crocodile_amd.synthesis as G
from crocodile_amd import kernels as K
from oracle import synthesis_ref as R

pytestmark = pytest.mark.gpu


def a_kernels(rng, n, shape):
    return {a: (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) / shape[0]
            for a in range(n)}


@pytest.mark.parametrize('ashape,S,Q', [((16, 16), 16, 32), ((8, 8), 8, 4), ((7, 4), 6, 2),
                                        ((5, 5), 9, 3)])
def test_aw_fft_matches_direct_convolutions(gpu, ashape, S, Q):
    """AWKernels = convolve2d(convolve2d(A1, A2, 'same'), wk, 'same') for
    every sub-kernel, the C5 shape (A 16x16, w-kernels Q=32 S=16) included."""
    print('case aw fft %s S=%d Q=%d' % (ashape, S, Q), flush=True)
    rng = numpy.random.default_rng(S * Q)
    ak = a_kernels(rng, 3, ashape)
    wk = {w: rng.standard_normal((Q, Q, S, S)) + 1j * rng.standard_normal((Q, Q, S, S))
          for w in (-40.0, 0.0, 125.0)}

    def a_fn(theta, a, t, f):
        return ak[a] * (1 + 0.01 * t) * (1 - 0.02 * f)

    def w_fn(theta, w):
        return wk[w]

    aw = K.AWKernels(a_fn, w_fn, method='fft')
    for (a1, a2, w) in [(0, 1, 125.0), (2, 1, -40.0), (0, 1, 0.0)]:
        got = aw(0.05, w, a1, a2, 3.0, 2.0)
        ref = R.aw_kernel_fn(a_fn, w_fn)(0.05, w, a1, a2, 3.0, 2.0)
        assert isinstance(got, numpy.ndarray) and got.shape == ref.shape
        assert_allclose(got, ref, rtol=0, atol=1e-12 * numpy.abs(ref).max())


def test_aw_fft_shares_transforms(gpu):
    """Spectra of A-kernels, antenna pairs and w sub-kernels are made once:
    a repeated (pair, w) costs only its Q^2 inverse transforms."""
    rng = numpy.random.default_rng(1)
    S, Q = 8, 4
    ak = a_kernels(rng, 3, (S, S))
    wk = {w: rng.standard_normal((Q, Q, S, S)) + 0j for w in (10.0, 20.0)}
    aw = K.AWKernels(lambda th, a: ak[a], lambda th, w: wk[w], method='fft')
    aw(0.1, 10.0, 0, 1)
    n1 = aw.transforms
    assert n1 == 4 + 2 * Q * Q          # A A pair (3) + its respread (1) + w spectra + inverse
    aw(0.1, 10.0, 0, 1)
    assert aw.transforms == n1 + Q * Q
    aw(0.1, 20.0, 0, 1)                 # new w: its spectra + inverse; pair reused
    assert aw.transforms == n1 + Q * Q + 2 * Q * Q
    aw(0.1, 20.0, 1, 2)                 # new pair: its spectrum; w reused
    assert aw.transforms == n1 + 3 * Q * Q + 4 + Q * Q


@pytest.mark.parametrize('S', [8, 24])
def test_aw_kernel_fn_methods_agree(gpu, S):
    """aw_kernel_fn's 'auto' (direct at S = 8, FFT at S = 24), 'fft',
    'direct' and 'uncached' forms give the same kernels."""
    rng = numpy.random.default_rng(7)
    ak = a_kernels(rng, 2, (S, S))

    def a_fn(theta, a):
        return ak[a]

    def w_fn(theta, w):
        return G.w_kernel(theta, w, 64, S, 4)

    y = G.aw_kernel_fn(a_fn, w_fn, method='uncached')(0.08, 300.0, 0, 1)
    for m in ('auto', 'fft', 'direct'):
        f = G.aw_kernel_fn(a_fn, w_fn, method=m)
        assert isinstance(f, K.AWKernels)
        x = f(0.08, 300.0, 0, 1)
        assert isinstance(x, numpy.ndarray)
        assert_allclose(x, y, rtol=0, atol=1e-12 * numpy.abs(y).max())


def test_kernel_cache_hits_eviction_and_disk(gpu, tmp_path):
    kw = dict(NpixFF=32, NpixKern=8, Qpx=4)
    c = K.KernelCache(G.w_kernel, **kw)
    k1 = c(0.05, 100.0)
    k2 = c(0.05, 100.0)
    assert c.hits == 1 and c.misses == 1 and c.made == 1 and k1 is k2
    assert_allclose(k1.cpu().numpy(), R.w_kernel(0.05, 100.0, 32, 8, 4), rtol=0,
                    atol=1e-11 * numpy.abs(k1.cpu().numpy()).max())
    one = k1.numel() * k1.element_size()
    small = K.KernelCache(G.w_kernel, max_bytes=2 * one, **kw)
    for w in (0.0, 10.0, 20.0):
        small(0.05, w)
    assert len(small) == 2 and small.bytes == 2 * one
    small(0.05, 0.0)                      # evicted first: made again
    assert small.made == 4
    d = K.KernelCache(G.w_kernel, directory=str(tmp_path), **kw)
    ref = d(0.05, -60.0).clone()
    assert d.made == 1 and (tmp_path / 'wkern' / '0.05' / '-60.0' / 'kern.npy').exists()
    d2 = K.KernelCache(G.w_kernel, directory=str(tmp_path), **kw)
    got = d2(0.05, -60.0)
    assert d2.loads == 1 and d2.made == 0 and torch.equal(got, ref)


def test_generate_w_kernels_and_cached_imaging(gpu, tmp_path):
    """generate_wkernels.py's kernel set written once, then used through a
    KernelCache by w_cache_imaging: the grid equals the one from the
    kernel function itself, and every kernel came from disk."""
    theta, wstep = 0.05, 50.0
    written = K.generate_w_kernels(str(tmp_path), theta, wstep, 6, 32, 8, 4)
    assert len(written) == 13
    assert K.generate_w_kernels(str(tmp_path), theta, wstep, 6, 32, 8, 4) == []
    cache = K.KernelCache(G.w_kernel, directory=str(tmp_path), NpixFF=32, NpixKern=8, Qpx=4)
    rng = numpy.random.default_rng(4)
    N, lam = 256, 256 / theta
    nv = 20000
    uvw = numpy.stack([rng.uniform(-0.4, 0.4, nv) * lam, rng.uniform(-0.4, 0.4, nv) * lam,
                       rng.uniform(-290.0, 290.0, nv)], axis=1)
    vis = rng.standard_normal(nv) + 1j * rng.standard_normal(nv)
    g1 = G.w_cache_imaging(theta, lam, uvw, None, vis, wstep=wstep, kernel_cache=cache)
    g2 = G.w_cache_imaging(theta, lam, uvw, None, vis, wstep=wstep, NpixFF=32, NpixKern=8,
                           Qpx=4)
    assert cache.made == 0 and cache.loads == 13
    assert_allclose(g1, g2, rtol=0, atol=1e-6 * numpy.abs(g2).max())


@pytest.mark.parametrize('S', [8, 16, 32])
def test_aw_fft_speed(gpu, S):
    """Timing of one AW kernel set (A S x S, Q = 32 sub-kernels of S x S):
    shared-spectrum FFT convolutions against the direct sums (reported)."""
    import time
    rng = numpy.random.default_rng(2)
    ak = {a: torch.as_tensor(rng.standard_normal((S, S)) + 0j, device='cuda')
          for a in range(8)}
    wk = torch.as_tensor(rng.standard_normal((32, 32, S, S)) + 0j, device='cuda')
    out = {}
    for name in ('fft', 'uncached'):
        fn = G.aw_kernel_fn(lambda th, a: ak[a], lambda th, w: wk, method=name)
        fn(0.05, 0.0, 0, 1)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for a in range(8):
            fn(0.05, 0.0, a, (a + 1) % 8)
        torch.cuda.synchronize()
        out[name] = (time.perf_counter() - t0) / 8 * 1e3
    print('AW kernel set S=%d (1024 sub-kernels): fft %.3f ms, direct %.3f ms'
          % (S, out['fft'], out['uncached']), flush=True)


@pytest.mark.parametrize('F,Q,supports', [(9, 1, [9]), (17, 3, [1, 2, 16]), (32, 8, [31, 8]),
                                          (33, 5, [13, 32]), (64, 16, [4, 5])])
def test_w_kernel_bank_edges(gpu, F, Q, supports):
    """Far fields and kernels off the sizes of the kernel generator's row
    groups (8 and 32 rows) and column blocks (64), planes of different
    supports in one launch.  Bound: F^2 unit terms summed in two passes of F,
    each term a few roundings: (2 F + 16) eps F^2."""
    ws = [3.5 * (k - 1) for k in range(len(supports))]
    for invert in (True, False):
        bank = G.w_kernel_bank(0.3, ws, F, supports, Q, invert, double=True)
        got = bank.kern.cpu().numpy()
        for k, S in enumerate(supports):
            ref = R.w_kernel(0.3, ws[k], F, S, Q, invert=invert)
            o = int(bank.plane_off_h[k])
            err = numpy.abs(got[o:o + ref.size].reshape(ref.shape) - ref).max()
            assert err <= (2 * F + 16) * 2.3e-16 * F * F, (F, Q, S, err)
