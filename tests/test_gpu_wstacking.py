"""W-stacking on the device (crocodile_amd.synthesis.w_stacking_imaging and
w_stacking_subgrid_imaging) against the FP64 oracle (oracle/wstacking_ref.py,
wstacking.ipynb cells 10 and 12), which test_oracle_wstacking.py pins.  The
device grids planes in complex64 and transforms them in complex64 FFTs, so
the bound is a few 1e-7 of the image's largest value."""
import numpy
import pytest
import torch

import crocodile_amd.synthesis as G
from oracle import synthesis_ref as R
from oracle import wstacking_ref as WS

pytestmark = pytest.mark.gpu

TOL = 2e-6


def case(seed, N, theta, nv, wmax, wstep, fill=0.35, ties=True):
    rng = numpy.random.default_rng(seed)
    lam = N / theta
    r = fill * lam * numpy.sqrt(rng.uniform(0, 1, nv))
    ph = rng.uniform(0, 2 * numpy.pi, nv)
    w = rng.uniform(-wmax, wmax, nv)
    if ties:
        # exact half-way w values: numpy.around's half-even rule decides the plane
        k = rng.integers(-int(wmax / wstep), int(wmax / wstep), nv // 20)
        w[:nv // 20] = (k + 0.5) * wstep
    uvw = numpy.stack([r * numpy.cos(ph), r * numpy.sin(ph), w], 1)
    vis = rng.standard_normal(nv) + 1j * rng.standard_normal(nv)
    return lam, uvw, vis


def rel(got, ref):
    return numpy.abs(got - ref).max() / numpy.abs(ref).max()


@pytest.mark.parametrize('N,theta,wstep,budget,fused', [
    (256, 0.5, 10.0, 4 << 30, True), (256, 0.5, 10.0, 4 << 30, False),
    (256, 0.5, 10.0, 5 * 256 * 256 * 8, True), (256, 0.5, 10.0, 5 * 256 * 256 * 8, False),
    (255, 0.5, 10.0, 4 << 30, False), (130, 0.25, 7.0, 3 * 130 * 130 * 8, False)])
def test_full_grid_matches_oracle(gpu, monkeypatch, N, theta, wstep, budget, fused):
    """Even N (centring folded into the kernels), odd N (shifted FFTs), and
    stacks split into batches of 5 and 3 planes; the fused transforms and the
    library's."""
    print('case wstack full N=%d budget=%d fused=%s' % (N, budget, fused), flush=True)
    monkeypatch.setattr(G, 'WSTACK_FUSED_CELLS', 0 if fused else 1 << 60)
    lam, uvw, vis = case(N, N, theta, 6000, 0.45 * N / theta * 0.5, wstep)
    ref = WS.w_stacking_imaging(theta, lam, uvw, None, vis, wstep)
    got = G.w_stacking_imaging(theta, lam, uvw, None, vis, wstep, max_stack_bytes=budget)
    assert got.dtype == numpy.complex128 and got.shape == (N, N)
    assert rel(got, ref) < TOL, rel(got, ref)


def test_full_grid_torch_in_torch_out(gpu):
    lam, uvw, vis = case(5, 128, 0.3, 3000, 100.0, 8.0)
    ref = WS.w_stacking_imaging(0.3, lam, uvw, None, vis, 8.0)
    got = G.w_stacking_imaging(0.3, lam, torch.as_tensor(uvw, device='cuda'),
                               None, torch.as_tensor(vis, device='cuda'), 8.0)
    assert isinstance(got, torch.Tensor) and got.is_cuda
    assert rel(got.cpu().numpy(), ref) < TOL


def test_full_grid_recovers_sources(gpu):
    """The physics check of the oracle test on the device result: each point
    source's peak is nv / N^2 sinc(px / N) sinc(py / N) within 6 %."""
    rng = numpy.random.default_rng(3)
    N, theta, nv = 256, 0.5, 4000
    lam = N / theta
    r = 0.35 * lam * numpy.sqrt(rng.uniform(0, 1, nv))
    ph = rng.uniform(0, 2 * numpy.pi, nv)
    uvw = numpy.stack([r * numpy.cos(ph), r * numpy.sin(ph), rng.uniform(-240, 240, nv)], 1)
    pix = [(60, 45), (-70, 30), (50, -65)]
    vis = sum(R.simulate_point(uvw, px * theta / N, py * theta / N) for px, py in pix)
    img = G.w_stacking_imaging(theta, lam, uvw, None, vis, 10.0)
    for px, py in pix:
        want = nv / N ** 2 * numpy.sinc(px / N) * numpy.sinc(py / N)
        assert abs(img[N // 2 + py, N // 2 + px] - want) < 0.06 * want


@pytest.mark.parametrize('N,theta,wstep,npk', [(256, 0.5, 10.0, 8), (256, 0.5, 25.0, 48),
                                                (200, 0.4, 9.0, 11)])
def test_subgrid_matches_oracle(gpu, N, theta, wstep, npk):
    print('case wstack subgrid N=%d wstep=%g npixkern=%d' % (N, wstep, npk), flush=True)
    lam, uvw, vis = case(N + 1, N, theta, 5000, 0.45 * N / theta * 0.5, wstep, fill=0.3)
    ref = WS.w_stacking_subgrid_imaging(theta, lam, uvw, None, vis, wstep, npk)
    got = G.w_stacking_subgrid_imaging(theta, lam, uvw, None, vis, wstep, npk)
    assert got.dtype == numpy.complex128 and got.shape == (N, N)
    assert rel(got, ref) < TOL, rel(got, ref)


def test_subgrid_and_full_grid_images_agree(gpu):
    """Both variants image the same sky, up to the sub-grid's truncation of
    each plane's Fresnel spread (|w| theta^2 / 2 = 25 cells here): 19 % of
    the image norm at npixkern = 16, 3 % at 48."""
    lam, uvw, vis = case(9, 256, 0.5, 5000, 200.0, 10.0, fill=0.25, ties=False)
    full = G.w_stacking_imaging(0.5, lam, uvw, None, vis, 10.0)
    err = {}
    for npk in (16, 48):
        sub = G.ifft(G.w_stacking_subgrid_imaging(0.5, lam, uvw, None, vis, 10.0, npk))
        err[npk] = numpy.linalg.norm(sub - full) / numpy.linalg.norm(full)
    assert err[48] < 0.04 and err[16] > 3 * err[48], err


def test_errors_and_empty(gpu):
    N, theta = 64, 0.5
    lam = N / theta
    uvw = numpy.array([[0.0, 0.0, 0.6 * lam]])
    with pytest.raises(AssertionError):
        G.w_stacking_imaging(theta, lam, uvw, None, numpy.ones(1), 10.0)
    wide = numpy.array([[1.0, 2.0, 0.0]])
    with pytest.raises(AssertionError):
        G.w_stacking_imaging(1.5, 64 / 1.5, wide, None, numpy.ones(1), 10.0)
    edge = numpy.array([[0.49 * lam, 0.0, 30.0], [-0.2 * lam, 0.1 * lam, 30.0]])
    with pytest.raises(ValueError):
        G.w_stacking_subgrid_imaging(theta, lam, edge, None, numpy.ones(2), 10.0, 16)
    with pytest.raises(ValueError):
        G.w_stacking_imaging(theta, lam, uvw[:, :2], None, numpy.ones(1), 10.0)
    empty = numpy.zeros((0, 3))
    assert not G.w_stacking_imaging(theta, lam, empty, None, numpy.zeros(0), 10.0).any()
    assert not G.w_stacking_subgrid_imaging(theta, lam, empty, None, numpy.zeros(0), 10.0,
                                            8).any()


@pytest.mark.parametrize('ntab,nv,stride', [(1, 70_001, 3), (65, 70_001, 3), (4096, 5000, 4),
                                            (4097, 5000, 3), (7, 1, 3)])
def test_plane_sums(gpu, ntab, nv, stride):
    """Counts and sums of w per plane, on both sides of the LDS table's size.
    The sums' bound: nv roundings of at most eps/2 of the sum of |w|."""
    from crocodile_amd import _lib
    rng = numpy.random.default_rng(ntab)
    wstep, plane0 = 2.5, -(ntab // 2)
    uvw = numpy.zeros((nv, stride))
    uvw[:, 2] = rng.uniform(plane0 - 0.49, plane0 + ntab - 0.51, nv) * wstep
    uvw[0, 2] = (plane0 + 0.5) * wstep if ntab > 1 else 0.0   # a half-even tie
    t = numpy.round(uvw[:, 2] / wstep).astype(int) - plane0
    d = torch.as_tensor(uvw, device='cuda')
    count = torch.full((ntab,), -1, dtype=torch.int64, device='cuda')
    total = torch.full((ntab,), 7.0, dtype=torch.float64, device='cuda')
    L = _lib.load()

    def call(n):
        return L.croc_wplane_sums(_lib.ctx(), _lib.ptr(d), nv, stride, wstep, plane0, n,
                                  _lib.ptr(count), _lib.ptr(total))

    _lib.check(call(ntab))
    assert (count.cpu().numpy() == numpy.bincount(t, minlength=ntab)).all()
    ref = numpy.bincount(t, weights=uvw[:, 2], minlength=ntab)
    bound = nv * 2.0 ** -53 * numpy.abs(uvw[:, 2]).sum() + 1e-300
    assert numpy.abs(total.cpu().numpy() - ref).max() <= bound
    if ntab > 1 and t.max() == ntab - 1:
        with pytest.raises(ValueError):
            _lib.check(call(ntab - 1))


@pytest.mark.parametrize('N,P', [(256, 1), (256, 7), (512, 3), (1024, 2), (2048, 1)])
def test_power_of_two_transforms(gpu, N, P):
    """croc_wstack_image against FP64 FFTs of the same stack, every last-pass
    radix, added to a non-zero image.  Bound, RMS over RMS: the 2 log2(N) levels
    of butterflies and the phase add independent errors of at most 1.5 roundings
    of 2^-24 each."""
    from crocodile_amd import _lib
    g = torch.Generator(device='cuda').manual_seed(N + P)
    theta = 0.3
    st = torch.randn((P, N, N), generator=g, device='cuda', dtype=torch.complex64)
    midw = torch.linspace(-300.0, 410.0, P, device='cuda', dtype=torch.float64)
    x = (torch.arange(N, device='cuda', dtype=torch.float64) - N // 2) / N * theta
    n1 = 1 - torch.sqrt(1 - x[None, :] ** 2 - x[:, None] ** 2)
    i = torch.arange(N, device='cuda')
    sign = (1 - 2 * ((i[:, None] + i[None, :]) % 2)).to(torch.float64)
    base = torch.randn((N, N), generator=g, device='cuda', dtype=torch.complex128)
    ref = base.clone()
    for p in range(P):
        ph = -2 * numpy.pi * midw[p] * n1
        ref += (torch.fft.ifftn(st[p].to(torch.complex128), norm='forward') * sign
                * torch.polar(torch.ones_like(ph), ph))
    img = base.clone()
    _lib.check(_lib.load().croc_wstack_image(_lib.ctx(), _lib.ptr(img), _lib.ptr(st.clone()), P, N,
                                             theta, _lib.ptr(midw)))
    err = (img - ref).abs().pow(2).mean().sqrt()
    assert float(err / (ref - base).abs().pow(2).mean().sqrt()) < (
        1.5 * 2.0 ** -24 * numpy.sqrt(2 * numpy.log2(N) + 1))


@pytest.mark.parametrize('N,P', [(256, 5), (512, 3), (1024, 2), (2048, 3)])
def test_power_of_two_phases(gpu, N, P):
    """The Fresnel weights of croc_wstack_image are those of croc_wstack_add: a
    plane holding one cell, the first, transforms to a constant exactly, so the
    images differ by FP64 roundings of the products and sums alone (at most
    eight per plane)."""
    from crocodile_amd import _lib
    rng = numpy.random.default_rng(N)
    v = torch.as_tensor(rng.standard_normal(P) + 1j * rng.standard_normal(P),
                        device='cuda').to(torch.complex64)
    midw = torch.as_tensor(rng.uniform(-900, 900, P), device='cuda')
    cells = torch.zeros((P, N, N), dtype=torch.complex64, device='cuda')
    cells[:, 0, 0] = v
    flat = v[:, None, None].expand(P, N, N).contiguous()
    a, b = (torch.zeros((N, N), dtype=torch.complex128, device='cuda') for _ in range(2))
    L = _lib.load()
    _lib.check(L.croc_wstack_image(_lib.ctx(), _lib.ptr(a), _lib.ptr(cells), P, N, 0.4,
                                   _lib.ptr(midw)))
    _lib.check(L.croc_wstack_add(_lib.ctx(), _lib.ptr(b), _lib.ptr(flat), P, N, 0.4,
                                 _lib.ptr(midw), 1))
    bound = 8 * (P + 1) * 2.0 ** -53 * float(v.abs().sum())
    assert float((a - b).abs().max()) <= bound
