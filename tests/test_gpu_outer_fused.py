"""The fused filter / bisection passes at the edges of their tiles and ranges (GPU).

Same bars as the OC parity tests: fields to 1e-12 and equal bisection counts (cone), 2e-12 fields and 2e-8 densities
(Gaussian, whose last of 45 branches may differ).
"""
import numpy as np
import pytest
import torch
from scipy.ndimage import gaussian_filter

from oracle import design
from pgj import _lib
from pgj.outer import GaussianOuter, PaperOuter

pytestmark = pytest.mark.gpu


# tiles are 16 x 8 x 8: smaller, exact, one over; reach 0, 1, 2, 3 and 4 (one launch per operation)
@pytest.mark.parametrize('n, rmin', [(2, 1.0), (5, 1.5), (7, 4.0), (16, 1.0), (16, 2.0), (17, 3.2), (20, 4.0), (9, 4.5),
                                     (33, 3.0)])
def test_cone_passes_match_oracle(n, rmin):
    print(f'fused cone n={n} rmin={rmin}', flush=True)
    rng = np.random.default_rng(n)
    x = rng.uniform(.15, .7, (n, n, n))
    e = -rng.uniform(.1, 1, (n, n, n))
    gpu = PaperOuter(n, .3, rmin=rmin, emin=1e-6, move=.2).capture()
    assert gpu.fused == (rmin <= 4.0)
    ref = design.PaperOC(n, .3, rmin=rmin, emin=1e-6, move=.2)
    for _ in range(2):
        gpu.set_initial(x)
        gpu.evaluate()
        ph, dp, a = ref.physical(x)
        for name, val in (('ph', ph), ('dp', dp), ('a', a)):
            assert np.abs(getattr(gpu, name).cpu().numpy() - val).max() < 1e-12, name
        count = gpu.step(torch.tensor(e, device='cuda'))
        new, rcount, g, dv = ref.update(x, ph, dp, e)
        assert count == rcount
        assert np.abs(gpu.g.cpu().numpy() - g).max() < 1e-12 * np.abs(g).max()
        assert np.abs(gpu.dv.cpu().numpy() - dv).max() < 1e-12 * np.abs(dv).max()
        assert np.abs(gpu.new.cpu().numpy() - new).max() < 1e-12


@pytest.mark.parametrize('n, beta', [(2, 1.), (15, 4.), (17, 2.), (40, 4.)])
def test_gaussian_loop_matches_oracle(n, beta):
    print(f'fused gaussian n={n}', flush=True)
    rng = np.random.default_rng(n)
    x = rng.uniform(.01, .99, (n, n, n))
    e = rng.uniform(.01, 2, (n, n, n))
    gpu = GaussianOuter(n)
    assert gpu.fused
    ref = design.GaussianOC(n)
    gpu.set_initial(x)
    gpu.evaluate(beta)
    ph, dp, a = ref.physical(x, beta)
    for name, val in (('ph', ph), ('dp', dp), ('a', a)):
        assert np.abs(getattr(gpu, name).cpu().numpy() - val).max() < 2e-12, name
    gpu.step(torch.tensor(e, device='cuda'))
    new, g, dv = ref.update(x, ph, dp, e, beta)
    assert np.abs(gpu.g.cpu().numpy() - g).max() < 2e-12
    assert np.abs(gpu.new.cpu().numpy() - new).max() < 2e-8


# radius 0; radius n (lines wrap once); radius n + 1 and strips past 64 KiB of LDS: one launch per axis
@pytest.mark.parametrize('n, sigma, radius, fused', [(6, .3, 0, 1), (9, 2.0, 9, 1), (9, 2.5, 10, 0), (33, .9, 4, 1),
                                                     (136, 3.8, 15, 0)])
def test_gaussian_filter_matches_scipy(n, sigma, radius, fused):
    print(f'gaussian filter n={n} radius={radius}', flush=True)
    assert _lib.lib().pgj_gauss_fused(n, radius) == fused
    x = np.random.default_rng(n).random((n, n, n))
    k = np.arange(-radius, radius + 1)
    w = np.exp(-.5 / sigma ** 2 * k ** 2)
    w /= w.sum()
    xd, wd = torch.tensor(x, device='cuda'), torch.tensor(w, device='cuda')
    t1, t2, y = (torch.empty_like(xd) for _ in range(3))
    _lib.call('pgj_gauss_filter', n, _lib.ptr(xd), _lib.ptr(wd), radius, _lib.ptr(t1), _lib.ptr(t2), _lib.ptr(y),
              _lib.stream())
    ref = gaussian_filter(x, sigma, mode='wrap', radius=radius)
    assert np.abs(y.cpu().numpy() - ref).max() < 1e-13
    # the output may be the first scratch field
    _lib.call('pgj_gauss_filter', n, _lib.ptr(xd), _lib.ptr(wd), radius, _lib.ptr(t1), _lib.ptr(t2), _lib.ptr(t1),
              _lib.stream())
    assert torch.equal(t1, y)
