"""Forms that only the largest and the smallest sizes take.

Column passes with both parts of an exchange in LDS at once (139 KB at nxy = 8192 in double and 16384 in single): a
profile beyond 255 pixels and an extent of few column pairs.  Tiled direct sums whose twiddle table exceeds 48 KB, and
tiles that a small image does not fill."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip('torch')


# extent of 409 cells: 208 workgroups, 216 in the adjoint pass, of the 256 that are resident at once
@pytest.mark.parametrize('N, dtype', [(8192, torch.float64), (16384, torch.float32)])
def test_extent_cut_of_the_largest_grids(N, dtype):
    from galario_amd import torch_api as ta
    dxy, Rmin, nr, rmax, n = 1e-7, 1e-10, 900, 400, 3000
    dR = (rmax - 0.5) * dxy / nr
    rng = np.random.default_rng(N)
    b = np.exp(rng.uniform(0.0, math.log(409.0), n)) / (N * dxy)
    th = rng.uniform(0, 2 * np.pi, n)
    ds = ta.Dataset(b * np.cos(th), b * np.sin(th), rng.standard_normal(n), rng.standard_normal(n),
                    rng.uniform(0.5, 2.0, n), device='cuda:0', dtype=dtype)
    I = torch.tensor(1e10 * np.exp(-np.linspace(0, 3, nr)), dtype=dtype, device='cuda:0')
    args, obs = (I, Rmin, dR, N, dxy, ds.u, ds.v), (ds.re, ds.im, ds.w)
    kw = dict(inc=0.6, PA=1.1, dRA=1.5e-7, dDec=-1e-7, check_central_pixel=False)
    assert ta.chi2_profile(*args, *obs, uvmax=ds.uvmax, **kw).item() == ta.chi2_profile(*args, *obs, **kw).item()
    assert torch.equal(ta.sample_profile(*args, uvmax=ds.uvmax, **kw), ta.sample_profile(*args, **kw))
    cut, full = (ta.chi2_profile_grad(*args, *obs, uvmax=x, **kw) for x in (ds.uvmax, 0.0))
    tol = 1e-12 if dtype == torch.float64 else 1e-5
    for a, c in zip(cut, full):
        assert (torch.linalg.norm(a - c) <= tol * torch.linalg.norm(c)).item()


def fft2d_error(N, dt):
    """Norm-wise error of _fft2d on noise, in units of eps."""
    import galario_amd.double as d
    import galario_amd.single as s
    img = np.random.default_rng(N).standard_normal((N, N)).astype(dt)
    got = (d if dt == np.float64 else s)._fft2d(img)
    ref = np.fft.rfft2(img.astype(np.float64))
    return np.linalg.norm(got - ref) / np.linalg.norm(ref) / float(np.finfo(dt).eps)


# Two passes of a sum of N terms, each with one rounding, of half an eps of the partial sum at most, and a twiddle
# rounded to half an eps.  On noise a partial sum of k terms is sqrt(k / N) of the result, so the roundings of
# a pass add to sqrt(N) / 2 / sqrt(2) eps (norm-wise), less than half of that since a rounding is half its bound and less
# on average: sqrt(N) / 2 eps for both passes and the twiddles, and 4 eps for the smallest sizes and the reference.
@pytest.mark.parametrize('N, dt', [(6146, np.float32), (8190, np.float32), (4090, np.float64)] +
                         [(N, dt) for N in (2, 4, 6, 8, 30, 62) for dt in (np.float64, np.float32)])
def test_tiled_sums(N, dt):
    assert fft2d_error(N, dt) <= 0.5 * math.sqrt(N) + 4
