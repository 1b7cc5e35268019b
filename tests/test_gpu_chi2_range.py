"""chi2 of residuals whose squares leave the range of a double, with weights that bring the terms back into it.

Every step from the profile to chi2 is linear in the profile or in the weights, or a product of two such numbers, so
scaling the profile and the observation by 2^k and the weights by 2^m scales chi2 by 2^(2k + m) exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip('torch')

N, DXY, NR = 256, 1e-7, 480
GRID = (1e-10, DXY / 12, N, DXY)
KW = dict(inc=0.5, PA=0.4, dRA=3e-7, dDec=-2e-7)


def values(k, m, n):
    """chi2 on each route, the profile and observation scaled by 2^k, the weights by 2^m."""
    import galario_amd.double as gd
    from galario_amd import torch_api as ta
    rng = np.random.default_rng(n)
    I = np.ldexp(1e10 * np.exp(-np.linspace(0, 3, NR)), k)
    u, v = (rng.uniform(-0.2, 0.2, n) / DXY for _ in range(2))
    re, im = (np.ldexp(rng.standard_normal(n), k) for _ in range(2))
    w = np.ldexp(rng.uniform(0.5, 2.0, n), m)
    ds = ta.Dataset(u, v, re, im, w, device='cuda:0')
    It = torch.from_numpy(I).cuda()
    vis = gd.sampleProfile(I, *GRID, u, v, **KW)
    out = {'host': gd.chi2Profile(I, *GRID, u, v, re, im, w, **KW),
           'device': ds.chi2_profile(It, *GRID, **KW).item(),
           'reduce': gd.reduce_chi2(re, im, w, vis),
           'gradient': ds.chi2_profile_grad(It, *GRID, **KW)[0].item()}
    for W in (1, 5):
        plan = ta.BatchedChi2Profile([(ds, N, DXY)], NR, GRID[0], GRID[1], W)
        geom = torch.tensor([[KW['inc'], KW['PA'], KW['dRA'], KW['dDec']]] * W, device='cuda:0', dtype=torch.float64)
        out[f'batch of {W}'] = plan(It.repeat(W, 1), geom)[0].item()
    return out


@pytest.mark.parametrize('k, m', [(520, -1000), (-520, 1000)])
@pytest.mark.parametrize('n', [1, 1000])
def test_terms_in_range(n, k, m):
    plain, scaled = values(0, 0, n), values(k, m, n)
    for route, c in plain.items():
        assert scaled[route] == np.ldexp(c, 2 * k + m), route
