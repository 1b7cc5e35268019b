"""Without an offset the visibilities of a profile are real numbers, and the sign of their zero imaginary part is plus:
np.angle is 0 or +pi, on every route that returns visibilities."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip('torch')


@pytest.mark.parametrize('dt', [np.float64, np.float32])
@pytest.mark.parametrize('PA', [0.0, 0.4])
def test_imaginary_part_is_plus_zero(dt, PA):
    import galario_amd.double as gd
    import galario_amd.single as gs
    from galario_amd import torch_api as ta
    N, dxy, n = 256, 1e-7, 3000
    # a disc with a sharp edge: its visibilities change sign several times within the grid
    I = np.full(480, 1e10, dtype=dt)
    rng = np.random.default_rng(3)
    u, v = ((rng.uniform(-0.3, 0.3, n) / dxy).astype(dt) for _ in range(2))
    grid = (1e-10, dxy / 12, N, dxy)
    ds = ta.Dataset(u, v, device='cuda:0', dtype=torch.float64 if dt is np.float64 else torch.float32)
    It = torch.from_numpy(I).cuda()
    for vis in ((gd if dt is np.float64 else gs).sampleProfile(I, *grid, u, v, PA=PA, inc=0.5),
                ds.sample_profile(It, *grid, PA=PA, inc=0.5).cpu().numpy()):
        assert (vis.real < 0).sum() > 100
        assert (vis.imag == 0).all() and not np.signbit(vis.imag).any()
        assert (np.angle(vis[vis.real < 0]) > 0).all()
