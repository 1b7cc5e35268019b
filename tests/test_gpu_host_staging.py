"""Host-array calls: inputs packed into pinned memory or copied by array, results written to pinned memory or
copied, on both sides of the sizes that decide (2 MiB per array, 8 MiB in all, 512 KiB per packed part)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DXY = 1e-7


def _case(n, dt, seed=0):
    rng = np.random.default_rng(seed)
    I = (1e10 * np.exp(-np.linspace(0, 3, 480))).astype(dt)
    u, v = ((rng.uniform(-0.2, 0.2, n) / DXY).astype(dt) for _ in range(2))
    re, im = (rng.standard_normal(n).astype(dt) for _ in range(2))
    return I, u, v, re, im, rng.uniform(0.5, 2.0, n).astype(dt)


def _mod(dt):
    import galario_amd.double as d
    import galario_amd.single as s
    return d if dt == np.float64 else s


# points per array: 0.5 MiB, 2 MiB, 2 MiB + 1, 3 MiB (by array) of doubles; the five arrays of 2 MiB exceed 8 MiB, so
# the last of them goes by itself
@pytest.mark.parametrize('n', [1, 255, 13000, 65536, 262144, 262145, 393216])
@pytest.mark.parametrize('dt', [np.float64, np.float32])
def test_host_equals_device(n, dt):
    import torch
    from galario_amd import torch_api as ta
    I, u, v, re, im, w = _case(n, dt)
    mod, kw = _mod(dt), dict(dRA=3e-7, dDec=-2e-7, PA=0.4, inc=0.5)
    grid = (1e-10, DXY / 12, 128, DXY)
    dev = [torch.from_numpy(a).cuda() for a in (I, u, v, re, im, w)]
    vis = mod.sampleProfile(I, *grid, u, v, **kw)
    assert np.array_equal(vis, ta.sample_profile(dev[0], *grid, dev[1], dev[2], **kw).cpu().numpy())
    chi2 = mod.chi2Profile(I, *grid, u, v, re, im, w, **kw)
    assert chi2 == dt(ta.chi2_profile(dev[0], *grid, *dev[1:], **kw).item())


def test_error_then_call():
    """A point outside the grid is reported, and the next calls are not."""
    I, u, v, re, im, w = _case(1000, np.float64)
    mod, grid = _mod(np.float64), (1e-10, DXY / 12, 128, DXY)
    good = mod.chi2Profile(I, *grid, u, v, re, im, w)
    far = u.copy()
    far[7] = 0.6 / DXY
    for call in (lambda: mod.chi2Profile(I, *grid, far, v, re, im, w), lambda: mod.sampleProfile(I, *grid, far, v)):
        with pytest.raises(ValueError, match='outside the Fourier grid'):
            call()
        assert mod.chi2Profile(I, *grid, u, v, re, im, w) == good


def test_sizes_in_turn():
    """Pinned and device buffers grow between calls."""
    mod, grid = _mod(np.float64), (1e-10, DXY / 12, 128, DXY)
    ref = {}
    for n in (10, 70000, 300000, 10, 70000, 5000, 300000):
        I, u, v, re, im, w = _case(n, np.float64, seed=n)
        c = mod.chi2Profile(I, *grid, u, v, re, im, w)
        assert ref.setdefault(n, c) == c
