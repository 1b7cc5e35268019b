"""A host-array call with a point outside the grid returns an error, and the visibilities all the same: NaN for that
point, the others' values as in a call without it."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DXY, N, INVALID = 1e-7, 128, 1


# visibilities of 16 bytes: below and above the 2 MiB up to which the kernel writes them to pinned memory
@pytest.mark.parametrize('n', [1000, 131072, 131073, 300000])
@pytest.mark.parametrize('kind', ['profile', 'image'])
def test_visibilities_beside_the_error(kind, n):
    from galario_amd import _lib
    rng = np.random.default_rng(n)
    u, v = (rng.uniform(-0.2, 0.2, n) / DXY for _ in range(2))
    far = u.copy()
    far[7] = 0.6 / DXY
    d, p = ctypes.c_double, lambda a: ctypes.c_void_p(a.ctypes.data)  # noqa: E731
    I, img = 1e10 * np.exp(-np.linspace(0, 3, 480)), rng.standard_normal((N, N))

    def call(u, vis):
        if kind == 'profile':
            return _lib.lib.galario_sample_profile_f64(480, p(I), d(1e-10), d(DXY / 12), d(DXY), N, d(0.5), d(3e-7), d(-2e-7),
                                                       d(1 / (N * DXY)), d(0.4), n, p(u), p(v), p(vis), 1)
        return _lib.lib.galario_sample_image_f64(N, N, p(img), d(1), d(3e-7), d(-2e-7), d(1 / (N * DXY)), d(0.4), n, p(u),
                                                 p(v), p(vis))

    good, got = np.zeros(n, dtype=complex), np.full(n, 5 + 5j)
    assert call(u, good) == 0
    assert call(far, got) == INVALID
    assert np.isnan(got[7])
    assert np.array_equal(np.delete(got, 7), np.delete(good, 7))
