"""Null arrays at the host-array C entry points are refused with an error code, before anything touches a device."""
import ctypes

import numpy as np
import pytest

from galario_amd import _lib

INVALID = 1


def arguments(name, real, null):
    """Arguments of a host-array entry point, the array `null` given as a null pointer."""
    n, N, dxy = 40, 64, 1e-7
    R = ctypes.c_double if real is np.float64 else ctypes.c_float
    arrays = {k: np.ones(n, dtype=real) for k in ('u', 'v', 're', 'im', 'w')}
    arrays.update(I=np.ones(480, dtype=real), image=np.ones((N, N), dtype=real),
                  vis=np.zeros(2 * n, dtype=real), chi2=np.zeros(1, dtype=real))
    p = {k: ctypes.c_void_p(None if k == null else a.ctypes.data) for k, a in arrays.items()}
    if 'profile' in name:
        head = [480, p['I'], R(1e-10), R(dxy / 12), R(dxy), N, R(0.3), R(0), R(0), R(1 / (N * dxy)), R(0), n]
    else:
        head = [N, N, p['image'], R(1), R(0), R(0), R(1 / (N * dxy)), R(0), n]
    tail = [p['u'], p['v']] + ([p['re'], p['im'], p['w']] if 'chi2' in name else [p['vis']])
    if 'profile' in name:
        tail.append(1)
    if 'chi2' in name:
        tail.append(p['chi2'])
    return head + tail, arrays


def used(name):
    first = ['I' if 'profile' in name else 'image', 'u', 'v']
    return first + (['re', 'im', 'w', 'chi2'] if 'chi2' in name else ['vis'])


@pytest.mark.parametrize('name', ['sample_profile', 'chi2_profile', 'sample_image', 'chi2_image'])
@pytest.mark.parametrize('real', [np.float64, np.float32])
def test_null_array_is_refused(name, real):
    f = getattr(_lib.lib, f"galario_{name}_{'f64' if real is np.float64 else 'f32'}")
    for null in used(name):
        args, keep = arguments(name, real, null)
        assert f(*args) == INVALID, null
        message = _lib.lib.galario_last_error().decode()
        assert 'null' in message and 'pointer' in message, (null, message)
