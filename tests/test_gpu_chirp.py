"""Transforms of sizes that are no power of two (Bluestein's chirp transform in double, direct sums in single), against
numpy's.

The 2-D transform makes two passes of two M-point transforms each (M the power of two >= 2N - 1).  Each of them
adds a rounding error of at most eps log2 M (norm-wise), the products with the chirp and with its
transform three eps each, so the result is within 2 (2 log2 M + 6) eps of the exact one.  A direct sum's N rounding
errors, of eps / 2 of a partial sum each, add up to about eps sqrt(N) / 3 (norm-wise) on these images of noise: 30 eps
in two passes at the largest size here, within the same bound."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mod(dt):
    import galario_amd.double as d
    import galario_amd.single as s
    return d if dt == np.float64 else s


def _bound(N, dt):
    L = max(7, math.ceil(math.log2(2 * N - 1)))
    return 2 * (2 * L + 6) * float(np.finfo(dt).eps)


# 62, 64: direct sums; 66 and 130: the first sizes of M = 256 and 512; 128 and 2048: powers of two;
# 2046, 2050: both sides of M = 4096; 4094: the largest M in double; 510, 1000, 2050: direct sums of whole and
# part tiles of 4 lines and 512 frequencies, and of stages of 256 terms; 4098: in single only
@pytest.mark.parametrize('N', [62, 64, 66, 126, 128, 130, 510, 1000, 2046, 2048, 2050])
@pytest.mark.parametrize('dt', [np.float64, np.float32])
def test_fft2d_sizes(N, dt):
    img = np.random.default_rng(N).standard_normal((N, N)).astype(dt)
    got = _mod(dt)._fft2d(img)
    ref = np.fft.rfft2(img.astype(np.float64))
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err <= _bound(N, dt), err


@pytest.mark.parametrize('N, dt', [(4094, np.float64), (4098, np.float32)])
def test_fft2d_largest(N, dt):
    img = np.random.default_rng(N).standard_normal((N, N)).astype(dt)
    got = _mod(dt)._fft2d(img)
    ref = np.fft.rfft2(img.astype(np.float64))
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err <= _bound(N, dt), err


def test_sizes_and_types_in_turn():
    """The table kept from one size is not used for another, nor in the other type."""
    for N, dt in ((100, np.float64), (100, np.float32), (98, np.float32), (98, np.float64), (100, np.float64)):
        img = np.random.default_rng(N).standard_normal((N, N)).astype(dt)
        ref = np.fft.rfft2(img.astype(np.float64))
        err = np.linalg.norm(_mod(dt)._fft2d(img) - ref) / np.linalg.norm(ref)
        assert err <= _bound(N, dt), (N, dt, err)


@pytest.mark.parametrize('N, rmax', [(100, 20), (250, 125), (1000, 134)])
def test_profile_support(N, rmax):
    """A swept profile (rows and columns beyond the disc left out) against the oracle's image."""
    import galario_amd.double as gD
    from oracle import galario_oracle as O
    dxy, nr = 1e-7, rmax * 12
    dR, Rmin = dxy / 12, 1e-10
    I = 1e10 * np.exp(-np.linspace(0, 3, nr))
    rng = np.random.default_rng(N)
    u, v = (rng.uniform(-0.3, 0.3, 500) / dxy for _ in range(2))
    got = gD.sampleProfile(I, Rmin, dR, N, dxy, u, v, dRA=3e-7, dDec=-2e-7, PA=0.4, inc=0.5)
    ref = O.sample_profile(I, Rmin, dR, dxy, N, 0.5, 3e-7, -2e-7, 1 / (N * dxy), 0.4, u, v)
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()
