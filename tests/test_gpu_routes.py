"""The sample and adjoint kernels' routes, at the sizes that decide between them.

Gradients are held to the bars of test_gpu_grad.py (1e-7 norm-wise for the profile, 1e-8 per geometry entry, against
the torch composition on the CPU); forward results that take the same arithmetic on two routes are equal."""
import math

import numpy as np
import pytest

from oracle import galario_oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip('torch')
import torch_reference as TR  # noqa: E402

DEV = 'cuda:0'
DXY = 0.02 * O.ARCSEC
RMIN = 1e-4 * O.ARCSEC
GEOM = (0.6, 1.1, 0.03 * O.ARCSEC, -0.02 * O.ARCSEC)


def points(n, N, near, far, seed=0):
    """n log-uniform baselines between near and far cells, noise for an observation."""
    rng = np.random.default_rng(seed)
    b = np.exp(rng.uniform(math.log(near), math.log(far), n)) / (N * DXY)
    th = rng.uniform(0, 2 * np.pi, n)
    return b * np.cos(th), b * np.sin(th), rng.standard_normal(n), rng.standard_normal(n), rng.uniform(0.5, 2.0, n)


def profile(nr=200, rmax=40):
    """(values, dR): nr bins out to rmax pixels."""
    return 1e10 * np.exp(-np.linspace(0, 3, nr)), (rmax - 0.5) * DXY / nr


def dataset(p, dtype=torch.float64, sort=True):
    from galario_amd import torch_api as ta
    return ta.Dataset(*p, device=DEV, dtype=dtype, sort=sort)


def kw():
    return dict(inc=GEOM[0], PA=GEOM[1], dRA=GEOM[2], dDec=GEOM[3], check_central_pixel=False)


def reference(I, dR, N, p):
    t = [torch.tensor(np.asarray(x, dtype=np.float64)) for x in (I, GEOM)]
    for x in t:
        x.requires_grad_(True)
    chi2 = TR.chi2_profile(t[0], t[1], RMIN, dR, N, DXY, *(torch.tensor(a) for a in p))
    gI, gg = torch.autograd.grad(chi2, t)
    return chi2.item(), gI.numpy(), gg.numpy()


def check_grad(got, ref):
    c, gI, gg = (x.cpu().numpy() for x in got)
    assert abs(c[0] - ref[0]) <= 1e-11 * ref[0]
    assert np.linalg.norm(gI - ref[1]) <= 1e-7 * np.linalg.norm(ref[1])
    assert (np.abs(gg - ref[2]) <= 1e-8 * np.abs(ref[2])).all(), (gg, ref[2])


def test_gradient_beside_invalid_point():
    """A point outside the grid with an infinite weight makes chi2 NaN, and adds nothing to its neighbours' cells."""
    from galario_amd import torch_api as ta
    N, (I, dR) = 256, profile()
    p = points(600, N, 1.0, 6.0)
    It = torch.tensor(I, device=DEV)
    ref = dataset(p, sort=False).chi2_profile_grad(It, RMIN, dR, N, DXY, **kw())[1]
    q = [np.insert(x, 301, y) for x, y in zip(p, (3.0 / DXY, 0.0, 1.0, 1.0, np.inf))]
    t = [torch.tensor(x, device=DEV) for x in q]
    chi2, gI, _ = ta.chi2_profile_grad(It, RMIN, dR, N, DXY, *t, **kw())
    assert torch.isnan(chi2).all()
    assert (torch.linalg.norm(gI - ref) <= 1e-12 * torch.linalg.norm(ref)).item()
    assert ta.take_oob_flag()


# up to 512 blocks of 256 points the sparse ones go straight to memory, beyond through the line table; in locality
# order the dense ones take the window, in random order no workgroup's cells fit it and the table overflows
@pytest.mark.parametrize('sort', [True, False])
@pytest.mark.parametrize('N, n', [(256, 1), (256, 257), (256, 8193), (1024, 20011), (256, 131072), (256, 131073),
                                  (1024, 131072), (1024, 131073)])
def test_gradient_scatter(N, n, sort):
    I, dR = profile()
    p = points(n, N, 1.0, 0.45 * N)
    ds = dataset(p, sort=sort)
    It = torch.tensor(I, device=DEV)
    got = ds.chi2_profile_grad(It, RMIN, dR, N, DXY, **kw())
    check_grad(got, reference(I, dR, N, p))
    assert got[0].item() == ds.chi2_profile(It, RMIN, dR, N, DXY, **kw()).item()      # (one order of sums)


# straight to memory (up to 512 workgroups), one and two points per thread (up to 8192 and more), each LDS window
@pytest.mark.parametrize('walkers, n', [(2, 20011), (7, 20011), (110, 20011)])
@pytest.mark.parametrize('window', [2048, 3072, 4096])
def test_batched_gradient_scatter(walkers, n, window):
    from galario_amd import torch_api as ta
    N, (I, dR) = 512, profile()
    p = points(n, N, 1.0, 0.45 * N)
    plan = ta.BatchedChi2Profile([(dataset(p), N, DXY)], len(I), RMIN, dR, walkers, check_central_pixel=False)
    plan.set_tile(walkers, 1, window, grad=True)
    plan.set_chunk(walkers, walkers, 1, grad=True)
    It = torch.tensor(np.tile(I, (walkers, 1)), device=DEV)
    geom = torch.tensor(np.tile(GEOM, (walkers, 1)), device=DEV)
    chi2, _, gI, gg = plan.grad(It, geom)
    ref = reference(I, dR, N, p)
    for k in (0, walkers - 1):
        check_grad((chi2[k:k + 1], gI[k], gg[k]), ref)


# all points in the hot tile: its replicas are folded by 64 to 1024 threads
@pytest.mark.parametrize('N', [128, 256, 512, 1024, 2048])
def test_hot_tile(N):
    I, dR = profile(rmax=20)
    p = points(9000, N, 0.5, 14.0)
    ds = dataset(p)
    It = torch.tensor(I, device=DEV)
    ref = reference(I, dR, N, p)
    for _ in range(2):                      # (the second call: the replicas were cleared)
        check_grad(ds.chi2_profile_grad(It, RMIN, dR, N, DXY, **kw()), ref)


def test_hot_tile_largest_single():
    """nxy = 16384: the gradient of the whole is the sum over the parts (which use other replicas)."""
    N, (I, dR) = 16384, profile(rmax=20)
    p = points(9000, N, 0.5, 14.0)
    It = torch.tensor(I, dtype=torch.float32, device=DEV)

    def grad(sl):
        d = dataset(tuple(x[sl] for x in p), torch.float32)
        return d.chi2_profile_grad(It, RMIN, dR, N, DXY, **kw())[1].cpu().numpy()

    whole, parts = grad(slice(None)), grad(slice(0, 1000)) + grad(slice(1000, None))
    assert np.linalg.norm(whole - parts) <= 1e-5 * np.linalg.norm(whole)


# one block of 256 points per workgroup up to 2048 blocks, two beyond
@pytest.mark.parametrize('n', [524288, 524289])
def test_forward_rounds(n):
    from galario_amd import torch_api as ta
    N, (I, dR) = 256, profile()
    ds = dataset(points(n, N, 1.0, 0.45 * N))
    It = torch.tensor(I, device=DEV)
    one = ds.chi2_profile(It, RMIN, dR, N, DXY, **kw()).item()
    plan = ta.BatchedChi2Profile([(ds, N, DXY)], len(I), RMIN, dR, 3, check_central_pixel=False)
    geom = torch.tensor(np.tile(GEOM, (3, 1)), device=DEV)
    for k in (1, 2, 4, 8):
        plan.set_chunk(3, 3, k)
        assert (plan(It.repeat(3, 1), geom) == one).all()


# spectra and adjoints within the extent only, residue and full forms (rmax 200, 400), few and many column pairs
@pytest.mark.parametrize('dtype', [torch.float64, torch.float32])
@pytest.mark.parametrize('rmax', [200, 400])
@pytest.mark.parametrize('reach', [0.01, 0.1, 0.4, 0.93])
def test_extent_cut(reach, rmax, dtype):
    from galario_amd import torch_api as ta
    N, (I, dR) = 1024, profile(nr=900, rmax=rmax)
    ds = dataset(points(3000, N, 1.0, max(2.0, reach * N / 2)), dtype)
    It = torch.tensor(I, dtype=dtype, device=DEV)
    args = (It, RMIN, dR, N, DXY, ds.u, ds.v)
    obs = (ds.re, ds.im, ds.w)
    k = kw()
    assert ta.chi2_profile(*args, *obs, uvmax=ds.uvmax, **k).item() == ta.chi2_profile(*args, *obs, **k).item()
    assert torch.equal(ta.sample_profile(*args, uvmax=ds.uvmax, **k), ta.sample_profile(*args, **k))
    cut, full = (ta.chi2_profile_grad(*args, *obs, uvmax=x, **k) for x in (ds.uvmax, 0.0))
    tol = 1e-12 if dtype == torch.float64 else 1e-5
    for a, b in zip(cut, full):
        assert (torch.linalg.norm(a - b) <= tol * torch.linalg.norm(b)).item()


def test_grids_of_one_plan():
    """Several grids, each with its own number of walkers per chunk (8 at nxy = 4096)."""
    from galario_amd import torch_api as ta
    I, dR = profile()
    grids = [(4096, 5000), (128, 3000), (1024, 700)]
    sets = [(dataset(points(n, N, 1.0, 0.4 * N, seed=N)), N, DXY) for N, n in grids]
    W = 11
    rng = np.random.default_rng(5)
    It = torch.tensor(I * np.exp(0.1 * rng.standard_normal((W, len(I)))), device=DEV)
    g = np.tile(GEOM, (W, 1)) * (1 + 0.01 * rng.standard_normal((W, 4)))
    plan = ta.BatchedChi2Profile(sets, len(I), RMIN, dR, W, check_central_pixel=False)
    for chunk in (W, 4):
        plan.set_chunk(W, chunk, 4)
        tot, per = plan(It, torch.tensor(g, device=DEV), return_sets=True)
        for k in range(W):
            for j, (ds, N, _) in enumerate(sets):
                one = ds.chi2_profile(It[k].contiguous(), RMIN, dR, N, DXY, inc=g[k, 0], PA=g[k, 1], dRA=g[k, 2],
                                      dDec=g[k, 3], check_central_pixel=False).item()
                assert abs(per[k, j].item() - one) <= 1e-12 * abs(one)


@pytest.mark.parametrize('N', [128, 1024])
def test_grid_edge(N):
    """A point on the last column, and on the first and last rows that have a cell, against points just inside."""
    import galario_amd.double as gD
    I, dR = profile()
    duv = 1 / (N * DXY)
    h = N // 2
    u = np.array([h, h, 3.25, 3.25]) * duv
    v = np.array([0.0, 5.5, (h - 1) * (1 - 1e-15), -h]) * duv
    inside = np.array([1 - 1e-13, 1 - 1e-13, 1.0, 1.0]), np.array([1.0, 1.0, 1 - 1e-13, 1 - 1e-13])
    a = gD.sampleProfile(I, RMIN, dR, N, DXY, u, v, inc=0.3, check_central_pixel=False)
    b = gD.sampleProfile(I, RMIN, dR, N, DXY, u * inside[0], v * inside[1], inc=0.3, check_central_pixel=False)
    assert np.isfinite(a).all()
    assert (np.abs(a - b) <= 1e-9 * np.abs(b).max()).all(), (a, b)


@pytest.mark.parametrize('offset', [0.0, 1e-9, 0.03 * O.ARCSEC, 40 * O.ARCSEC, 3.0])
def test_phase(offset):
    """Offsets from none to many turns across the uv plane: exp(2 pi i (u dRA + v dDec)) in long double."""
    import galario_amd.double as gD
    N, (I, dR) = 256, profile()
    u, v = points(2000, N, 1.0, 0.45 * N)[:2]
    base = gD.sampleProfile(I, RMIN, dR, N, DXY, u, v, check_central_pixel=False)
    got = gD.sampleProfile(I, RMIN, dR, N, DXY, u, v, dRA=offset, dDec=-0.5 * offset, check_central_pixel=False)
    # the argument itself carries two roundings of its terms
    turns = u.astype(np.longdouble) * offset - v.astype(np.longdouble) * (0.5 * offset)
    x = (turns - np.rint(turns)).astype(np.float64)
    ref = base.real * np.exp(2j * np.pi * x)
    slack = 2 * np.pi * 4 * 2.2e-16 * (np.abs(u) + np.abs(v)).max() * abs(offset)
    assert np.abs(got - ref).max() <= (4e-15 + slack) * np.abs(base).max()
