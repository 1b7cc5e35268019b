"""Plans with several grids: the buffers hold the walkers that a grid takes at once and no more, a chunk set by the caller
is taken as it is, and results do not depend on the chunk."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip('torch')

W, DXY, NR = 64, 1e-7, 100
GRIDS = [(4096, 3000), (2048, 700)]
LIMIT = 32              # walkers whose half spectra of 1025 x 1025 doubles come to 288 MB, a power of two


def plan_and_parameters():
    from galario_amd import torch_api as ta
    rng = np.random.default_rng(8)
    sets = []
    for N, n in GRIDS:
        u, v = (rng.uniform(-0.2, 0.2, n) / DXY for _ in range(2))
        sets.append((ta.Dataset(u, v, rng.standard_normal(n), rng.standard_normal(n), rng.uniform(0.5, 2.0, n),
                                device='cuda:0'), N, DXY))
    plan = ta.BatchedChi2Profile(sets, NR, 1e-10, DXY / 5, W, check_central_pixel=False)
    I = 1e10 * np.exp(-np.linspace(0, 3, NR) + 0.1 * rng.standard_normal((W, NR)))
    geom = np.tile((0.6, 1.1, 3e-7, -2e-7), (W, 1)) * (1 + 0.01 * rng.standard_normal((W, 4)))
    return plan, torch.tensor(I, device='cuda:0'), torch.tensor(geom, device='cuda:0')


def used():
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


def test_buffers_and_chunks():
    plan, I, geom = plan_and_parameters()
    spectrum = 8 * 2050 * 2056          # the largest grid's half spectrum, with the padding
    before = used()
    tuned = plan(I, geom).clone()
    # (row spectra of 22 rows, graphs and the allocator's rounding: below a tenth of the spectra)
    assert used() - before <= 1.1 * LIMIT * spectrum + (32 << 20)
    assert 1 <= plan.info(W)[0] <= LIMIT
    for chunk in (1, 7, 8, 33, W):
        plan.set_chunk(W, chunk, 2)
        assert torch.equal(plan(I, geom), tuned)
        assert plan.info(W)[:2] == (chunk, 2)
    assert used() - before >= W * spectrum               # (the caller's chunk is taken as it is)
    plan.close()
