"""Dynamic maps that grow by a plan's work list: the same table and count as the entry point that takes the
plan's entries, over grids from one cell to 1024 a side, with cells present and masked; plans whose list
is too long for one block too."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ny,nx,masked", [
    (5, 60, 60, False), (3000, 64 * 31, 64 * 33, False), (3000, 64 * 31, 64 * 33, True), (40000, 65536, 65536, False),
    (20000, 65536, 100, True), (20000, 100, 65536, False), (32 * 5000, 640, 640, False), (60000, 16384, 16384, True)])
def test_expand_by_plan(gmm, dev, n, ny, nx, masked):
    rng = np.random.default_rng(n + ny)
    nyc, nxc = -(-ny // 64), -(-nx // 64)
    mask = (rng.uniform(size=(nyc, nxc)) < 0.6) if masked else None
    dmap = gmm.DynamicMap(ny, nx, np.float32, cell_mask=mask, periodic_xcoord=False, initial_ncells=65536)
    table = dmap._table.cell_offsets_gpu.clone()
    count = torch.zeros(1, dtype=torch.uint32, device=dev)
    for part in range(3):                                # the later ones find cells present
        m = n // (3 - part)
        xp = np.stack([rng.uniform(0, ny - 1.5, m), rng.uniform(0, nx - 2.5, m), np.zeros(m)]).astype(np.float32)
        if part == 1:
            xp[:2] *= 0.5
        xg = torch.from_numpy(xp).to(dev)
        plan = gmm.PointingPlan(gmm.PointingPrePlan(xg, ny, nx, periodic_xcoord=False), xg)
        want = gmm.expand_dynamic_map(count, table, torch.from_numpy(plan.get_plan_mt()).to(dev))
        dmap.expand(plan)
        assert dmap.ncells_curr == want and int(dmap._count.cpu()[0]) == want
        assert torch.equal(dmap._table.cell_offsets_gpu, table)
