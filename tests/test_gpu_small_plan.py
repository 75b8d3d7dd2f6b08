"""Plans made in one block: entries, flags and work lists around the sizes of a wave, of the block and of
the largest plan that it takes; one cell, many, more chunks than it orders, and the widest keys."""

import numpy as np
import pytest
import torch

from test_gpu_work_lists import CHUNK, align128, bound, check_list, make_pointing, sizes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n,ny,nx", [
    ("samples", 40, 64, 64), ("one cell", 32 * 64 + 5, 200, 330), ("one cell", 32 * 1025, 200, 330),
    ("one cell", 32 * 8192, 200, 330), ("one cell", 32 * 8192 + 1, 200, 330), ("lines", 32 * 63, 640, 1281),
    ("lines", 32 * 2500, 640, 1281), ("samples", 64, 65536, 65536), ("samples", 1000, 65536, 65536),
    ("samples", 1400, 640, 640), ("samples", 3000, 65536, 65536), ("samples", 7600, 2000, 65536)])
def test_small_plan(gmm, orc, dev, kind, n, ny, nx):
    xp = make_pointing(kind, n, ny, nx)
    ref, err = orc.plan_build(xp, ny, nx, False)
    assert err == 0
    xg = torch.from_numpy(xp).to(dev)
    pre = gmm.PointingPrePlan(xg, ny, nx, periodic_xcoord=False)
    plan = gmm.PointingPlan(pre, xg, debug=True)
    mt = plan.get_plan_mt()
    assert np.array_equal(mt, ref)
    assert plan.nmlines == int(np.sum(ref >> np.uint64(47) & np.uint64(1)))
    nmt, nkeys = pre.plan_nmt, -(-ny // 64) * -(-nx // 64)
    buf = plan.buf.cpu().numpy()
    end = pre.plan_nbytes - align128(2 * nmt)
    for opt in sizes(nmt)[::-1]:                         # tod2map's list, before it map2tod's
        nmax = bound(opt, nmt, nkeys)
        end -= align128(16 * nmax)
        check_list(buf[end:end + 16 * nmax].view(CHUNK), mt, opt, True)
