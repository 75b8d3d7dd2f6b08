"""The operators' work lists: every run of a cell's entries is cut into equal chunks of at most the
list's size, the chunks are marked when they share a cell, and the list goes from the largest to the
smallest. Lists short enough to be ranked (equal ones then in plan order), possibly long but short in
fact, and long ones, which a radix sort orders.
"""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

RANK_MAX = 16384
CHUNK = np.dtype([("icell", "<u4"), ("begin", "<u4"), ("end", "<u4"), ("flags", "<u4")])


def align128(n):
    return (n + 127) // 128 * 128


def make_pointing(kind, n, ny, nx):
    rng = np.random.default_rng(n)
    if kind == "one cell":
        y, x = rng.uniform(70, 120, n), rng.uniform(70, 120, n)
    else:                               # "lines": each line in one cell; "samples": each sample in any
        k = np.arange(n) // (32 if kind == "lines" else 1)
        y, x = rng.uniform(1, ny - 2, k[-1] + 1)[k], rng.uniform(1, nx - 3, k[-1] + 1)[k]
    return np.stack([y, x, 0 * y]).astype(np.float32)


def check_list(chunks, mt, cap, ranked):
    cell = mt & np.uint64(0xfffff)
    begin = np.flatnonzero(np.r_[True, cell[1:] != cell[:-1]])
    cnt = np.diff(np.r_[begin, len(mt)])
    nc = (cnt + cap - 1) // cap
    want = [(int(cell[b]), b + c * j // m, b + c * (j + 1) // m, int(m > 1))
            for b, c, m in zip(begin.tolist(), cnt.tolist(), nc.tolist()) for j in range(m)]
    got = [tuple(int(v) for v in c) for c in chunks[:len(want)]]
    assert sorted(got, key=lambda c: c[1]) == want
    size = np.array([c[2] - c[1] for c in got])
    assert np.all(size[1:] <= size[:-1])
    if ranked:
        assert got == sorted(want, key=lambda c: (c[1] - c[2], c[1]))


@pytest.mark.parametrize("kind,n,ny,nx", [
    ("one cell", 1, 200, 330), ("one cell", 32 * 512, 200, 330), ("one cell", 32 * 1024 + 1, 200, 330),
    ("one cell", 32 * 70001, 200, 330), ("lines", 32 * 4096, 640, 1281), ("samples", 20000, 640, 1281),
    ("lines", 32 * 1000, 8960, 8960), ("samples", 16384, 8960, 8960), ("samples", 60000, 8960, 8960)])
def test_work_lists(gmm, dev, kind, n, ny, nx):
    xg = torch.from_numpy(make_pointing(kind, n, ny, nx)).to(dev)
    pre = gmm.PointingPrePlan(xg, ny, nx, periodic_xcoord=False)
    plan = gmm.PointingPlan(pre, xg, debug=True)
    nmt, mt = pre.plan_nmt, plan.get_plan_mt()
    nkeys = -(-ny // 64) * -(-nx // 64)
    buf = plan.buf.cpu().numpy()
    end = pre.plan_nbytes - align128(2 * nmt)           # the owned-quad masks end the buffer
    caps = min(8192, max(512, -(-nmt // 3072))), min(8192, max(1024, -(-nmt // 512)))
    bound = [-(-nmt // cap) + min(nmt, nkeys) for cap in caps]
    assert pre.max_nchunks == bound[0]
    for cap, nmax in zip(caps[::-1], bound[::-1]):      # tod2map's list, before it map2tod's
        end -= align128(16 * nmax)
        check_list(buf[end:end + 16 * nmax].view(CHUNK), mt, cap, max(bound) <= RANK_MAX)
