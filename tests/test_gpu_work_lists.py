"""The operators' work lists: every run of a cell's entries is cut into equal chunks of at most the
list's size (one that fits full rounds of the card's blocks, where there is one), the chunks are marked
when they share a cell, and the list goes from the largest to the smallest. Lists short enough to be ranked (equal ones then in plan order), possibly long but short in
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


def sizes(nmt):
    """(cap, limit) options of map2tod's and of tod2map's list, in the order of preference."""
    def options(slots, fixed, kmax, least, general):
        opt = [(max(least, -(-nmt * m // (100 * k * slots))), k * slots) for k in range(1, kmax + 1)
               for m in (105, 115, 130, 150)]
        opt = [o for o in opt if o[0] <= 8192][:11]
        opt.sort(key=lambda o: o[1] // slots * (fixed + o[0]))
        return opt + [(general, 1 << 32)]
    return (options(512, 100, 1 if nmt <= 512 * 512 else 0, 128, min(8192, max(512, -(-nmt // 3072)))),
            options(256, 700, 3, 512, min(8192, max(1024, -(-nmt // 512)))))


def bound(opt, nmt, nkeys):
    return max([-(-nmt // opt[-1][0]) + min(nmt, nkeys)] + [min(lim, nmt) for _, lim in opt[:-1]])


def check_list(chunks, mt, opt, ranked):
    cell = mt & np.uint64(0xfffff)
    begin = np.flatnonzero(np.r_[True, cell[1:] != cell[:-1]])
    cnt = np.diff(np.r_[begin, len(mt)])
    cap = next(cap for cap, lim in opt if ((cnt + cap - 1) // cap).sum() <= lim)
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
    ("lines", 32 * 15000, 640, 640), ("lines", 32 * 15000, 300, 300), ("lines", 32 * 70000, 1000, 2000),
    ("lines", 32 * 70000, 1600, 2000), ("lines", 32 * 1000, 8960, 8960), ("samples", 16384, 8960, 8960), ("samples", 60000, 8960, 8960)])
def test_work_lists(gmm, dev, kind, n, ny, nx):
    xg = torch.from_numpy(make_pointing(kind, n, ny, nx)).to(dev)
    pre = gmm.PointingPrePlan(xg, ny, nx, periodic_xcoord=False)
    plan = gmm.PointingPlan(pre, xg, debug=True)
    nmt, mt = pre.plan_nmt, plan.get_plan_mt()
    nkeys = -(-ny // 64) * -(-nx // 64)
    buf = plan.buf.cpu().numpy()
    end = pre.plan_nbytes - align128(2 * nmt)           # the owned-quad masks end the buffer
    opts = sizes(nmt)
    bounds = [bound(opt, nmt, nkeys) for opt in opts]
    assert pre.max_nchunks == bounds[0]
    for opt, nmax in zip(opts[::-1], bounds[::-1]):     # tod2map's list, before it map2tod's
        end -= align128(16 * nmax)
        check_list(buf[end:end + 16 * nmax].view(CHUNK), mt, opt, max(bounds) <= RANK_MAX)


@pytest.mark.parametrize("kind,n,ny,nx", [("samples", 60000, 8960, 8960), ("lines", 32 * 25000, 12800, 12800),
                                          ("samples", 20000, 65536, 65536)])
def test_long_list_ties(gmm, dev, kind, n, ny, nx):
    """Lists that the radix sort orders: equal chunks in plan order, so that a plan has one list."""
    xg = torch.from_numpy(make_pointing(kind, n, ny, nx)).to(dev)
    pre = gmm.PointingPrePlan(xg, ny, nx, periodic_xcoord=False)
    plan = gmm.PointingPlan(pre, xg)
    nmt, mt = pre.plan_nmt, plan.get_plan_mt()
    buf = plan.buf.cpu().numpy()
    end = pre.plan_nbytes - align128(2 * nmt)
    for opt in sizes(nmt)[::-1]:
        nmax = bound(opt, nmt, -(-ny // 64) * -(-nx // 64))
        end -= align128(16 * nmax)
        check_list(buf[end:end + 16 * nmax].view(CHUNK), mt, opt, True)
    assert plan.nchunks > RANK_MAX


@pytest.mark.parametrize("rows", [88, 90, 91, 112])              # x 100 cells: ranked up to 9000, sorted above
def test_list_order_limit(gmm, dev, rows):
    ny, nx, n = 64 * rows, 6400, 32 * 1500 * rows
    xg = torch.from_numpy(make_pointing("lines", n, ny, nx)).to(dev)
    pre = gmm.PointingPrePlan(xg, ny, nx, periodic_xcoord=False)
    plan = gmm.PointingPlan(pre, xg, debug=True)
    assert plan.nchunks == 100 * rows
    nmt, mt = pre.plan_nmt, plan.get_plan_mt()
    buf = plan.buf.cpu().numpy()
    end = pre.plan_nbytes - align128(2 * nmt)
    for opt in sizes(nmt)[::-1]:
        nmax = bound(opt, nmt, 100 * rows)
        end -= align128(16 * nmax)
        check_list(buf[end:end + 16 * nmax].view(CHUNK), mt, opt, True)


@pytest.mark.parametrize("kind,n", [("samples", 60000), ("lines", 32 * 90000)])
def test_plan_on_another_stream(gmm, dev, kind, n):
    """A plan may be used on any stream once its constructor returns, also where a list is sorted after
    the counts have come back: operators started at once on a second stream against the same later."""
    ny = nx = 6400                                       # 10000 cells
    xg = torch.from_numpy(make_pointing(kind, n, ny, nx)).to(dev)
    lp = gmm.LocalPixelization.make_rectangle(ny, nx, periodic_xcoord=False)
    m = gmm.LocalMap(lp, torch.randn(3 * lp.npix, device=dev))
    tod = torch.randn(n, device=dev)
    made, used = torch.cuda.Stream(), torch.cuda.Stream()
    out = torch.zeros(n, device=dev)
    acc = gmm.LocalMap(lp, torch.zeros(3 * lp.npix, device=dev))
    torch.cuda.synchronize()
    with torch.cuda.stream(made):
        pre = gmm.PointingPrePlan(xg, ny, nx, periodic_xcoord=False)
        plan = gmm.PointingPlan(pre, xg)
    with torch.cuda.stream(used):
        gmm.map2tod(out, m, xg, plan)
        gmm.tod2map(acc, tod, xg, plan)
    torch.cuda.synchronize()
    assert plan.nchunks > 9000
    out2, acc2 = torch.zeros(n, device=dev), gmm.LocalMap(lp, torch.zeros(3 * lp.npix, device=dev))
    gmm.map2tod(out2, m, xg, plan)
    gmm.tod2map(acc2, tod, xg, plan)
    assert torch.equal(out, out2)
    # Blocks add to a pixel in any order: float32 rounding of a few deposits.
    assert torch.allclose(acc.arr, acc2.arr, rtol=1e-5, atol=1e-5)
