"""Error flags and counts that a call waits for: after work that is still running on the call's stream,
from several threads on streams of their own, and with errors in some of the calls."""

import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

NY, NX = 100, 130


def make_pointing(n, seed, dev):
    rng = np.random.default_rng(seed)
    xp = np.stack([rng.uniform(0, NY - 1.5, n), rng.uniform(0, NX - 2.5, n), rng.uniform(0, 3, n)])
    return torch.from_numpy(xp.astype(np.float32)).to(dev)


@pytest.mark.parametrize("cycles", [0, 10000, 4000000])     # the last far longer than the polled wait
def test_waits_for_the_stream(gmm, dev, cycles):
    xg = make_pointing(4096, 1, dev)
    plan = gmm.PointingPlan(gmm.PointingPrePlan(xg, NY, NX, periodic_xcoord=False), xg)
    lp = gmm.LocalPixelization.make_rectangle(NY, NX, periodic_xcoord=False)
    m = gmm.LocalMap(lp, torch.ones(3 * lp.npix, dtype=torch.float32, device=dev))
    tod = torch.zeros(4096, dtype=torch.float32, device=dev)
    good = xg.clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        torch.cuda._sleep(cycles) if cycles else None
        xg[0, 7] = -3.0                                     # bad by the time the operator runs
        with pytest.raises(RuntimeError, match="y-value"):
            gmm.map2tod(tod, m, xg, plan)
        torch.cuda._sleep(cycles) if cycles else None
        xg.copy_(good)
        assert gmm.PointingPrePlan(xg, NY, NX, periodic_xcoord=False).plan_nmt == plan.plan_nmt
        gmm.map2tod(tod, m, xg, plan)                       # flags were cleared
    torch.cuda.current_stream().wait_stream(s)
    want = 1 + torch.cos(2 * good[2]) + torch.sin(2 * good[2])
    assert torch.allclose(tod, want, atol=1e-5)             # unit map: weights sum to 1


def test_threads(gmm, dev):
    """More calls at once than one thread's, each with its own outcome."""
    nthreads, ncalls = 12, 40
    xgs = [make_pointing(1000 + 37 * i, i, dev) for i in range(nthreads)]
    bad = [x.clone() for x in xgs]
    for i, b in enumerate(bad):
        b[0, 5 * i] = NY + 1.0
    nmt = [gmm.PointingPrePlan(x, NY, NX, periodic_xcoord=False).plan_nmt for x in xgs]
    torch.cuda.synchronize()
    failures = []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for k in range(ncalls):
                    if (i + k) % 3:
                        assert gmm.PointingPrePlan(xgs[i], NY, NX, periodic_xcoord=False).plan_nmt == nmt[i]
                    else:
                        with pytest.raises(RuntimeError, match="y-value"):
                            gmm.PointingPrePlan(bad[i], NY, NX, periodic_xcoord=False)
        except BaseException as e:                          # an assertion in a thread fails the test
            failures.append((i, repr(e)))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(nthreads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join(60)
    assert not failures and not any(t.is_alive() for t in ts)


@pytest.mark.parametrize("bad", [None, 0, 4095 * 256, 4096 * 256, 5000 * 256 - 1])
def test_many_words(gmm, dev, bad):
    """A word of 5000 blocks, more than the reading block takes at a time."""
    n = 5000 * 256
    xg = make_pointing(n, 3, dev)
    if bad is not None:
        xg[0, bad] = -1.0
    lp = gmm.LocalPixelization.make_rectangle(NY, NX, periodic_xcoord=False)
    m = torch.ones(3 * lp.npix, dtype=torch.float32, device=dev)
    tod = torch.zeros(n, dtype=torch.float32, device=dev)
    words = torch.empty(8192, dtype=torch.uint32, device=dev)
    ext = gmm.gpu_mm._ext
    call = lambda: ext.unplanned_map2tod(tod, m, xg, lp, words, False, False, check_errors=True, stream=0)
    torch.cuda.synchronize()
    if bad is None:
        call()
    else:
        with pytest.raises(RuntimeError, match="y-value"):
            call()


def test_more_callers_than_slots(gmm, dev):
    """80 calls that wait at once, behind work on one stream: those that find no slot of pinned memory
    (there are 64) take a copy."""
    nthreads = 80
    good, bad = make_pointing(3000, 5, dev), make_pointing(3000, 5, dev)
    bad[0, 1234] = NY + 1.0
    nmt = gmm.PointingPrePlan(good, NY, NX, periodic_xcoord=False).plan_nmt
    lp = gmm.LocalPixelization.make_rectangle(NY, NX, periodic_xcoord=False)
    m = gmm.LocalMap(lp, torch.ones(3 * lp.npix, dtype=torch.float32, device=dev))
    tods = torch.zeros((nthreads, 3000), dtype=torch.float32, device=dev)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        torch.cuda._sleep(40000000)
    failures = []

    def work(i):
        try:
            with torch.cuda.stream(s):
                if i % 4 == 0:
                    assert gmm.PointingPrePlan(good, NY, NX, periodic_xcoord=False).plan_nmt == nmt
                elif i % 4 == 1:
                    with pytest.raises(RuntimeError, match="y-value"):
                        gmm.PointingPrePlan(bad, NY, NX, periodic_xcoord=False)
                elif i % 4 == 2:
                    gmm.map2tod(tods[i], m, good, None)
                else:
                    with pytest.raises(RuntimeError, match="y-value"):
                        gmm.map2tod(tods[i], m, bad, None)
        except BaseException as e:
            failures.append((i, repr(e)))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(nthreads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join(60)
    assert not failures and not any(t.is_alive() for t in ts)
    want = 1 + torch.cos(2 * good[2]) + torch.sin(2 * good[2])
    assert torch.allclose(tods[2::4], want.expand(20, 3000), atol=1e-5)
