"""Gains and 16-bit scales whose rows are whole groups of four samples or of any length, one or both: the
planned and batched operators against the FP64 response oracle."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

F32 = np.float32
NY, NX, N = 200, 300, 20160
BAR = 1e-5                                   # as for the response operators elsewhere


def make_case(gmm, dev, seed):
    rng = np.random.default_rng(seed)
    t = np.arange(N)
    xp = np.stack([100 + 90 * np.sin(t / 300.0 + seed), 150 + 140 * np.sin(t / 410.0), rng.uniform(-3, 3, N)]).astype(F32)
    xg = torch.from_numpy(xp).to(dev)
    plan = gmm.PointingPlan(gmm.PointingPrePlan(xg, NY, NX, periodic_xcoord=False), xg)
    return rng, xp, xg, plan


def l1rel(a, ref):
    return float(np.abs(a - ref).sum() / np.abs(ref).sum())


@pytest.mark.parametrize("dtype,eps,tiny", [(torch.float16, 2.0 ** -11, 2.0 ** -25), (torch.bfloat16, 2.0 ** -8, 0.0)])
@pytest.mark.parametrize("ndet,nrows", [(24, 24), (24, 2240), (24, 32), (2240, 24), (2016, 2240), (0, 24), (0, 2240)])
def test_planned_16bit(gmm, orc, dev, ndet, nrows, dtype, eps, tiny):
    rng, xp, xg, plan = make_case(gmm, dev, ndet + nrows)
    lp, pix = gmm.LocalPixelization.make_rectangle(NY, NX, periodic_xcoord=False), orc.Pix.rectangle(NY, NX, False)
    resp = rng.uniform(0.5, 2, size=(2, max(ndet, 1))).astype(F32) if ndet else np.ones((2, 1), F32)
    kw = dict(response=torch.from_numpy(resp).to(dev)) if ndet else {}
    tod = rng.standard_normal((nrows, N // nrows)).astype(F32)
    t16, sc = gmm.encode_tod16(torch.from_numpy(tod).to(dev), dtype)
    dec = (t16.float() * sc[:, None]).cpu().numpy().reshape(-1)
    out = gmm.LocalMap(lp, torch.zeros(3 * lp.npix, dtype=torch.float32, device=dev))
    gmm.tod2map(out, t16.view(-1), xg, plan, tod_scale=sc, **kw)
    ref, err = orc.response_tod2map(dec, xp, resp, pix)
    assert err == 0 and l1rel(out.arr.cpu().numpy(), ref) < BAR
    m = rng.standard_normal(3 * lp.npix).astype(F32)
    osc = sc * 16                            # headroom for the gains and T + Q + U
    gmm.map2tod(t16.view(-1), gmm.LocalMap(lp, torch.from_numpy(m).to(dev)), xg, plan, tod_scale=osc, **kw)
    got = (t16.double() * osc.double()[:, None]).cpu().numpy().reshape(-1)
    ref, err = orc.response_map2tod(m, xp, resp, pix)
    assert err == 0
    step = np.repeat(osc.cpu().numpy().astype(np.float64), N // nrows)
    assert np.all(np.abs(got - ref) <= eps * np.abs(ref) + tiny * step + BAR * np.abs(ref).max())


@pytest.mark.parametrize("ndets", [(24, 48), (24, 2240), (2240, 2016)])
def test_batched(gmm, orc, dev, ndets):
    lp, pix = gmm.LocalPixelization.make_rectangle(NY, NX, periodic_xcoord=False), orc.Pix.rectangle(NY, NX, False)
    case = [make_case(gmm, dev, i) for i in range(len(ndets))]
    rng = case[0][0]
    resps = [rng.uniform(0.5, 2, size=(2, nd)).astype(F32) for nd in ndets]
    tods = [rng.standard_normal(N).astype(F32) for _ in ndets]
    tg = [torch.from_numpy(t).to(dev) for t in tods]
    b = gmm.PlanBatch(lp, [c[3] for c in case], [c[2] for c in case], tg)
    b.set_response([torch.from_numpy(r).to(dev) for r in resps])
    out = gmm.LocalMap(lp, torch.zeros(3 * lp.npix, dtype=torch.float32, device=dev))
    b.tod2map(out)
    ref = sum(orc.response_tod2map(t, c[1], r, pix)[0] for t, c, r in zip(tods, case, resps))
    assert l1rel(out.arr.cpu().numpy(), ref) < BAR
    m = rng.standard_normal(3 * lp.npix).astype(F32)
    b.map2tod(gmm.LocalMap(lp, torch.from_numpy(m).to(dev)))
    for t, c, r in zip(tg, case, resps):
        assert l1rel(t.cpu().numpy(), orc.response_map2tod(m, c[1], r, pix)[0]) < BAR
