"""Planner passes that find a line's cells from the range of its coordinates: plans bit for bit and
owned-quad masks against their rule, on lines of one cell, of two in a row or a column, around a cell
corner, of many cells and across the periodic boundary; with odd lengths and unaligned pointing. The
reference compares its planner with a brute-force one in the same way (gpu_mm/tests.py:227-254).
"""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

F32 = np.float32
HALO_X, TAKES_RIGHT = 12, 0x100


def make_pointing(kind, n, ny, nx, seed):
    """Scans through the middle of cell (1, 1) and its borders, a different one every 32 samples."""
    rng = np.random.default_rng(seed)
    line = np.arange(n) // 32
    t = np.arange(n) % 32
    nl = line[-1] + 1
    y0 = rng.uniform(50, 80, nl) if kind != "rows" else rng.uniform(70, 100, nl)
    x0 = rng.uniform(105, 140, nl)
    speed = {"slow": 0.3, "rows": 0.6, "corner": 0.7, "fast": 6.0, "wrap": 0.5, "still": 0.0}[kind]
    phi = rng.uniform(0, 2 * np.pi, nl)
    if kind == "rows":
        phi[:] = rng.choice([0.0, np.pi], nl)
    y = y0[line] + speed * t * np.sin(phi[line])
    x = x0[line] + speed * t * np.cos(phi[line])
    if kind == "wrap":
        x = x + (nx - 120)
    if kind == "still":
        y, x = np.floor(y), np.floor(x)
    return np.stack([np.clip(y, 0, ny - 1), x if kind == "wrap" else np.clip(x, 0, nx - 2), 0 * y]).astype(F32)


def masks(orc, mt, xp, ny, nx, periodic):
    """Owned-quad mask of every plan entry, from the ownership rule."""
    n = xp.shape[1]
    iy0, _, ix0, _ = np.array([orc.locate(float(y), float(x), ny, nx, periodic)[1] for y, x in xp[:2].T]).T
    lines = {}
    for e in mt:
        lines.setdefault(int(e) >> 20 & (2 ** 26 - 1), set()).add((int(e) >> 10 & 1023, int(e) & 1023))
    out = np.zeros(len(mt), np.uint16)
    for k, e in enumerate(mt):
        icl, cy, cx = int(e) >> 20 & (2 ** 26 - 1), int(e) >> 10 & 1023, int(e) & 1023
        s = np.arange(32 * icl, min(n, 32 * icl + 32))
        quad = (s - 32 * icl) // 4
        cells = lines[icl]
        if len(cells) == 1:
            out[k] = (1 << (quad[-1] + 1)) - 1
            continue
        own = {c: (iy0[s] >> 6 == cy) & (ix0[s] >> 6 == c) for c in (cx - 1, cx, cx + 1)}
        fits = (ix0[s] & 63 <= HALO_X - 2) & (ix0[s] + 1 < nx)

        def given(c):             # the samples of column c, if it has any, fit the halo of column c - 1
            return own[c].any() and fits[own[c]].all()

        def eligible(c):
            return given(c) and (cy, c - 1) in cells

        taken, takes = eligible(cx) and not eligible(cx - 1), given(cx + 1) and not eligible(cx)
        sel = (own[cx] & (not taken)) | (own[cx + 1] & takes)
        out[k] = np.bitwise_or.reduce(1 << quad[sel]) if sel.any() else 0
        out[k] |= TAKES_RIGHT if takes else 0
    return out


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("n", [1, 33, 4000, 4031])
@pytest.mark.parametrize("kind", ["slow", "rows", "corner", "fast", "wrap", "still"])
def test_plan_lines(gmm, orc, dev, kind, n, offset):
    ny, nx, periodic = 200, 330, kind == "wrap"
    xp = make_pointing(kind, n, ny, nx, 17 * n + offset)
    buf = torch.empty(3 * n + offset, dtype=torch.float32, device=dev)     # aligned to 16 bytes or not
    xg = buf[offset:].view(3, n)
    xg.copy_(torch.from_numpy(xp))
    ref, err = orc.plan_build(xp, ny, nx, periodic)
    assert err == 0
    pre = gmm.PointingPrePlan(xg, ny, nx, periodic_xcoord=periodic)
    cum, nmt, _ = orc.plan_count(xp, ny, nx, periodic)
    assert pre.plan_nmt == nmt and np.array_equal(pre.get_nmt_cumsum(), cum)
    plan = gmm.PointingPlan(pre, xg, debug=True)
    assert np.array_equal(plan.get_plan_mt(), ref)
    assert plan.nmlines == int(np.sum(ref >> np.uint64(47) & np.uint64(1)))
    # The masks end the plan's buffer.
    nb = (2 * nmt + 127) // 128 * 128
    got = plan.buf[pre.plan_nbytes - nb:pre.plan_nbytes - nb + 2 * nmt].cpu().numpy().view(np.uint16)
    assert np.array_equal(got, masks(orc, ref, xp, ny, nx, periodic))


@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("n", [31, 500, 32 * 40 + 7, 32 * 16 * 70, 32 * 1024 * 20 + 65])
@pytest.mark.parametrize("share", [0.1, 0.5, 1.0])
def test_scattered_lines(gmm, orc, dev, n, share, periodic):
    """Lines of many cells among ordinary ones, one, several or all of a wave's, of up to 128 cells (every
    sample at a corner of four) and with few lines to a block or many."""
    ny, nx = 1000, 2000
    rng = np.random.default_rng(n + int(10 * share))
    line = np.arange(n) // 32
    nl = line[-1] + 1
    kind = rng.choice([0, 1, 2], nl, p=[1 - share, share / 2, share / 2])[line]
    t = np.arange(n) % 32
    y, x = rng.uniform(0, ny - 20, nl)[line] + 0.1 * t, rng.uniform(0, nx - 20, nl)[line] + 0.3 * t
    ys, xs = rng.uniform(0, ny - 1.5, n), rng.uniform(0, nx - 2.5, n)
    corner = lambda m, k: 64.0 * rng.integers(1, (m - 2) // 64, k) - 0.5
    y = np.choose(kind, [y, ys, corner(ny, n)])
    x = np.choose(kind, [x, xs, corner(nx, n)])
    if periodic:
        x = np.where(kind == 1, x + rng.choice([-nx, 0, nx], n), x)
    xp = np.stack([y, x, 0 * y]).astype(F32)
    xp[1] = np.clip(xp[1], -nx, 2 * nx) if periodic else xp[1]
    ref, err = orc.plan_build(xp, ny, nx, periodic)
    assert err == 0
    xg = torch.from_numpy(xp).to(dev)
    pre = gmm.PointingPrePlan(xg, ny, nx, periodic_xcoord=periodic)
    cum, nmt, _ = orc.plan_count(xp, ny, nx, periodic)
    assert pre.plan_nmt == nmt and np.array_equal(pre.get_nmt_cumsum(), cum)
    plan = gmm.PointingPlan(pre, xg, debug=True)
    assert np.array_equal(plan.get_plan_mt(), ref)
    assert plan.nmlines == int(np.sum(ref >> np.uint64(47) & np.uint64(1)))
