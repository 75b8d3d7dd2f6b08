"""Plan-free tod2map sums four samples per lane over windows of 1024 samples: scan directions, speeds
and lengths at the edges of that, scattered and wrapping pointing, absent cells and non-finite values,
against the FP64 oracle. The reference compares its unplanned kernels with its CPU ones in the same way
(gpu_mm/tests.py:280-354).
"""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

F32 = np.float32
NY, NX = 300, 700

# name: (y, x) of sample index t, in pixels
SCANS = {
    "along_x": lambda t: (150.3 + 0.0025 * t, 350 + 200 * np.abs((t / 4096.0) % 2 - 1) - 100),
    "back_x": lambda t: (150.7 - 0.004 * t % 20, 500 - 0.21 * t % 300),
    "steep": lambda t: (20 + 0.13 * t % 250, 300.5 + 0.02 * t % 40),
    "diagonal": lambda t: (30 + 0.07 * t % 200, 80.5 + 0.07 * t % 200),
    "antidiagonal": lambda t: (280 - 0.09 * t % 200, 80.5 + 0.2 * t % 500),
    "fast": lambda t: (150 + 0.3 * t % 100, 20 + 0.74 * t % 600),
    "still": lambda t: (63.5 + 0 * t, 127.5 + 0 * t),
    "grid_corner": lambda t: (63.2 + 0.0004 * t % 2, 191.1 + 0.0007 * t % 2),
    "scattered": None,
}


def make_scan(name, n, periodic, seed):
    t = np.arange(n, dtype=np.float64)
    rng = np.random.default_rng(seed)
    if SCANS[name] is None:
        y, x = rng.uniform(0, NY - 1, n), rng.uniform(0, NX - 2, n)
    else:
        y, x = SCANS[name](t)
        if periodic:                       # cross the boundary at x = NX, and start one map width off
            x = x + NX - 350.0 - (NX if seed % 2 else 0)
    xp = np.stack([y, x, 0.3 + 0.001 * t]).astype(F32)
    return np.ascontiguousarray(xp)


def run(gmm, dev, lp, xp, tod, partial=False):
    m = gmm.LocalMap(lp, torch.zeros(3 * lp.npix, dtype=torch.float32, device=dev))
    gmm.tod2map(m, torch.from_numpy(tod).to(dev), torch.from_numpy(xp).to(dev), None, partial_pixelization=partial)
    return m.arr.cpu().numpy()


@pytest.mark.parametrize("name", sorted(SCANS))
@pytest.mark.parametrize("n", [1, 3, 4, 1023, 1024, 1029, 9000])
@pytest.mark.parametrize("periodic", [False, True])
def test_planfree_tod2map_window(gmm, orc, dev, name, n, periodic):
    xp = make_scan(name, n, periodic, n)
    tod = np.random.default_rng(n).standard_normal(n).astype(F32)
    lp = gmm.LocalPixelization.make_rectangle(NY, NX, periodic_xcoord=periodic)
    # Pixel location wraps periodic x by a float32 addition of +-NX: the oracle gets x after it.
    xw = xp.copy()
    if periodic:
        xw[1] = np.where(xw[1] < 0, xw[1] + F32(NX), xw[1])
        xw[1] = np.where(xw[1] > NX, xw[1] - F32(NX), xw[1])
    ref, err = orc.tod2map(tod.astype(np.float64), xw, orc.Pix.rectangle(NY, NX, periodic), f64=True)
    assert err == 0
    got = run(gmm, dev, lp, xp, tod).astype(np.float64)
    # Each deposit carries a few roundings of its weight (x wraps with the rounding of x +- NX, half
    # an ulp of 2 NX), a pixel's sums fewer than its deposits.
    mag, _ = orc.tod2map(np.abs(tod).astype(np.float64), np.stack([xw[0], xw[1], 0 * xw[2]]),
                         orc.Pix.rectangle(NY, NX, periodic), f64=True)
    mag = mag.reshape(3, -1)[0]
    bound = 2e-6 * mag + (1e-4 * np.abs(tod).max() if periodic else 0) + 1e-6 * np.abs(tod).max()
    assert np.all(np.abs(got - ref).reshape(3, -1) <= bound)
    assert np.sum(np.abs(got - ref)) <= 1e-5 * np.sum(np.abs(ref))


def test_planfree_tod2map_absent_cells(gmm, orc, dev):
    # The four samples of a lane step diagonally over a cell corner: the cells beside the path are
    # absent and not touched; one that is touched with a zero value is an error.
    n = 4096
    t = np.arange(n) * (8.0 / n)
    xp = np.ascontiguousarray(np.stack([60.0 + t, 60.0 + t, 0 * t]).astype(F32))
    off = np.full((3, 3), -1, dtype=np.int64)
    off[0, 0], off[1, 1], off[0, 1], off[1, 0] = 0, 12288, 24576, 36864
    lp = gmm.LocalPixelization(192, 192, off, ystride=64, polstride=4096, periodic_xcoord=False)
    got = run(gmm, dev, lp, xp, np.ones(n, F32))
    ref, err = orc.tod2map(np.ones(n), xp, orc.Pix(192, 192, off, 64, 4096, False), f64=True)
    assert err == 0
    assert np.sum(np.abs(got - ref)) <= 1e-5 * np.sum(np.abs(ref))
    # Steps of a whole pixel along the diagonal, whose footprints do not reach (63, 65) and (65, 63).
    xs = np.ascontiguousarray(np.repeat(np.array([[62.5], [62.5], [0.0]]), 4, axis=1).astype(F32))
    xs[:2, 2:] = 64.5
    off2 = off.copy()
    off2[0, 1] = off2[1, 0] = -1
    off2[1, 1] = 12288
    lp2 = gmm.LocalPixelization(192, 192, off2, ystride=64, polstride=4096, periodic_xcoord=False)
    run(gmm, dev, lp2, xs, np.ones(4, F32))
    with pytest.raises(RuntimeError, match="not in LocalPixelization"):
        run(gmm, dev, lp2, xp, np.zeros(n, F32))
    run(gmm, dev, lp2, xp, np.ones(n, F32), partial=True)


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_planfree_tod2map_nonfinite(gmm, dev, bad):
    # A value that is not finite reaches its own four pixels and no others, also in a group of four
    # that steps over a pixel boundary.
    n = 1024
    xp = make_scan("diagonal", n, False, 0)
    tod = np.ones(n, F32)
    tod[513] = bad
    lp = gmm.LocalPixelization.make_rectangle(NY, NX, periodic_xcoord=False)
    got = run(gmm, dev, lp, xp, tod).reshape(3, lp.nycells * 64, lp.nxcells * 64)
    iy, ix = int(xp[0, 513]), int(xp[1, 513])
    hit = np.zeros(got.shape, bool)
    hit[:, iy:iy + 2, ix:ix + 2] = True
    assert np.all(np.isfinite(got[~hit]))
    assert not np.any(np.isfinite(got[hit]))


@pytest.mark.parametrize("kind", ["corners", "scattered", "jumps"])
@pytest.mark.parametrize("periodic", [False, True])
def test_planfree_tod2map_large_map(gmm, orc, dev, kind, periodic):
    # Positions up to the largest map (16 bits a coordinate), and samples of one block that lie tens of
    # thousands of pixels apart, in a map of a few cells.
    ny = nx = 65536
    n = 5000
    rng = np.random.default_rng(n)
    cells = [(0, 0), (0, 1023), (1023, 0), (1023, 1023), (511, 512), (512, 511)]
    k = {"corners": np.arange(n) // 1024, "scattered": rng.integers(0, 6, n), "jumps": np.arange(n) // 300}[kind] % 6
    c = np.array(cells)[k]
    t = np.arange(n)
    step = rng.uniform(0, 62, (2, n)) if kind == "scattered" else np.stack([0.02 * t % 60, 0.2 * t % 60])
    xp = np.stack([64 * c[:, 0] + step[0] + 0.5, 64 * c[:, 1] + step[1] + 0.5, 0.001 * t]).astype(F32)
    xp[0] = np.minimum(xp[0], ny - 2)
    xp[1] = np.minimum(xp[1], nx - 2.5)
    tod = rng.standard_normal(n).astype(F32)
    lp = gmm.LocalPixelization.make_cells(ny, nx, cells, periodic_xcoord=periodic)
    pix = orc.Pix(ny, nx, lp.cell_offsets_cpu, 64, 4096, periodic)
    ref, err = orc.tod2map(tod.astype(np.float64), xp, pix, f64=True)
    assert err == 0
    got = run(gmm, dev, lp, xp, tod).astype(np.float64)
    mag, _ = orc.tod2map(np.abs(tod).astype(np.float64), np.stack([xp[0], xp[1], 0 * xp[2]]), pix, f64=True)
    mag = np.repeat(mag.reshape(len(cells), 3, 4096)[:, :1], 3, axis=1).reshape(-1)
    # The bound of the smaller maps: roundings of the weights (exact differences of coordinates here too).
    assert np.all(np.abs(got - ref) <= 2e-6 * mag + 1e-6 * np.abs(tod).max())
    assert np.sum(np.abs(got - ref)) <= 1e-5 * np.sum(np.abs(ref))


def make_runs(kind, n, periodic, seed):
    """Samples of which a window holds some or none: detectors of 16 samples at places of their own, short
    turns, and scans too fast for four samples in 3 x 3 pixels."""
    rng = np.random.default_rng(seed)
    t = np.arange(n, dtype=np.float64)
    hi = NX - (0 if periodic else 2)
    if kind == "detectors":
        run = np.arange(n) // 16
        y, x = rng.uniform(0, NY - 4, run[-1] + 1)[run] + 0.1 * (t % 16), rng.uniform(0, hi, run[-1] + 1)[run] + 0.13 * (t % 16)
    elif kind == "turns":
        y, x = 100 + 60 * np.sin(t / 700), 300 + 90 * np.abs((t / 150) % 2 - 1)
    elif kind == "fast_x":
        y, x = 40 + 0.02 * t % 200, 1.3 * t % hi
    else:                                # "fast_y"
        y, x = NY / 2 + (NY / 2 - 3) * (2 * np.abs((t / 250) % 2 - 1) - 1), 50 + 0.011 * t % 600
    x = x % hi if periodic else np.clip(x, 0, hi)
    xp = np.stack([np.clip(y, 0, NY - 1), x, 0.3 + 0.001 * t]).astype(F32)
    xp[1] = np.minimum(xp[1], np.nextafter(F32(NX), F32(0)) if periodic else F32(hi))
    return np.ascontiguousarray(xp)


@pytest.mark.parametrize("kind", ["detectors", "turns", "fast_x", "fast_y"])
@pytest.mark.parametrize("n", [33, 3001, 70002])                # one block, a few, and more than 64
@pytest.mark.parametrize("periodic", [False, True])
def test_planfree_tod2map_outside(gmm, orc, dev, kind, n, periodic):
    xp = make_runs(kind, n, periodic, n)
    tod = np.random.default_rng(n).standard_normal(n).astype(F32)
    # Every third cell is absent.
    cells = [(cy, cx) for cy in range(5) for cx in range(11) if (cy + cx) % 3]
    lp = gmm.LocalPixelization.make_cells(NY, NX, cells, periodic_xcoord=periodic)
    pix = orc.Pix(NY, NX, lp.cell_offsets_cpu, 64, 4096, periodic)
    for lmap, opix, partial in [(lp, pix, True), (gmm.LocalPixelization.make_rectangle(NY, NX, periodic_xcoord=periodic),
                                                  orc.Pix.rectangle(NY, NX, periodic), False)]:
        ref, err = orc.tod2map(tod.astype(np.float64), xp, opix, partial=partial, f64=True)
        assert err == 0
        got = run(gmm, dev, lmap, xp, tod, partial).astype(np.float64)
        mag, _ = orc.tod2map(np.abs(tod).astype(np.float64), np.stack([xp[0], xp[1], 0 * xp[2]]), opix, partial=partial,
                             f64=True)
        if partial:
            mag = np.repeat(mag.reshape(-1, 3, 4096)[:, :1], 3, axis=1).reshape(-1)
        else:
            mag = np.tile(mag.reshape(3, -1)[0], 3)
        assert np.all(np.abs(got - ref) <= 2e-6 * mag + 1e-6 * np.abs(tod).max())
    if n > 100:
        with pytest.raises(RuntimeError, match="not in LocalPixelization"):
            run(gmm, dev, lp, xp, tod)
    # A value that is not finite reaches its own four pixels alone.
    k = n // 2
    tod[k] = np.nan
    got = run(gmm, dev, lmap, xp, tod).reshape(3, lmap.nycells * 64, lmap.nxcells * 64)
    iy, ix = min(int(xp[0, k]), NY - 2), int(xp[1, k]) if periodic else min(int(xp[1, k]), NX - 2)
    hit = np.zeros(got.shape, bool)
    hit[:, iy:iy + 2, [ix, (ix + 1) % NX]] = True
    assert np.all(np.isnan(got[hit])) and not np.any(np.isnan(got[~hit]))


@pytest.mark.parametrize("nx", [64, 65, 66, 128, 129, 130])
def test_planfree_tod2map_last_column(gmm, orc, dev, nx):
    # Detectors of 16 slow samples around the column where periodic x wraps, at rows of their own, so that
    # windows hold few of them: the last cell column may be one or two pixels wide.
    ny, n = 2000, 300000
    rng = np.random.default_rng(nx)
    t, run_ = np.arange(n), np.arange(n) // 16
    y = rng.uniform(0, ny - 4, run_[-1] + 1)[run_] + 0.1 * (t % 16)
    x = (rng.uniform(nx - 4, nx + 2, run_[-1] + 1)[run_] + 0.07 * (t % 16)) % nx
    xp = np.ascontiguousarray(np.stack([y, np.minimum(x, np.nextafter(F32(nx), F32(0))), 0.3 + 0.001 * t]).astype(F32))
    tod = rng.standard_normal(n).astype(F32)
    lp, pix = gmm.LocalPixelization.make_rectangle(ny, nx, periodic_xcoord=True), orc.Pix.rectangle(ny, nx, True)
    ref, err = orc.tod2map(tod.astype(np.float64), xp, pix, f64=True)
    assert err == 0
    got = run(gmm, dev, lp, xp, tod).astype(np.float64)
    mag, _ = orc.tod2map(np.abs(tod).astype(np.float64), np.stack([xp[0], xp[1], 0 * xp[2]]), pix, f64=True)
    mag = np.tile(mag.reshape(3, -1)[0], 3)
    # A pixel takes some 100 (at most 200) roundings of 6e-8 of its sum, sine, cosine and weights a few more.
    assert np.all(np.abs(got - ref) <= 2e-5 * mag + 1e-6 * np.abs(tod).max())
