"""Plan-free map2tod on samples whose corners lie in one cell, on cell borders and corners, on both, across
the periodic boundary and in cells that the map does not hold; odd lengths, adding to the TOD or not."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

F32 = np.float32
BAR = 1e-5                                   # as for the operators elsewhere, against FP64


def make_pointing(kind, n, ny, nx, rng):
    if kind == "inside":
        y, x = rng.uniform(66, 126, n), rng.uniform(130, 190, n)
    elif kind == "border":                   # rows 63 | 64 and columns 127 | 128, on and between the pixels
        y, x = 63 + rng.choice([0, 0.5, 1], n), 127 + rng.choice([0, 0.25, 1], n)
    elif kind == "scan":
        t = np.arange(n)
        y, x = 5 + 0.01 * t % (ny - 8), 160 + 150 * np.sin(t / 300.0)
    elif kind == "wrap":                     # the last column's right-hand neighbour is column 0
        y, x = rng.uniform(1, ny - 3, n), np.mod(nx - 3 + rng.uniform(0, 6, n), nx)
        x = np.minimum(x, np.nextafter(F32(nx), F32(0)))
    else:
        y, x = rng.uniform(0, ny - 1.5, n), rng.uniform(0, nx - 2.5, n)
    return np.stack([y, x, rng.uniform(-4, 4, n)]).astype(F32)


@pytest.mark.parametrize("cells", [False, True])
@pytest.mark.parametrize("n", [1, 255, 257, 4099, 70001])
@pytest.mark.parametrize("kind", ["inside", "border", "scan", "random", "wrap"])
def test_planfree_map2tod(gmm, orc, dev, kind, n, cells):
    rng = np.random.default_rng(n)
    ny, nx, periodic = 250, 330, kind == "wrap"
    if cells:
        held = [(cy, cx) for cy in range(4) for cx in range(6) if (cy + cx) % 3 != 0]
        lp = gmm.LocalPixelization.make_cells(ny, nx, held, periodic_xcoord=periodic)
        pix = orc.Pix(ny, nx, lp.cell_offsets_cpu, 64, 4096, periodic)
    else:
        lp, pix = gmm.LocalPixelization.make_rectangle(ny, nx, periodic_xcoord=periodic), orc.Pix.rectangle(ny, nx, periodic)
    xp = make_pointing(kind, n, ny, nx, rng)
    m = rng.standard_normal(3 * lp.npix).astype(F32)
    old = rng.standard_normal(n).astype(F32)
    xg = torch.from_numpy(xp).to(dev)
    mg = gmm.LocalMap(lp, torch.from_numpy(m).to(dev))
    ref, err = orc.map2tod(m.astype(np.float64), xp, pix, partial=cells, f64=True)
    assert err == 0
    for accum in (False, True):
        t = torch.from_numpy(old).to(dev)
        gmm.map2tod(t, mg, xg, None, partial_pixelization=cells, accum=accum)
        want = ref + old.astype(np.float64) * accum
        # |T| + |Q| + |U| of the four corners with weights that sum to 1 is below 3 max |m|.
        assert np.abs(t.cpu().numpy() - want).max() <= BAR * (3 * np.abs(m).max() + np.abs(old).max())
