"""The work that programs built on this library have it do, as timed cases.

A map-making program plans the pointing of each timestream (PointingPrePlan, PointingPlan) and
then applies map2tod and tod2map over and over: single calls on one timestream, the weighted
normal operator of an iterative solver over several, accumulation of many timestreams into a
DynamicMap, 16-bit timestreams and their encoding, and, where a plan does not pay, the plan-free
operators.

A case is a dict of plain values:
  op        'plan', 'map2tod', 'tod2map', 'step' (map2tod, then tod2map), 'normal', 'dynamic',
            'planfree_map2tod', 'planfree_tod2map' or 'encode16'
  scan      ndet detectors x nt samples on an ny x nx map: a triangle sweep of amplitude 'amp'
            (pixels) and period 'period' (samples) at angle 'phi', drifting across the sweep by
            'drift' pixels per sample; detectors spread over a disk of radius 'radius', detector
            angles turning by 'rate' per sample
  layout    'dense' (the whole map as one rectangle) or 'cells' (only the 64x64 cells touched)
  dtype     'f32', 'f16' or 'bf16': how the timestream is held
  response  per-detector gains; deferred: error flags left on the plan, as in a solver's loop;
  ntod      timestreams ('normal', 'dynamic'); feedback: order of the encoder's error feedback.
"""

import math

import numpy as np
import torch

import gpu_mm_amd as gmm
from gpu_mm_amd import mapmaker

_DEV = "cuda"
_TORCH16 = {"f16": torch.float16, "bf16": torch.bfloat16}
_HALF_MAX = {"f16": 32752.0, "bf16": float.fromhex("0x1.fep126")}
_CHUNK = 1 << 24           # samples handled at once by the 64-bit evaluation


def _case(op, ndet, nt, ny, nx, amp, period, drift, radius, rate, phi=0.0, periodic=False, layout="dense",
          dtype="f32", response=False, deferred=False, ntod=1, feedback=0, name=None):
    c = dict(op=op, ndet=ndet, nt=nt, ny=ny, nx=nx, amp=amp, period=period, drift=drift, radius=radius, rate=rate,
             phi=phi, periodic=periodic, layout=layout, dtype=dtype, response=response, deferred=deferred, ntod=ntod,
             feedback=feedback)
    if name is not None:
        c["name"] = name
    return c


# The three scans below are the library's own workloads: the 64 x 65536 raster on a 256 x 512 map,
# the 2048 x 262144 raster on a sparse 4096 x 8192 map, and 512 x 131072 scans crossing at 45
# degrees on a 1024 x 2048 map.
_SMALL = dict(ny=256, nx=512, amp=200.0, period=8192.0, drift=0.0025, radius=20.0, rate=0.001)
_RASTER = dict(ny=4096, nx=8192, amp=3000.0, period=40000.0, drift=0.01, radius=300.0, rate=2 * math.pi / 1.0e6)
_CROSS = dict(ny=1024, nx=2048, amp=300.0, period=8192.0, drift=0.0025, radius=20.0, rate=0.001)


def listed():
    return [
        # A short stretch of a few detectors with an odd sample count is planned: a test, a
        # calibration scan, a piece of a timestream. Launches and waits count.
        _case("plan", 7, 4099, **_SMALL, periodic=True, name="plan_small"),
        # A whole observation is planned; it is planned again whenever its plan is not kept.
        _case("plan", 2048, 262144, **_RASTER, name="plan_raster"),
        # The smallest operator calls: 8 detectors, both directions, error flags checked as by default.
        _case("step", 8, 4096, **_SMALL, name="step_small"),
        # An ordinary call of each direction, the whole map in one rectangle.
        _case("step", 64, 65536, **_SMALL, name="step_ordinary"),
        # The largest single timestream, on a map of only the touched cells: simulation ...
        _case("map2tod", 2048, 262144, **_RASTER, layout="cells", deferred=True, name="map2tod_raster"),
        # ... and map accumulation.
        _case("tod2map", 2048, 262144, **_RASTER, layout="cells", deferred=True, name="tod2map_raster"),
        # 16-bit timestreams with per-detector gains on a fast rotated scan that crosses the
        # periodic boundary; rows that are no multiple of a 32-sample line.
        _case("step", 768, 50004, ny=2048, nx=4096, amp=1500.0, period=8192.0, drift=0.0025, radius=20.0, rate=0.001,
              phi=0.6, periodic=True, layout="cells", dtype="f16", response=True, deferred=True,
              name="step_f16_fast"),
        # One application of A^T N^-1 A over four crossing scans, the step of a conjugate-gradient solve.
        _case("normal", 512, 131072, **_CROSS, ntod=4, deferred=True, name="normal_operator"),
        # Timestreams accumulated one after the other into a map that grows as they need it.
        _case("dynamic", 300, 16421, **_CROSS, ntod=3, name="dynamic_map"),
        # The plan-free operators, used where pointing changes at every call.
        _case("planfree_map2tod", 64, 65536, **_SMALL, name="planfree_map2tod"),
        _case("planfree_tod2map", 64, 65536, **_SMALL, name="planfree_tod2map"),
        # A timestream is put into 16 bits with the error feedback that map-making uses.
        _case("encode16", 512, 131072, **_CROSS, dtype="f16", feedback=2, name="encode_f16"),
    ]


# Samples (over all timestreams) of each op's drawn cases.
_DRAW_RANGE = {"plan": (2 ** 13, 2 ** 29), "map2tod": (2 ** 13, 2 ** 29), "tod2map": (2 ** 13, 2 ** 29),
               "step": (2 ** 13, 2 ** 27), "normal": (2 ** 16, 2 ** 28), "dynamic": (2 ** 14, 2 ** 24),
               "planfree_map2tod": (2 ** 13, 2 ** 22), "planfree_tod2map": (2 ** 13, 2 ** 22),
               "encode16": (2 ** 13, 2 ** 26)}


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(sorted(_DRAW_RANGE))
    lo, hi = _DRAW_RANGE[op]
    ntod = rng.randint(2, 5) if op in ("normal", "dynamic") else 1
    nsamp = _logint(rng, lo, hi)
    ndet = min(_logint(rng, 1, 2048), max(1, nsamp // (ntod * 512)))
    nt = max(256, min(nsamp // (ndet * ntod), 1 << 21))
    dtype = rng.choice(["f32", "f32", "f16", "bf16"]) if op in ("map2tod", "tod2map", "step") else "f32"
    if op == "encode16":
        dtype = rng.choice(["f16", "bf16"])
    if op == "normal" or (dtype != "f32" and op != "encode16"):
        nt = (nt + 3) // 4 * 4                   # these need whole groups of four samples
    side_lo = 128 if nsamp < 2 ** 22 else 512
    ny, nx = _logint(rng, side_lo, 4096), _logint(rng, side_lo, 8192)
    periodic = rng.random() < 0.3
    phi = rng.choice([0.0, 0.0, rng.uniform(0.0, math.pi)])
    side = min(ny, nx)
    radius = min(300.0, rng.uniform(0.02, 0.12) * side)
    half_drift = min(0.5 * rng.uniform(0.001, 0.01) * nt, 0.15 * side)
    room_y = 0.5 * (ny - 1) - 4.0 - radius - half_drift
    room_x = (nx if periodic else 0.5 * (nx - 2)) - 4.0 - radius - half_drift
    if op == "normal":                           # its timestreams cross at other angles: fits at each of them
        room = min(room_y, room_x)
    else:
        room = min(room_y / max(abs(math.sin(phi)), 1e-3), room_x / max(abs(math.cos(phi)), 1e-3))
    amp = rng.uniform(0.4, 0.98) * min(room, 3000.0)
    speed = math.exp(rng.uniform(math.log(0.03), math.log(0.8)))
    return _case(op, ndet, nt, ny, nx, amp=round(amp, 3), period=round(4.0 * amp / speed, 3),
                 drift=2.0 * half_drift / nt, radius=round(radius, 3), rate=rng.choice([0.0, 6.0e-6, 0.001]), phi=phi,
                 periodic=periodic, layout=rng.choice(["dense", "cells"]), dtype=dtype,
                 response=(op in ("map2tod", "tod2map", "step") and rng.random() < 0.25),
                 deferred=(op == "normal" or rng.random() < 0.5), ntod=ntod, feedback=rng.randint(0, 2))


# ------------------------------------------------------------------------------------------
# Inputs.

def _pointing(case, seed, i=0):
    """xpointing float32 (3, ndet, nt) of timestream i, computed in float64 and rounded once. The
    scan is the case's; the seed gives the order of the detectors and their angles."""
    ndet, nt = case["ndet"], case["nt"]
    scan_rng, rng = np.random.default_rng([ndet, nt, i]), np.random.default_rng([seed, i, 1])
    order = rng.permutation(ndet)
    r, a = case["radius"] * np.sqrt(scan_rng.random(ndet)[order]), 2 * np.pi * scan_rng.random(ndet)[order]
    theta = rng.uniform(0.0, np.pi, ndet)
    phi = case["phi"] + (math.pi / 4) * i if case["op"] == "normal" else case["phi"]
    sn, cs = math.sin(phi), math.cos(phi)
    yc = 0.5 * (case["ny"] - 1) + scan_rng.uniform(-1.0, 1.0)
    xc = 0.5 * (case["nx"] - 2) + scan_rng.uniform(-1.0, 1.0)
    t = torch.arange(nt, dtype=torch.float64, device=_DEV)
    w = t / case["period"] + float(scan_rng.random())
    u = case["amp"] * (1.0 - 4.0 * torch.abs(w - torch.floor(w) - 0.5))
    v = case["drift"] * (t - 0.5 * (nt - 1))
    xp = torch.empty((3, ndet, nt), dtype=torch.float32, device=_DEV)
    step = max(1, _CHUNK // nt)
    for row, base, ofs in ((0, yc + u * sn + v * cs, r * np.sin(a)), (1, xc + u * cs - v * sn, r * np.cos(a)),
                           (2, case["rate"] * t, theta)):
        o = torch.from_numpy(ofs).to(_DEV)
        for d in range(0, ndet, step):
            xp[row, d:d + step] = base[None, :] + o[d:d + step, None]
    return xp


def _generator(seed, i, what):
    g = torch.Generator(device=_DEV)
    g.manual_seed((seed * 64 + i) * 8 + what)
    return g


def _tod(case, seed, i=0):
    """White noise of unit variance over a slow common drift."""
    t = torch.randn((case["ndet"], case["nt"]), generator=_generator(seed, i, 2), device=_DEV)
    t += 2.0 * torch.sin(torch.arange(case["nt"], device=_DEV) * (6.0 / case["nt"]))
    return t


def _split16(case, tod):
    """A 16-bit timestream with one scale per detector, as it comes from storage."""
    scale = (tod.abs().amax(dim=1) / _HALF_MAX[case["dtype"]]).clamp(min=torch.finfo(torch.float32).tiny)
    return (tod / scale[:, None]).to(_TORCH16[case["dtype"]]).contiguous(), scale.contiguous()


def _gains(case, seed, i=0):
    """Per-detector gains (2, ndet) near 1, or inverse noise variances (ndet,) in [0.5, 2]."""
    rng = np.random.default_rng([seed, i, 3])
    shape = (case["ndet"],) if case["op"] == "normal" else (2, case["ndet"])
    return torch.from_numpy(rng.uniform(0.5, 2.0, shape).astype(np.float32)).to(_DEV)


def _cells(case, xps):
    """Flat indices of the 64x64 cells the pointings touch, in increasing order."""
    nyc, nxc = (case["ny"] + 63) // 64, (case["nx"] + 63) // 64
    hit = torch.zeros(nyc * nxc, dtype=torch.bool, device=_DEV)
    for xp in xps:
        for _, _, iy, ix, _, _ in _corners(case, xp):
            for j in range(2):
                for k in range(2):
                    col = torch.remainder(ix + k, case["nx"]) if case["periodic"] else ix + k
                    hit[((iy + j) >> 6) * nxc + (col >> 6)] = True
    return torch.nonzero(hit).reshape(-1).cpu()


def _sky(case, seed):
    """A map (3, padded ny, padded nx) of unit variance."""
    shape = (3, (case["ny"] + 63) // 64 * 64, (case["nx"] + 63) // 64 * 64)
    return torch.randn(shape, generator=_generator(seed, 0, 4), device=_DEV)


def _to_layout(case, dense, cells):
    """The dense map (3, Y, X) as the flat array of the case's local map."""
    if case["layout"] == "dense":
        return dense.reshape(-1).contiguous()
    _, y, x = dense.shape
    tiles = dense.reshape(3, y // 64, 64, x // 64, 64).permute(1, 3, 0, 2, 4).reshape(-1, 3, 64, 64)
    return tiles[cells.to(dense.device)].reshape(-1).contiguous()


def _pixelization(case, cells):
    if case["layout"] == "dense":
        return gmm.LocalPixelization.make_rectangle(case["ny"], case["nx"], periodic_xcoord=case["periodic"])
    nxc = (case["nx"] + 63) // 64
    return gmm.LocalPixelization.make_cells(case["ny"], case["nx"], [(int(c) // nxc, int(c) % nxc) for c in cells],
                                            periodic_xcoord=case["periodic"])


def _plan(case, xp):
    pre = gmm.PointingPrePlan(xp, case["ny"], case["nx"], periodic_xcoord=case["periodic"])
    return gmm.PointingPlan(pre, xp)


def prepare(case, seed):
    op = case["op"]
    s = dict(case=case)
    if op == "encode16":
        s["tod"] = _tod(case, seed)
        return s
    s["xp"] = [_pointing(case, seed, i) for i in range(case["ntod"])]
    if op == "plan":
        # Entries kept by the caller: as many as any such scan needs (its lines touch one to three cells).
        s["entries"] = torch.zeros(3 * ((case["ndet"] * case["nt"] + 31) // 32) + 64, dtype=torch.int64, device=_DEV)
        return s
    cells = _cells(case, s["xp"]) if case["layout"] == "cells" and op not in ("dynamic", "normal") else None
    if not op.startswith("planfree"):
        s["plan"] = [_plan(case, x) for x in s["xp"]]
    if op == "dynamic":
        s["tod"] = [_tod(case, seed, i) for i in range(case["ntod"])]
        return s
    if op == "normal":
        lp = gmm.LocalPixelization.make_rectangle(case["ny"], case["nx"], periodic_xcoord=case["periodic"])
        ninv = [_gains(case, seed, i) for i in range(case["ntod"])]
        s["wp"] = mapmaker.WeightedPointing(lp, s["plan"], s["xp"], ninv)
        s["map"] = _sky(case, seed).reshape(-1).contiguous()
        s["out"] = torch.zeros_like(s["map"])
        return s
    lp = _pixelization(case, cells)
    s["response"] = _gains(case, seed) if case["response"] else None
    s["scale"] = None
    if op in ("tod2map", "planfree_tod2map", "step"):
        s["tod"] = _tod(case, seed)
        if case["dtype"] != "f32":
            s["tod"], s["scale"] = _split16(case, s["tod"])
        s["acc"] = gmm.LocalMap(lp, torch.zeros(3 * lp.npix, dtype=torch.float32, device=_DEV))
    if op in ("map2tod", "planfree_map2tod", "step"):
        s["sky"] = gmm.LocalMap(lp, _to_layout(case, _sky(case, seed), cells))
        s["out"] = torch.empty((case["ndet"], case["nt"]), device=_DEV,
                               dtype=torch.float32 if case["dtype"] == "f32" else _TORCH16[case["dtype"]])
        if case["dtype"] != "f32" and s["scale"] is None:
            s["scale"] = _split16(case, _tod(case, seed))[1]
    return s


# ------------------------------------------------------------------------------------------
# One pass.

def _operators(s):
    case = s["case"]
    plan = s["plan"][0] if "plan" in s else None
    kw = {}
    if plan is not None:
        kw = dict(response=s["response"], tod_scale=s["scale"])
    out = []
    if "sky" in s:
        gmm.map2tod(s["out"], s["sky"], s["xp"][0], plan, **kw)
        out.append(s["out"])
    if "acc" in s:
        s["acc"].arr.zero_()
        gmm.tod2map(s["acc"], s["tod"], s["xp"][0], plan, **kw)
        out.append(s["acc"].arr)
    return out


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "encode16":
        t16, scale = gmm.encode_tod16(state["tod"], _TORCH16[case["dtype"]], error_feedback=case["feedback"])
        return [t16, scale]
    if op == "plan":
        xp = state["xp"][0]
        cumsum = torch.empty(gmm.PointingPrePlan.preplan_size, dtype=torch.uint32, device=_DEV)
        pre = gmm.PointingPrePlan(xp, case["ny"], case["nx"], buf=cumsum, periodic_xcoord=case["periodic"])
        plan = gmm.PointingPlan(pre, xp)
        # The plan's buffer begins with its sorted entries, 8 bytes each.
        state["entries"][:plan.plan_nmt].copy_(plan.buf[:8 * plan.plan_nmt].view(torch.int64))
        return [state["entries"], cumsum.view(torch.int32), int(plan.plan_nmt), int(plan.nmlines)]
    if op == "normal":
        return [state["wp"].apply_normal(state["map"], state["out"])]
    if op == "dynamic":
        dmap = gmm.DynamicMap(case["ny"], case["nx"], np.float32, periodic_xcoord=case["periodic"])
        for xp, plan, tod in zip(state["xp"], state["plan"], state["tod"]):
            gmm.tod2map(dmap, tod, xp, plan)
        m = dmap.finalize()
        return [m.arr, m.pixelization.cell_offsets_cpu]
    if case["deferred"]:
        with gmm.deferred_errflags():
            return _operators(state)
    return _operators(state)


# ------------------------------------------------------------------------------------------
# The bytes and operations a pass cannot do without.

def work(case):
    nsamp = case["ndet"] * case["nt"] * case["ntod"]
    op = case["op"]
    tsize = 4 if case["dtype"] == "f32" else 2
    if op == "encode16":
        return {"bytes": (4 + 2) * nsamp, "flops": 2 * nsamp}
    if op == "plan":
        # y and x once; an entry of 8 bytes for each line of 32 samples.
        return {"bytes": 8 * nsamp + 8 * ((nsamp + 31) // 32), "flops": 10 * nsamp}
    # Pixels inside the scan's outline, three components of 4 bytes.
    sweep = 2 * case["amp"] + 2 * case["radius"]
    across = case["drift"] * case["nt"] + 2 * case["radius"]
    npix = min(sweep * across * case["ntod"], case["ny"] * case["nx"])
    per_map = int(12 * npix)
    m2t = {"bytes": (12 + tsize) * nsamp + per_map, "flops": 30 * nsamp}
    t2m = {"bytes": (12 + tsize) * nsamp + 2 * per_map, "flops": 30 * nsamp}
    if op in ("map2tod", "planfree_map2tod"):
        return m2t
    if op in ("step", "normal"):
        return {k: m2t[k] + t2m[k] for k in m2t}
    return t2m


# ------------------------------------------------------------------------------------------
# The same outputs in 64 bits, in plain torch.

def _corners(case, xp):
    """Chunks (first, last, iy0, ix0, dy, dx) over the flat samples of xp."""
    flat = xp.reshape(3, -1)
    n, ny, nx = flat.shape[1], case["ny"], case["nx"]
    for a in range(0, n, _CHUNK):
        b = min(n, a + _CHUNK)
        y, x = flat[0, a:b].double(), flat[1, a:b].double()
        iy = y.floor().long().clamp_(0, ny - 2)
        if case["periodic"]:
            x = torch.where(x < 0, x + nx, x)
            x = torch.where(x > nx, x - nx, x)
            fx = x.floor()
            ix = fx.long()
            dx = x - fx
            ix = torch.where(ix >= nx, torch.zeros_like(ix), ix)
        else:
            ix = x.floor().long().clamp_(0, nx - 2)
            dx = x - ix
        yield a, b, iy, ix, y - iy, dx


def _weights(case, iy, ix, dy, dx, stride):
    """(pixel index, weight) of the four corners."""
    for j in range(2):
        for k in range(2):
            col = torch.remainder(ix + k, case["nx"]) if case["periodic"] else ix + k
            yield (iy + j) * stride + col, (dy if j else 1 - dy) * (dx if k else 1 - dx)


def _rows(case, gain, a, b):
    """Per-detector values 'gain' (float64) at the flat samples a..b-1."""
    return gain[torch.arange(a, b, device=gain.device) // case["nt"]]


def _exact_map2tod(case, sky, xp, gt=None, gp=None):
    out = torch.empty(case["ndet"] * case["nt"], dtype=torch.float64, device=_DEV)
    flat, stride = sky.double().reshape(3, -1), sky.shape[2]
    alpha = xp[2].reshape(-1)
    for a, b, iy, ix, dy, dx in _corners(case, xp):
        v = [0.0, 0.0, 0.0]
        for idx, w in _weights(case, iy, ix, dy, dx, stride):
            for p in range(3):
                v[p] = v[p] + w * flat[p][idx]
        ang = 2.0 * alpha[a:b].double()
        pol = v[1] * torch.cos(ang) + v[2] * torch.sin(ang)
        out[a:b] = v[0] + pol if gt is None else _rows(case, gt, a, b) * v[0] + _rows(case, gp, a, b) * pol
    return out.reshape(case["ndet"], case["nt"])


def _exact_tod2map(case, tod, xp, gt=None, gp=None):
    """A^T tod as a dense padded map (3, Y, X); tod float64 values by flat slice via tod(a, b)."""
    y, x = (case["ny"] + 63) // 64 * 64, (case["nx"] + 63) // 64 * 64
    acc = torch.zeros((3, y * x), dtype=torch.float64, device=_DEV)
    alpha = xp[2].reshape(-1)
    for a, b, iy, ix, dy, dx in _corners(case, xp):
        t = tod(a, b)
        ang = 2.0 * alpha[a:b].double()
        tt = t if gt is None else t * _rows(case, gt, a, b)
        tp = t if gp is None else t * _rows(case, gp, a, b)
        vals = (tt, tp * torch.cos(ang), tp * torch.sin(ang))
        for idx, w in _weights(case, iy, ix, dy, dx, x):
            for p in range(3):
                acc[p].index_add_(0, idx, w * vals[p])
    return acc.reshape(3, y, x)


def exact(case, seed):
    op = case["op"]
    if op == "plan":
        return None                      # whole numbers only
    if op == "encode16":
        tod = _tod(case, seed).double()
        scale = (tod.abs().amax(dim=1) / _HALF_MAX[case["dtype"]]).clamp(min=torch.finfo(torch.float32).tiny)
        # With error feedback each value holds its predecessors' rounding too.
        return [None if case["feedback"] else tod / scale[:, None], scale]
    xps = [_pointing(case, seed, i) for i in range(case["ntod"])]
    if op == "normal":
        sky = _sky(case, seed)
        total = 0.0
        for i, xp in enumerate(xps):
            w = _gains(case, seed, i).double()
            t = (_exact_map2tod(case, sky, xp) * w[:, None]).reshape(-1)
            total = total + _exact_tod2map(case, lambda a, b: t[a:b], xp)
        return [total.reshape(-1)]
    if op == "dynamic":
        # Cells in the order they came: by timestream, inside one by increasing index.
        order, total = [], 0.0
        for i, xp in enumerate(xps):
            order += [int(c) for c in _cells(case, [xp]) if int(c) not in order]
            t = _tod(case, seed, i).reshape(-1)
            total = total + _exact_tod2map(case, lambda a, b: t[a:b].double(), xp)
        arr = _to_layout(dict(case, layout="cells"), total, torch.tensor(order, dtype=torch.long))
        return [arr, None]
    cells = _cells(case, xps) if case["layout"] == "cells" else None
    gt = gp = None
    if case["response"]:
        gt, gp = _gains(case, seed).double()
    out = []
    tod, scale = None, None
    if op in ("tod2map", "planfree_tod2map", "step") or case["dtype"] != "f32":
        tod = _tod(case, seed)
        if case["dtype"] != "f32":
            tod, scale = _split16(case, tod)
            scale = scale.double()
    if op in ("map2tod", "planfree_map2tod", "step"):
        t = _exact_map2tod(case, _sky(case, seed), xps[0], gt, gp)
        out.append(t if scale is None else t / scale[:, None])
    if op in ("tod2map", "planfree_tod2map", "step"):
        flat = tod.reshape(-1)

        def values(a, b):
            v = flat[a:b].double()
            return v if scale is None else v * _rows(case, scale, a, b)

        out.append(_to_layout(case, _exact_tod2map(case, values, xps[0], gt, gp), cells))
    return out
