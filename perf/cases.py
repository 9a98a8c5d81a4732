"""The work that programs built on this package have it do, as timed cases.

Every case goes through the public entry points a user's program calls: a
``Solver`` stepped through the driver loop (``advance`` / ``run``) and read out
(``get_state``), a ``Batch`` of runs advanced together, or the drop-in operators
(``ddx`` ... ``filtz``) on host arrays.  Sizes are those of the package's own
workloads (the 64 x 64 x 128 acoustic run, the 256^3 sunspot run, the batched
population's 48 to 192 by 96 to 256) and generic ones between and beside them,
odd and ragged ones among them.  A pass of a run is one stretch of the time loop
between two read-outs of the state; the run goes on from where the last pass
left it, as the driver loop does.

``listed`` gives the cases, ``draw`` one more of the same ranges, ``prepare`` what
a program holds before the call, ``run`` one pass, ``work`` what a pass cannot do
without, and ``exact`` the same results from a plain 64-bit torch statement of
the scheme (the class ``Plain``), which shares no code with the package.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from sparc2_amd.batch import Batch
from sparc2_amd.config import RunConfig
from sparc2_amd.forcing import ForcingSeries
from sparc2_amd.solver import Solver

FIELDS = ("rho", "vx", "vy", "vz", "p", "bx", "by", "bz")
RSUN, PI = 69598946770.0, 3.14159265358979


# --------------------------------------------------------------------- cases
def _run(name, nx, ny, nz, steps, magnetic=0, open_sides=False, precision="fp64", taps=11,
         t_xy=30.0, t_z=10.0, damping=False, cube=False, checked=False, psi=False):
    return {"name": name, "kind": "run", "nx": nx, "ny": ny, "nz": nz, "steps": steps,
            "magnetic": magnetic, "open_sides": open_sides, "precision": precision, "taps": taps,
            "t_xy": t_xy, "t_z": t_z, "damping": damping, "cube": cube, "checked": checked, "psi": psi}


def listed():
    return [
        # the smallest run of the package's range, watched step by step as the
        # reference's driver prints it (norm and minima after every step): latency
        _run("quiet-48-watched", 48, 48, 96, 10, checked=True),
        # the plain acoustic run; the state is wanted every 45 s of solar time,
        # the cadence of the instrument the runs are compared with
        _run("quiet-64", 64, 64, 128, 45),
        # a region with its own horizontal structure, open sides, odd sizes
        # (3-D backgrounds, CPML on all six faces), stopped for a restart file
        _run("thermal-odd-open", 107, 75, 117, 40, magnetic=1, open_sides=True, psi=True),
        # a run under FFT damping of the velocities
        _run("quiet-damped", 128, 96, 100, 20, damping=True),
        # a run driven by an observed velocity cube instead of the pulse
        _run("quiet-cube-driven", 160, 160, 128, 30, cube=True),
        # the large quiet runs, in both precisions; the single-precision one,
        # taken for long series, is read out every two minutes of solar time
        _run("quiet-large", 384, 384, 160, 45),
        _run("quiet-large-fp32", 384, 384, 160, 120, precision="fp32"),
        # sunspot runs: a small one with odd sizes and the short filter at every
        # few steps, the full one, and a single-precision one
        _run("sunspot-odd", 63, 79, 101, 40, magnetic=2, open_sides=True, taps=7, t_xy=2.0, t_z=1.0),
        _run("sunspot-256", 256, 256, 256, 45, magnetic=2, open_sides=True),
        _run("sunspot-192-fp32", 192, 192, 160, 60, magnetic=2, open_sides=True, precision="fp32"),
        # a parameter study: independent sunspot runs of mixed sizes, advanced together
        {"name": "study-fp32", "kind": "batch", "precision": "fp32", "steps": 25,
         "grids": "48x64x101 96x48x120 64x128x160 96x96x133 128x96x96 64x64x200"},
        # the operators on host arrays, as an analysis or set-up program uses them
        {"name": "operators", "kind": "operators", "nx": 150, "ny": 130, "nz": 121, "periodic": True},
    ]


def _size(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi] that open sides accept (the
    last tile of a row or column holds at least six points)."""
    while True:
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        if n % 16 == 0 or n % 16 >= 6:
            return n


def draw(rng):
    what = rng.choice(("quiet", "quiet", "sunspot", "sunspot", "thermal", "batch", "operators"))
    precision = rng.choice(("fp64", "fp32"))
    if what == "operators":
        return {"kind": "operators", "nx": _size(rng, 48, 192), "ny": _size(rng, 48, 192),
                "nz": rng.randint(96, 160), "periodic": rng.random() < 0.5}
    if what == "batch":
        grids = " ".join("%dx%dx%d" % (_size(rng, 48, 128), _size(rng, 48, 128), rng.randint(96, 160))
                         for _ in range(rng.randint(3, 6)))
        return {"kind": "batch", "precision": precision, "steps": rng.randint(10, 25), "grids": grids}
    hi = 384 if what == "quiet" else 256
    while True:
        nx, ny, nz = _size(rng, 48, hi), _size(rng, 48, hi), rng.randint(96, 256)
        if nx * ny * nz <= (12 if what == "quiet" else 8) * 10 ** 6:
            break
    # the damping grows with the wavenumber and is used up to moderate ones
    # (beyond, its rate times the time step leaves the scheme's stable range)
    damping = what == "quiet" and max(nx, ny) <= 112 and rng.random() < 0.5
    case = _run("", nx, ny, nz, rng.randint(10, 45), magnetic={"quiet": 0, "thermal": 1, "sunspot": 2}[what],
                open_sides=what != "quiet", precision=precision, taps=rng.choice((11, 11, 7)),
                t_xy=rng.choice((30.0, 2.0)), t_z=rng.choice((10.0, 1.0)),
                damping=damping, cube=what == "quiet" and rng.random() < 0.2,
                checked=rng.random() < 0.2, psi=rng.random() < 0.3)
    del case["name"]
    return case


def _members(case):
    """The runs of a case: itself, or each run of a batch."""
    if case["kind"] != "batch":
        return [case]
    out = []
    for g in case["grids"].split():
        nx, ny, nz = (int(v) for v in g.split("x"))
        out.append(_run(g, nx, ny, nz, case["steps"], magnetic=2, open_sides=True, precision=case["precision"]))
    return out


# -------------------------------------------------------------------- inputs
def _settings(case, seed):
    """The control-file values of a run; the seed places the pulse."""
    rng = random.Random(seed)
    mhd = case["magnetic"] == 2
    width = 100.0e8 if mhd else 50.0e8
    zbot, ztop = (-20.0, 1.0) if mhd else (-10.0, 0.5)
    # the reference's CFL estimate over the column: 117 km/s (sound and capped
    # Alfven speed) or 43 km/s at the bottom, with a margin
    dz = (ztop - zbot) * 1e8 / (case["nz"] - 1)
    dt = math.floor(0.7 * dz / (1.18e7 if mhd else 4.4e6) / 0.05) * 0.05
    n = 10
    return {"width": width, "zbot": zbot, "ztop": ztop, "dt": dt,
            "npml": (n,) * 6 if case["open_sides"] else (0, 0, 0, 0, n, n),
            "pml": (9.2103, 2.0, 8.0, 0.1), "px": width * rng.uniform(0.3, 0.7), "py": width * rng.uniform(0.3, 0.7),
            "pz": -0.15e8, "sr": 1.0e8 * width / 50.0e8, "sz": 1.0e8, "amp": rng.uniform(50.0, 150.0),
            "t0": 1000.0 / 3.0, "t1": 450.0, "st": 150.0, "cad": 60.0, "depth": -0.15e8, "sigma": 0.1e8,
            "maxva": 1.0e7}


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _sky(case, s, seed):
    """The background file of a run (cgs, the reference's arrays): a polytrope
    under an isothermal layer, with 5 % of horizontal structure in a thermal run
    and a flux tube in a sunspot run.  Torch arrays (nz, ny, nx)."""
    rng, dev = random.Random(seed + 1), _device()
    f8 = dict(dtype=torch.float64, device=dev)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    z = torch.linspace(s["zbot"], s["ztop"], nz, **f8)
    gamma, grav, m, rho_s, c_s = 5.0 / 3.0, 2.74e4, 1.5, 2.8e-7, 7.0e5
    zc = z * 1e8
    d0, h, p_s = c_s * c_s * (m + 1) / (gamma * grav), c_s * c_s / (gamma * grav), c_s * c_s * rho_s / gamma
    ratio = torch.where(zc <= 0, (d0 - zc) / d0, torch.ones_like(zc))
    iso = torch.where(zc <= 0, torch.ones_like(zc), torch.exp(-zc / h))
    col = lambda v: v[:, None, None]  # noqa: E731
    rho, p, c = col(rho_s * ratio ** m * iso), col(p_s * ratio ** (m + 1) * iso), col(c_s * ratio.sqrt())
    n = (nx, ny) if not case["open_sides"] else (nx - 1, ny - 1)
    x = torch.arange(nx, **f8)[None, None, :] / n[0] * s["width"]
    y = torch.arange(ny, **f8)[None, :, None] / n[1] * s["width"]
    full = torch.ones((nz, ny, nx), **f8)
    out = {}
    if case["magnetic"] == 2:
        b0, r0, hr = rng.uniform(1500.0, 3000.0), 4.0e8, 1.0e8
        xc, yc = s["width"] * rng.uniform(0.45, 0.55), s["width"] * rng.uniform(0.45, 0.55)
        ez = col(torch.exp(zc / hr))
        r2 = r0 * r0 * (1 + ez) / 2
        grow = 0.5 * (ez / hr) / (1 + ez)
        bz = b0 * (r0 * r0 / r2) * torch.exp(-((x - xc) ** 2 + (y - yc) ** 2) / r2)
        bx, by = (x - xc) * grow * bz, (y - yc) * grow * bz
        gas = torch.maximum(p - (bx * bx + by * by + bz * bz) / (8 * math.pi), 0.5 * p)
        rho, p, c = rho * (gas / p), gas, c * full
        out = {"bx0": bx, "by0": by, "bz0": bz}
    else:
        if case["magnetic"] == 1:
            a, b = rng.uniform(0, 2 * math.pi), rng.uniform(0, 2 * math.pi)
            full = full * (1 + 0.05 * torch.sin(2 * math.pi * x / s["width"] + a) * torch.cos(2 * math.pi * y / s["width"] + b))
        rho, p, c = rho * full, p * full, c * torch.ones_like(full)
    out.update(rho0=rho, pre0=p, cs0=c, zaxis=z, grav=torch.full((nz,), grav, **f8))
    return out


def _waves(case, raw, seed):
    """A wave field in progress: a few smooth modes per field, about 1e-5 of the
    local background, fading towards the top and bottom."""
    rng, dev = random.Random(seed + 2), _device()
    f8 = dict(dtype=torch.float64, device=dev)
    shape = tuple(raw["rho0"].shape)
    r0, c0 = raw["rho0"][0, 0, 0], raw["cs0"][0, 0, 0]
    rho, c, p = raw["rho0"] / r0, raw["cs0"] / c0, raw["pre0"] / (r0 * c0 * c0)
    scale = [rho, c, c, c, p] + ([rho.sqrt() * c] * 3 if case["magnetic"] == 2 else [])
    fade = torch.sin(math.pi * (torch.arange(shape[0], **f8) + 0.5) / shape[0]) ** 2
    out = torch.empty((len(scale),) + shape, **f8)
    for f, s in enumerate(scale):
        total = torch.zeros(shape, **f8)
        for _ in range(3):
            parts = []
            for n in shape:
                u = torch.arange(n, **f8) / n
                parts.append(torch.cos(2 * math.pi * (rng.randint(1, max(1, n // 12)) * u + rng.random())))
            total += rng.uniform(-1, 1) * (parts[0] * fade)[:, None, None] * parts[1][None, :, None] * parts[2][None, None, :]
        out[f] = 1e-5 * total * s
    return out


MAPS = 64


def _cube(case, seed):
    """Velocity maps at the driver's cadence, (maps, ny, nx) in units of the
    run's driving amplitude: smooth modes that turn slowly."""
    rng = random.Random(seed + 3)
    u, v, t = np.arange(case["nx"]) / case["nx"], np.arange(case["ny"]) / case["ny"], np.arange(MAPS)
    out = np.zeros((MAPS, case["ny"], case["nx"]))
    for _ in range(6):
        kx, ky, w, a, b = rng.randint(1, 8), rng.randint(1, 8), rng.uniform(0.2, 1.5), rng.random(), rng.random()
        out += (np.cos(2 * np.pi * ky * v + b + w * t[:, None])[:, :, None]) * np.cos(2 * np.pi * (kx * u + a))
    return out


def _config(case, s):
    sides = case["open_sides"]
    return RunConfig(
        nx=case["nx"], ny=case["ny"], nz=case["nz"], xlength=s["width"], ylength=s["width"], timestep=s["dt"],
        solartime=0.5, magnetic=case["magnetic"], periodic=not sides, use_pml=True, use_hpml=sides,
        npml=s["npml"], pmlc=(s["pml"],) * 6, damping=case["damping"], filter_mode_xy=1 if case["taps"] == 11 else 2,
        filter_mode_z=1 if case["taps"] == 11 else 2, t_xy=case["t_xy"], t_z=case["t_z"], pulse=not case["cube"],
        pulse_dir=3, pulse_t0=s["t0"], pulse_t1=s["t1"], pulse_st=s["st"], pulse_px=s["px"], pulse_py=s["py"],
        pulse_pz=s["pz"], pulse_sr=s["sr"], pulse_sz=s["sz"], pulse_amp=s["amp"], cadforcing=s["cad"],
        randomexcitedepth=s["depth"], randomexcitesigma=s["sigma"], randomexciteampl=s["amp"], maxva=s["maxva"],
        precision=case["precision"])


def _solver(case, seed):
    s = _settings(case, seed)
    raw = _sky(case, s, seed)
    solver = Solver(_config(case, s), {k: v.cpu().numpy() for k, v in raw.items()})
    solver.put_state(_waves(case, raw, seed).cpu().numpy())
    return solver


def _grid_of(case):
    """The run whose grid the operators act on."""
    return _run("", case["nx"], case["ny"], case["nz"], 1, open_sides=not case["periodic"])


def _field(case, seed):
    rng = np.random.default_rng(seed)
    shape = (case["nz"], case["ny"], case["nx"])
    z, y, x = (np.arange(n).reshape([-1 if q == a else 1 for q in range(3)]) / n for a, n in enumerate(shape))
    k = rng.integers(1, 9, size=3)
    return np.sin(2 * np.pi * (k[0] * x + k[1] * y) + 3.0 * k[2] * z) + 0.01 * rng.standard_normal(shape)


def prepare(case, seed):
    if case["kind"] == "operators":
        return {"kind": "operators", "solver": _solver(_grid_of(case), seed), "field": _field(case, seed),
                "bc": 5 if case["periodic"] else 1}
    if case["kind"] == "batch":
        solvers = [_solver(m, seed + 100 * q) for q, m in enumerate(_members(case))]
        return {"kind": "batch", "batch": Batch(solvers), "case": case}
    out = {"kind": "run", "solver": _solver(case, seed), "case": case, "time": 0}
    if case["cube"]:
        out["cube"] = _cube(case, seed)
        out["solver"].use_forcing(ForcingSeries(out["solver"].st, out["cube"]))
    return out


# ----------------------------------------------------------------- one pass
def _fields(case, state):
    return {FIELDS[f]: _kept(case, v) for f, v in enumerate(state)}


def _kept(case, v):
    # a single-precision run is looked at in single precision
    return torch.from_numpy(v).to(torch.float32) if case["precision"] == "fp32" else v


def run(state):
    if state["kind"] == "operators":
        s, f, bc = state["solver"], state["field"], state["bc"]
        return {"ddx": s.ddx(f, bc), "ddy": s.ddy(f, bc), "ddz": s.ddz(f, 1),
                "filtx": s.filtx(f), "filty": s.filty(f), "filtz": s.filtz(f)}
    case = state["case"]
    if state["kind"] == "batch":
        failed = state["batch"].advance(case["steps"])
        if failed:
            raise next(iter(failed.values()))
        return [_fields(case, s.get_state()) for s in state["batch"].solvers]
    s, t, n = state["solver"], state["time"], case["steps"]
    if case["cube"] and (t + n) * s.cfg.timestep > (MAPS - 6) * s.cfg.cadforcing:
        # a long driven run plays its maps again from the start before they end
        s.use_forcing(ForcingSeries(s.st, state["cube"]))
        t = 0
    out = {}
    if case["checked"]:
        out["history"] = s.run(t, t + n - 1)
    else:
        s.advance(t, t + n - 1)
    state["time"] = t + n
    if case["psi"]:
        a, psi = s.get_state(with_psi=True)
        out["psi"] = {str(f): _kept(case, v) for f, v in psi.items()}
    else:
        a = s.get_state()
    out.update(_fields(case, a))
    return out


# --------------------------------------------------------------------- work
def work(case):
    if case["kind"] == "operators":
        n = case["nx"] * case["ny"] * case["nz"]
        # six operators: each reads the field and writes its result (an
        # 11-point row is 10 multiply-adds with a scale)
        return {"bytes": 6.0 * 2 * 8 * n, "flops": 6.0 * 21 * n}
    total_b = total_f = 0.0
    for m in _members(case):
        n = float(m["nx"] * m["ny"] * m["nz"])
        w = 4.0 if m["precision"] == "fp32" else 8.0
        mhd = m["magnetic"] == 2
        nv, npsi, nderiv = (8, 6, 18) if mhd else (5, 2, 6)
        # 3-D backgrounds read in a stage; profiles along z in the periodic quiet runs
        nbg = 16 if mhd else (5 if m["magnetic"] or m["open_sides"] else 0)
        s = _settings(m, 0)
        face = sum(p / d for p, d in zip(s["npml"], (m["nx"], m["nx"], m["ny"], m["ny"], m["nz"], m["nz"])))
        # a stage reads the stage value, the base and the backgrounds and writes
        # the next stage value; the CPML layers stream their psi the same way
        stage = w * n * (3 * nv + nbg + 3 * npsi * face)
        step = 5 * stage + (2 * 2 * nv * n if w == 4 else 0.0)  # FP32: the compensation, 2 bytes
        for t in (m["t_xy"], m["t_z"]):
            step += 2 * w * nv * n / max(1, math.floor(max(t, s["dt"]) / s["dt"] + 1e-5))
        if m["damping"]:
            step += 5 * 3 * 2 * w * n
        total_b += m["steps"] * step + 8 * nv * n  # and the state handed back in FP64
        total_f += m["steps"] * 5 * n * (15 * nderiv + (130 if mhd else 40))
    return {"bytes": total_b, "flops": total_f}


# -------------------------------------------------------------------- exact
# Coefficients of the scheme: the right half of the centred 11-point row, the
# five one-sided rows, and the 11- and 7-point filters.
CENTRE = (0.872756993962, -0.286511173973, 0.090320001280, -0.020779405824, 0.002484594688)
EDGE = (
    (-2.391602219538, 5.832490322294, -7.650218001182 + 1e-12, 7.907810563576, -5.922599052629, 3.071037015445,
     -1.014956769726, 0.170022256519, 0.002819958377, -0.004791009708, -0.000013063429),
    (-0.180022054228, -1.237550583044, 2.484731692990, -1.810320814061, 1.112990048440, -0.481086916514,
     0.126598690230, -0.015510730165, 0.000024609059 - 0.000003, 0.000156447571 - 1e-12, -0.000007390277),
    (0.057982271137, -0.536135360383, -0.264089548967 + 2e-12, 0.917445877606 - 2e-12, -0.169688364841,
     -0.029716326170, 0.029681617641, -0.005222483773, -0.000118806260, -0.000118806260, -0.000020069730),
    (-0.013277273810, 0.115976072920, -0.617479187931, -0.274113948206 + 2e-12, 1.086208764655 - 2e-12,
     -0.402951626982, 0.131066986242, -0.028154858354, 0.002596328316, 0.000128743150, 0.0),
    (0.016756572303, -0.117478455239, 0.411034935097, -1.130286765151, 0.341435872100 - 1e-12, 0.556396830543,
     -0.082525734207, 0.003565834658, 0.001173034777, -0.000071772671 + 6.4e-11, -0.000000352273))
TAPS = {5: (0.7539062500, 0.205078125, -0.1171875, 0.043945312500, -0.009765625, 0.0009765625),
        3: (0.3125, -0.234375, 0.09375, -0.015625)}
Z, Y, X = 0, 1, 2


def _slice(f, axis, lo, n):
    return f.narrow(axis, lo, n)


def _padded(f, axis, g, wrapped):
    if wrapped:
        n = f.shape[axis]
        return torch.cat([_slice(f, axis, n - g, g), f, _slice(f, axis, 0, g)], axis)
    shape = list(f.shape)
    shape[axis] = g
    zero = f.new_zeros(shape)
    return torch.cat([zero, f, zero], axis)


def _along(v, axis):
    return v.reshape([-1 if q == axis else 1 for q in range(3)])


def derivative(f, axis, metric, wrapped=False):
    """d/dx, d/dy or d/dz of the scheme: centred rows; on a side that does not
    wrap the one-sided rows, except at the bottom in z, where the centred row
    reads zeros below the grid.  metric: a number, or one for each plane."""
    n = f.shape[axis]
    g = _padded(f, axis, 5, wrapped)
    out = torch.zeros_like(f)
    for m, c in enumerate(CENTRE, 1):
        out += c * (_slice(g, axis, 5 + m, n) - _slice(g, axis, 5 - m, n))
    if not wrapped:
        for r, row in enumerate(EDGE):
            for side in ((1,) if axis == Z else (0, 1)):
                at = n - 1 - r if side else r
                total = sum(b * _slice(f, axis, n - 1 - m if side else m, 1) for m, b in enumerate(row))
                _slice(out, axis, at, 1).copy_(-total if side else total)
    return out * metric


def filtered(f, axis, g, wrapped, strength=None):
    """The filter operator along an axis (strength None), or FILTER_VARS's pass:
    the edges smoothed first, and the short filter taken off with its strength."""
    n = f.shape[axis]
    if strength is not None and not wrapped:
        # each smoothed edge value is the mean of its unsmoothed neighbours
        s = f.clone()
        for lo, count in ((1, g - 1), (n - g, g - 1)):
            _slice(s, axis, lo, count).copy_((_slice(f, axis, lo - 1, count) + _slice(f, axis, lo + 1, count)) / 2)
        f = s
    pad = _padded(f, axis, g, wrapped)
    out = TAPS[g][0] * f
    for m in range(1, g + 1):
        out += TAPS[g][m] * (_slice(pad, axis, g + m, n) + _slice(pad, axis, g - m, n))
    if not wrapped:
        for lo in (0, n - g):
            edge = _slice(f, axis, lo, g)
            _slice(out, axis, lo, g).copy_(edge if axis == Z or g == 5 else torch.zeros_like(edge))
    return out if strength is None or g == 5 else f - strength * out


class Plain:
    """One run in plain 64-bit torch: set-up, right-hand sides, CPML, the
    five-stage Runge-Kutta step, filters, damping and source."""

    def __init__(self, case, seed):
        s = self.s = _settings(case, seed)
        raw = _sky(case, s, seed)
        self.case, self.mhd, self.wrapped = case, case["magnetic"] == 2, not case["open_sides"]
        nx, ny, nz = self.n = case["nx"], case["ny"], case["nz"]
        col = lambda v: v[:, None, None]  # noqa: E731
        rho0, p0, cs, grav = raw["rho0"], raw["pre0"], raw["cs0"], raw["grav"]
        self.dimc, self.dimrho = float(cs[0, 0, 0]), float(rho0[0, 0, 0])
        dimb = (4.0 * PI * self.dimc ** 2 * self.dimrho) ** 0.5
        z = self.z = 1.0 + raw["zaxis"] * 1e8 / RSUN
        g, cq = grav * RSUN / self.dimc ** 2, cs[:, 0, 0] / self.dimc
        p0, rho0, c2 = p0 / (self.dimrho * self.dimc ** 2), rho0 / self.dimrho, (cs / self.dimc) ** 2
        self.rho0, self.p0, self.c2 = rho0, p0, c2
        # metric: the plane spacing as the scheme's own rows see it
        cells = (nx, ny) if self.wrapped else (nx - 1, ny - 1)
        self.sx, self.sy = RSUN / s["width"] * cells[0], RSUN / s["width"] * cells[1]
        zz = z.cpu().numpy()
        spacing = np.empty(nz)
        for k in range(nz):
            if k < 5 or k >= nz - 5:
                row, line, sign = (EDGE[k], zz, 1) if k < 5 else (EDGE[nz - 1 - k], zz[::-1], -1)
                spacing[k] = sign * sum(b * line[m] for m, b in enumerate(row))
            else:
                spacing[k] = sum(c * (zz[k + m] - zz[k - m]) for m, c in enumerate(CENTRE, 1))
        self.sz = col(torch.from_numpy(1.0 / spacing).to(z.device))
        self.dt = s["dt"] * self.dimc / RSUN
        weights = (1.0, 0.5, 0.1665579725791151184, 0.03950410250586729987, 0.007810706393337838236)
        b5 = weights[1]
        b4 = weights[2] / b5
        b3 = weights[3] / (b5 * b4)
        b2 = weights[4] / (b5 * b4 * b3)
        self.weights = [w * self.dt for w in (b2, b3, b4, b5)]
        if self.mhd:
            self.b0 = [raw[k] / dimb for k in ("bx0", "by0", "bz0")]
            self._limit(dimb, cq)
            bx, by, bz = self.b0
            self.curl0 = (self.ddy(bz) - self.ddz(by), self.ddz(bx) - self.ddx(bz), self.ddx(by) - self.ddy(bx))
        # background gradients, held convectively stable
        grz, gpz = self.ddz(rho0), self.ddz(p0)
        held = -rho0 * col(g)
        near = col((z > float(np.float32(0.9998))) & (z < 1.0))
        rest = col((z <= float(np.float32(0.9998))) | (z >= float(np.float32(1.0001))))
        gpz = torch.where(near, torch.maximum(c2 * grz + 1e-4 * RSUN / (self.dimrho * self.dimc ** 2), held),
                          torch.where(rest, torch.maximum(c2 * grz, held), gpz))
        self.grad_rho, self.grad_p = [None, None, grz], [None, None, gpz]
        if self.mhd:
            self.grad_rho[:2], self.grad_p[:2] = [self.ddx(rho0), self.ddy(rho0)], [self.ddx(p0), self.ddy(p0)]
        self.g, self.sponge = g, torch.zeros_like(rho0)
        self._layers()
        self._source(seed)
        self.u = list(_waves(case, raw, seed))

    def ddx(self, f):
        return derivative(f, X, self.sx, self.wrapped)

    def ddy(self, f):
        return derivative(f, Y, self.sy, self.wrapped)

    def ddz(self, f):
        return derivative(f, Z, self.sz)

    def _limit(self, dimb, cq):
        """The Alfven limiter: the largest value of a decimal search that keeps
        the limited Alfven speed under its cap."""
        b2 = sum(b * b for b in self.b0)
        ratio = b2 / (self.rho0 * (cq * cq)[:, None, None])
        temp, step = -1e9, 1e9
        while step > 1e-5 and temp < 1e10 - 1.1:
            va = 0.0
            while va < self.s["maxva"] and temp < 1e10:
                temp += step
                v = torch.sqrt(dimb * dimb * temp / (temp + ratio) * b2 / (4 * PI * self.dimrho * self.rho0))
                va = float(torch.where(torch.isnan(v), -torch.inf, v).max())
            temp -= step
            step /= 10.0
        self.red = temp / (temp + ratio)

    def _layers(self):
        """CPML coefficients of each face; the z layers scale gradients and gravity."""
        s, z = self.s, self.z
        speed = self.c2 + (self.red * sum(b * b for b in self.b0) / self.rho0 if self.mhd else 0.0)
        speed = torch.sqrt(speed)
        rc, power, kmax, sponge = s["pml"]
        f0 = PI * 0.005 * RSUN / self.dimc
        nx, ny, nz = self.n
        cells = (nx, ny) if self.wrapped else (nx - 1, ny - 1)
        axes = {X: torch.arange(nx, dtype=z.dtype, device=z.device) / cells[0],
                Y: torch.arange(ny, dtype=z.dtype, device=z.device) / cells[1], Z: z}
        self.layers, self.damp_xy = [], {}
        for face in (4, 5, 0, 1, 2, 3):
            n = s["npml"][face]
            if not n:
                continue
            axis, top = {0: X, 1: Y, 2: Z}[face // 2], face % 2
            x = axes[axis]
            lo = x.shape[0] - n if top else 0
            part = x[lo:lo + n]
            inner, outer = (part[0], part[-1]) if top else (part[-1], part[0])
            length = (outer - inner).abs()
            depth = (part - inner).abs() / length
            alpha = _along(f0 * (outer - part).abs() / length, axis)
            grade = _along(depth ** power, axis)
            edge = _slice(speed, axis, lo if top else n - 1, 1)
            damp = rc * edge * (power + 1.0) / (2.0 * length) * grade
            kappa = 1.0 + (kmax - 1.0) * grade + torch.zeros_like(damp)
            b = -alpha - damp / kappa
            self.layers.append({"face": face, "axis": axis, "lo": lo, "n": n, "a": -damp / (kappa * kappa), "b": b,
                                "kappa": kappa, "psi": None})
            _slice(self.sponge, axis, lo, n).add_(sponge * edge * _along(depth ** (power + 1.0), axis))
            if axis == Z:
                scale = alpha / kappa / (damp / kappa + alpha)
                for v in (self.grad_rho[2], self.grad_p[2]):
                    _slice(v, Z, lo, n).mul_(scale)
                self.g[lo:lo + n] *= scale[:, 0, 0]
        self.layers.sort(key=lambda layer: layer["face"])

    def _source(self, seed):
        """The pulse's shape in space, or the cube's weight in depth; the damping rates."""
        s, (nx, ny, nz), dev = self.s, self.n, self.z.device
        cells = (nx, ny) if self.wrapped else (nx - 1, ny - 1)

        def bell(x, width):
            return torch.exp(-(x * x) / (2.0 * (width / RSUN) ** 2))

        def offsets(n, cell, at):
            return torch.arange(n, dtype=torch.float64, device=dev) / cell * s["width"] / RSUN - at / RSUN

        if self.case["cube"]:
            self.maps = torch.from_numpy(_cube(self.case, seed)).to(dev) * (s["amp"] / self.dimc)
            away = (self.z - (1.0 + s["depth"] / RSUN)).abs().cpu().numpy()
            at = max(k for k in range(nz) if away[k] == away.min())
            self.shape = torch.exp(-0.25 * ((self.z - self.z[at]) / (s["sigma"] / RSUN)) ** 2)[:, None, None]
        else:
            x, y = bell(offsets(nx, cells[0], s["px"]), s["sr"]), bell(offsets(ny, cells[1], s["py"]), s["sr"])
            self.shape = bell(self.z - (s["pz"] / RSUN + 1.0), s["sz"])[:, None, None] * y[None, :, None] * x
        kx = torch.arange(nx // 2 + 1, dtype=torch.float64, device=dev)
        ky = torch.arange(ny, dtype=torch.float64, device=dev)
        k = 2.0 * PI * RSUN / s["width"] * torch.sqrt(kx ** 2 + torch.minimum(ky, ny - ky)[:, None] ** 2)
        self.rates = RSUN / self.dimc / (nx * ny) * 1e-6 * 500.0 * (k / 902.0) ** 2.2 * 20.0

    def source(self, time):
        """The source term of vz at a time index."""
        s, t = self.s, time * self.s["dt"]
        if not self.case["cube"]:
            wave = math.sin(2.0 * PI * (t - s["t1"] + 2.0 * s["t0"]) / s["t0"])
            return s["amp"] / 0.56458272 / self.dimc * wave * math.exp(-(t - s["t1"]) ** 2 / (2.0 * s["st"] ** 2)) * self.shape
        # Lagrange's polynomial through the maps of the interval's seven nodes,
        # those before the start left out
        first = math.floor(float(time) * s["dt"] / s["cad"]) + 1
        nodes = [(first - 4 + q) * s["cad"] for q in range(7)]
        total = 0.0
        for q, node in enumerate(nodes):
            if node >= 0:
                weight = math.prod((t - x) / (node - x) for x in nodes if x != node)
                total = total + weight * self.maps[first - 4 + q]
        return total[None] * self.shape

    def rates_of(self, u, stage_psi, source):
        """The right-hand side of every field, and of every layer's psi."""
        rho, vx, vy, vz, p = u[:5]
        along = {X: [(vx, "vx"), (p, "px")], Y: [(vy, "vy"), (p, "py")], Z: [(vz, "vz"), (p, "pz")]}
        if self.mhd:
            bx, by, bz = u[5:]
            b0x, b0y, b0z = self.b0
            f1, f2, f3 = vy * b0z - vz * b0y, vz * b0x - vx * b0z, vx * b0y - vy * b0x
            along[X] += [(by, "byx"), (bz, "bzx"), (f3, "f3x"), (f2, "f2x")]
            along[Y] += [(bx, "bxy"), (bz, "bzy"), (f3, "f3y"), (f1, "f1y")]
            along[Z] += [(bx, "bxz"), (by, "byz"), (f2, "f2z"), (f1, "f1z")]
        d, psi_rates = {}, [[] for _ in self.layers]
        for axis, take in ((X, self.ddx), (Y, self.ddy), (Z, self.ddz)):
            for i, (f, name) in enumerate(along[axis]):
                v = take(f)
                for q, layer in enumerate(self.layers):
                    if layer["axis"] == axis:
                        part, psi = _slice(v, axis, layer["lo"], layer["n"]), stage_psi[q][i]
                        psi_rates[q].append(layer["a"] * part + layer["b"] * psi)
                        part.copy_(part / layer["kappa"] + psi)
                d[name] = v
        div, sp, inv = d["vx"] + d["vy"] + d["vz"], self.sponge, 1.0 / self.rho0
        g = self.g[:, None, None]
        out = [-self.rho0 * div - sp * rho, -inv * d["px"] - sp * vx, -inv * d["py"] - sp * vy,
               -inv * (d["pz"] + rho * g) - sp * vz, -self.c2 * self.rho0 * div - sp * p]
        for v, gr, gp in zip((vx, vy, vz), self.grad_rho, self.grad_p):
            if gr is not None:
                out[0] -= gr * v
                out[4] -= gp * v
        if self.mhd:
            cx, cy, cz = d["bzy"] - d["byz"], d["bxz"] - d["bzx"], d["byx"] - d["bxy"]
            ox, oy, oz = self.curl0
            force = inv * self.red
            out[1] += force * (cy * b0z - cz * b0y + oy * bz - oz * by)
            out[2] += force * (cz * b0x - cx * b0z + oz * bx - ox * bz)
            out[3] += force * (cx * b0y - cy * b0x + ox * by - oy * bx)
            out += [self.red * (d["f3y"] - d["f2z"]), self.red * (d["f1z"] - d["f3x"]), self.red * (d["f2x"] - d["f1y"])]
        out[3] += source
        for k in out:
            k[0], k[-1] = 0.0, 0.0
            if not self.wrapped:
                k[:, 0], k[:, -1], k[:, :, 0], k[:, :, -1] = 0.0, 0.0, 0.0, 0.0
        if self.case["damping"]:
            for f in (1, 2, 3):
                w = torch.fft.rfft2(u[f]) * self.rates
                out[f] -= torch.fft.irfft2(w, s=u[f].shape[1:], norm="forward")
        return out, psi_rates

    def step(self, time):
        """One step; the driver's watch values of it (norm, minima)."""
        source = self.source(time)
        if self.layers[0]["psi"] is None:
            for layer in self.layers:
                layer["psi"] = [torch.zeros_like(layer["kappa"]) for _ in range(6 if self.mhd else 2)]
        base, psi_base = self.u, [layer["psi"] for layer in self.layers]
        u, psi = base, psi_base
        for w in self.weights + [self.dt]:
            least = [float((u[f] + b).min()) for f, b in ((0, self.rho0), (4, self.p0))] if w == self.dt else None
            k, kp = self.rates_of(u, psi, source)
            u = [a + w * r for a, r in zip(base, k)]
            psi = [[a + w * r for a, r in zip(pa, pk)] for pa, pk in zip(psi_base, kp)]
        self.u = u
        for layer, v in zip(self.layers, psi):
            layer["psi"] = v
        m = (self.rho0 + u[0]) * (u[1] ** 2 + u[2] ** 2 + u[3] ** 2) / 2.0
        return [float((m * m).mean().sqrt()) * self.dimc ** 2 * self.dimrho] + least

    def filter_vars(self, time):
        g = 5 if self.case["taps"] == 11 else 3
        for seconds, axes in ((self.case["t_xy"], (Y, X)), (self.case["t_z"], (Z,))):
            if time % math.floor(max(seconds, self.s["dt"]) / self.s["dt"] + 1e-5) == 0:
                for axis in axes:
                    self.u = [filtered(f, axis, g, self.wrapped and axis != Z, 1.0) for f in self.u]

    def results(self, steps):
        out, history = {}, []
        for t in range(steps):
            history.append(self.step(t))
            if t:
                self.filter_vars(t)
        if self.case["checked"]:
            out["history"] = np.array(history)
        if self.case["psi"]:
            out["psi"] = {str(layer["face"]): torch.stack(layer["psi"]) for layer in self.layers}
        out.update({FIELDS[f]: v for f, v in enumerate(self.u)})
        return out


def exact(case, seed):
    if case["kind"] == "operators":
        plain = Plain(_grid_of(case), seed)
        f, w = torch.from_numpy(_field(case, seed)).to(_device()), case["periodic"]
        return {"ddx": plain.ddx(f), "ddy": plain.ddy(f), "ddz": plain.ddz(f),
                "filtx": filtered(f, X, 5, w), "filty": filtered(f, Y, 5, w), "filtz": filtered(f, Z, 5, False)}
    if case["kind"] == "batch":
        return [Plain(m, seed + 100 * q).results(case["steps"]) for q, m in enumerate(_members(case))]
    return Plain(case, seed).results(case["steps"])
