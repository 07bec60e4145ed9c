"""Workloads that time the hydro step through the package's public entry points.

``listed()`` holds one case for each way in which a program uses the package,
``draw(rng)`` gives further cases of the same ranges.  A case is a dict of plain
values; ``prepare`` makes what a program holds before the call (grids, batches,
input fields made on the GPU from the seed), ``run`` takes one pass,
``work`` states the bytes and operations that pass cannot do without, and
``exact`` gives the same outputs from plain torch in FP64.

Kinds of case:

* ``rollout``: conserved planes on the device are set into a grid, ``steps``
  steps are taken, the planes are read back -- the device-resident use of
  ``HydroGrid``.  Options: grid size (odd sizes, flat z), walls, step mode,
  the call-by-call driver sequence, the tabulated EOS, flux_ang, gravity.
* ``host``: the boundary of the Fortran driver: upload of host arrays, steps,
  download; FP64 or the mixed form.
* ``tubes`` / ``boxes``: the batched launches of many small problems.
* ``adjoint``: a forward and its gradient through the autograd function.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from boxzyhydro_amd import ics
from boxzyhydro_amd import native as nv
from boxzyhydro_amd.adjoint import AdjointStepper, hydro_function
from boxzyhydro_amd.batch import TubeBatch
from boxzyhydro_amd.boxes import GridBatch
from boxzyhydro_amd.hydro import HydroGrid, step_sequence
from boxzyhydro_amd.params import HydroParams

MODES = {"exact": nv.BX_STEP_EXACT, "fused": nv.BX_STEP_FUSED, "graph": nv.BX_STEP_GRAPH}
FLOPS = 1100.0  # FP64 operations of one cell-update: both stages' slopes, states, faces and updates


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu", 0 if torch.cuda.is_available() else None)


# ------------------------------------------------------------------- cases
def listed():
    return [
        # the reference's own first run: the 400-cell Sod tube, replayed from graphs; launches and latency are all of it
        _rollout("sod_400", 400, 4, 4, steps=200, mode="graph", ic="sod"),
        # a small box in HydroGrid.run's default mode, each dt handed back to the host
        _rollout("box_32_fused", 32, 32, 32, steps=48, mode="fused"),
        # the reference's shipped in.nml walls every side; sizes that fill no tile
        _rollout("box_walls_ragged", 97, 61, 43, steps=40, mode="graph", walls="xXyYzZ"),
        # the headline box
        _rollout("box_256", 256, 256, 256, steps=24, mode="graph"),
        # a driver that keeps the reference's calls, one subroutine at a time
        _rollout("calls_96", 96, 96, 96, steps=4, mode="calls"),
        # molecular cloud with the tabulated H2 equation of state
        _rollout("cloud_eos_128", 128, 128, 128, steps=8, mode="fused", ic="cloud", eos=True),
        # rotating disk with angular-momentum fluxes about a point mass, the potential of its surroundings given
        _rollout("disk_ang_point", 120, 120, 24, steps=8, mode="fused", ic="disk", ang=True, gravity="point"),
        # gas in a given potential, the caller's own solver in between
        _rollout("potential_160", 160, 144, 128, steps=24, mode="graph", gravity="potential"),
        # host arrays in, 100 mixed-precision steps, host arrays out
        {"name": "host_mixed_192", "kind": "host", "x": 192, "y": 192, "z": 192, "steps": 100, "mode": "graph",
         "precision": "mixed", "walls": ""},
        # many shock tubes of uneven length in one launch
        {"name": "tubes_256", "kind": "tubes", "count": 256, "lmin": 64, "lmax": 1024, "endtime": 0.1,
         "members": 6, "gangs": 24, "layout": 0},
        # many small boxes of uneven size, walled on some sides, in one launch
        {"name": "boxes_192", "kind": "boxes", "count": 192, "lmin": 8, "lmax": 32, "endtime": 1.0, "walls": True,
         "layout": 0},
        # gradient of a loss on the final density with respect to the initial state
        {"name": "adjoint_96", "kind": "adjoint", "x": 96, "y": 96, "z": 96, "steps": 40, "every": 20, "walls": ""},
    ]


def _rollout(name, x, y, z, *, steps, mode, ic="box", walls="", eos=False, ang=False, gravity="none"):
    return {"name": name, "kind": "rollout", "x": x, "y": y, "z": z, "steps": steps, "mode": mode, "ic": ic,
            "walls": walls, "eos": eos, "ang": ang, "gravity": gravity}


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box_sizes(rng, lo, hi, most):
    while True:
        x, y, z = (_log_int(rng, lo, hi) for _ in range(3))
        if x * y * z <= most:
            return x, y, z


def draw(rng):
    kind = rng.choice(["tube", "small", "walls", "large", "calls", "eos", "ang", "potential", "host", "tubes", "boxes",
                       "adjoint"])
    walls = "".join(s for s in "xXyYzZ" if rng.random() < 0.5)
    mode = rng.choice(["fused", "graph"])
    if kind == "tube":
        c = _rollout("", _log_int(rng, 64, 4096), rng.choice([4, 5, 7, 8]), rng.choice([1, 3, 4]),
                     steps=rng.randrange(100, 240, 2), mode=mode, ic="sod")
    elif kind == "small":
        c = _rollout("", *_box_sizes(rng, 8, 64, 64**3), steps=rng.randint(30, 64), mode=mode)
    elif kind == "walls":
        c = _rollout("", *_box_sizes(rng, 24, 144, 100**3), steps=rng.randint(24, 48), mode=mode, walls=walls or "xX")
    elif kind == "large":
        c = _rollout("", *_box_sizes(rng, 128, 320, 256**3), steps=rng.randint(16, 24), mode=mode)
    elif kind == "calls":
        c = _rollout("", *_box_sizes(rng, 24, 160, 128**3), steps=rng.randint(3, 6),
                     mode=rng.choice(["calls", "exact"]), walls=walls)
    elif kind == "eos":
        c = _rollout("", *_box_sizes(rng, 32, 160, 128**3), steps=rng.randint(4, 8), mode="fused", ic="cloud",
                     eos=True, walls=rng.choice(["", walls]))
    elif kind == "ang":
        x, y, z = _box_sizes(rng, 32, 160, 100**3)
        c = _rollout("", x - x % 2, y, z, steps=rng.randint(4, 10), mode="fused", ic="disk",  # no cell centre on the axis
                     ang=rng.random() < 0.7, gravity="point")
    elif kind == "potential":
        c = _rollout("", *_box_sizes(rng, 32, 192, 160**3), steps=rng.randint(16, 32), mode=mode, gravity="potential",
                     walls=rng.choice(["", walls]))
    elif kind == "host":
        x, y, z = _box_sizes(rng, 48, 192, 160**3)
        c = {"kind": "host", "x": x, "y": y, "z": z, "steps": rng.randint(20, 100), "mode": mode,
             "precision": rng.choice(["fp64", "mixed"]), "walls": rng.choice(["", "xXyY"])}
    elif kind == "tubes":
        c = {"kind": "tubes", "count": rng.randint(48, 320), "lmin": rng.randint(32, 96), "lmax": _log_int(rng, 256, 1200),
             "endtime": 0.1, "members": rng.choice([0, 4, 6, 8]), "gangs": rng.randint(8, 24),
             "layout": rng.randrange(1000)}
    elif kind == "boxes":
        c = {"kind": "boxes", "count": rng.randint(48, 240), "lmin": 8, "lmax": rng.randint(20, 36), "endtime": 1.0,
             "walls": rng.random() < 0.5, "layout": rng.randrange(1000)}
    else:
        x, y, z = _box_sizes(rng, 32, 128, 96**3)
        c = {"kind": "adjoint", "x": x, "y": y, "z": z, "steps": rng.randint(20, 48), "every": rng.choice([5, 10, 20]),
             "walls": rng.choice(["", "xX", "zZ"])}
    c.pop("name", None)
    return c


# -------------------------------------------------------------- parameters
def _params(case) -> HydroParams:
    kind = case["kind"]
    flat = kind == "rollout" and case["ic"] == "sod"  # tubes: nz < 6 has no ghost planes in z
    walls = case.get("walls", "")
    no = {f"no_outflow_{'xyz'['xyz'.index(s.lower())]}{'l' if s.islower() else 'r'}": s in walls for s in "xXyYzZ"}
    p = dict(nx=case["x"] + 4, ny=case["y"] + 4, nz=case["z"] + (0 if flat else 4), small_eps=1e-40, cfl=0.5,
             endtime=1e30, dtout=1e30, **no)
    if flat:
        d = 1.0 / case["x"]
        return HydroParams(dx=d, dy=d, dz=d, small_rho=1e-12, vlimit=10.0, gammafix=1.4, **p)
    if case.get("eos"):
        return HydroParams(dx=1.0, dy=1.0, dz=1.0, small_rho=1e-10, vlimit=10.0, gammafix=1.4, H2STAT=0,
                           tk_bgrnd=10.0, NEOS_RHO=400, dTk_eos=10.0, **p)
    return HydroParams(dx=1.0, dy=1.0, dz=1.0, small_rho=1e-10, vlimit=10.0, gammafix=5.0 / 3.0,
                       fluxangmom=bool(case.get("ang")), **p)


def _coords(prm, dev):
    """Centred cell coordinates as broadcastable (nz, ny, nx) views."""
    x, y, z = (d * (torch.arange(1, n + 1, dtype=torch.float64, device=dev) - (n + 1.0) / 2.0)
               for d, n in ((prm.dx, prm.nx), (prm.dy, prm.ny), (prm.dz, prm.nz)))
    return x[None, None, :], y[None, :, None], z[:, None, None]


def _unit(shape, gen, passes):
    """White noise smoothed along each axis, with zero mean and unit spread."""
    f = torch.randn(shape, generator=gen, device=gen.device, dtype=torch.float64)
    for dim in range(3):
        if shape[dim] > 2:
            for _ in range(passes):
                f = 0.5 * f + 0.25 * (torch.roll(f, 1, dim) + torch.roll(f, -1, dim))
    f = f - f.mean()
    return f / f.std()


def _fields(case, prm, seed, dev):
    """Density, velocity and pressure of the set-up, each on (nz, ny, nx)."""
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    shp = prm.shape
    if case.get("ic") == "sod":  # Sod's tube with the diaphragm and the two states moved a little by the seed
        r = torch.rand(4, generator=gen, device=dev, dtype=torch.float64).tolist()
        left = (_coords(prm, dev)[0] < 0.1 * (r[0] - 0.5)).expand(shp)
        rho = torch.where(left, 1.0 + 0.1 * r[1], 0.125)
        p = torch.where(left, 1.0 + 0.1 * r[2], 0.1 + 0.01 * r[3])
        return rho.double(), torch.zeros((3,) + shp, dtype=torch.float64, device=dev), p.double()
    g1, g2 = _unit(shp, gen, 8), _unit(shp, gen, 8)
    vel = torch.randn((3,) + shp, generator=gen, device=dev, dtype=torch.float64)
    if case.get("ic") == "cloud":  # density and temperature over the tables' range
        rho = 0.1 * torch.exp(g1)
        lo, hi = math.log(20.0), math.log(4000.0)
        tk = torch.exp(torch.clamp(0.5 * (lo + hi) + 0.25 * (hi - lo) * g2, lo, hi))
        rgas, muc = _gas(prm)
        p = rho * rgas * tk / muc
    else:
        rho = torch.exp(0.1 * g1)
        p = 1.0 + 0.05 * g2
    mach = 0.3 if case.get("ic") == "disk" else 0.5
    vel = vel * (mach * (prm.gammafix * p.mean() / rho.mean()).sqrt() / vel.square().sum(0).mean().sqrt())
    if case.get("ic") == "disk":
        x, y, _ = _coords(prm, dev)
        vel = torch.stack([vel[0] - 0.002 * y, vel[1] + 0.002 * x, vel[2]])
    return rho, vel, p


def _edge(prm, dev, width):
    """Cells of the outer `width` layers (x, y, and z where it has ghost planes)."""
    m = torch.zeros(prm.shape, dtype=torch.bool, device=dev)
    for dim, n in ((0, prm.nz), (1, prm.ny), (2, prm.nx)):
        if dim == 0 and n < 6:
            continue
        m.narrow(dim, 0, width).fill_(True)
        m.narrow(dim, n - width, width).fill_(True)
    return m


def _planes(case, prm, seed, dev, frame=True):
    """(5, nz, ny, nx) conserved planes of the set-up, its outermost layer empty as the reference's set-ups leave it."""
    rho, v, p = _fields(case, prm, seed, dev)
    c = torch.empty((5,) + prm.shape, dtype=torch.float64, device=dev)
    c[0] = rho
    c[1:4] = rho * v
    c[4] = p / (prm.gammafix - 1.0) + rho * 0.5 * v.square().sum(0)
    if frame:
        e = _edge(prm, dev, 1)
        c[0][e] = prm.small_rho
        c[1:4] = torch.where(e, 0.0, c[1:4])
        c[4][e] = prm.small_eps
    return c, v, p


def _phi(prm, dev):
    x, y, z = _coords(prm, dev)
    return -1.0 / torch.sqrt(x * x + y * y + z * z + 100.0)


POINT = {"object_mass": 1.0, "object_radius": 20.0}


def _tubes(case, seed):
    """Riemann problems of uneven length (log-uniform, given by the case's layout) with the package's set-up
    convention: densities and pressures log-uniform in [0.1, 10], velocities uniform in [-1, 1], from the seed."""
    shape = np.random.Generator(np.random.PCG64(case["layout"]))
    rng = np.random.Generator(np.random.PCG64(seed))
    out = []
    for _ in range(case["count"]):
        length = int(np.rint(np.exp(shape.uniform(np.log(case["lmin"]), np.log(case["lmax"])))))
        d = 1.0 / length
        prm = HydroParams(nx=length + 4, ny=8, nz=4, dx=d, dy=d, dz=d, no_outflow_xl=False, no_outflow_xr=False,
                          no_outflow_yl=False, no_outflow_yr=False, no_outflow_zl=False, no_outflow_zr=False,
                          small_rho=1e-12, small_eps=1e-40, vlimit=1e3, endtime=case["endtime"], dtout=1e30, cfl=0.5,
                          gammafix=1.4)
        left = ics.cell_centres(prm)[0] < 0.0
        rl, rr, pl, pr = np.exp(rng.uniform(np.log(0.1), np.log(10.0), 4))
        vl, vr = rng.uniform(-1.0, 1.0, 2)
        out.append((prm, ics.tube_row(prm, np.where(left, rl, rr), np.where(left, vl, vr), np.where(left, pl, pr))))
    return out


def _grids(case, seed):
    """Uneven boxes: interior cells per axis log-uniform and walls on random sides (given by the case's layout),
    smoothed density and pressure."""
    rng = np.random.Generator(np.random.PCG64(case["layout"]))
    dev = _device()
    out = []
    for i in range(case["count"]):
        x, y, z = (int(round(v)) for v in np.exp(rng.uniform(np.log(case["lmin"]), np.log(case["lmax"]), 3)))
        walls = "".join(s for s, w in zip("xXyYzZ", rng.integers(0, 2, 6)) if w and case["walls"])
        one = {"kind": "box", "x": x, "y": y, "z": z, "walls": walls}
        prm = _params(one)
        c, v, p = _planes(one, prm, seed * 1000 + i, dev)
        out.append((prm, {"cons": c.reshape(5, -1).T.contiguous().cpu().numpy(),
                          "u": v.reshape(3, -1).T.contiguous().cpu().numpy(), "p": p.reshape(-1).cpu().numpy()}))
    return out


# ----------------------------------------------------------------- prepare
def prepare(case, seed):
    kind = case["kind"]
    if kind == "tubes":
        b = TubeBatch(_tubes(case, seed))
        b.run()
        b.sync()  # the steps of each tube, by which the gangs are chosen
        b.gang(case["members"], case["gangs"] if case["members"] else 0)
        return {"kind": kind, "batch": b}
    if kind == "boxes":
        grids = _grids(case, seed)
        return {"kind": kind, "batch": GridBatch(grids, endtimes=[case["endtime"]] * len(grids))}
    prm, dev = _params(case), torch.device("cuda", 0)
    if kind == "adjoint":
        rho, v, p = _fields(case, prm, seed, dev)
        st = AdjointStepper(prm, v.reshape(3, -1).T.contiguous().cpu().numpy(), case["steps"], case["every"])
        target = _fields(case, prm, seed + 7919, dev)[0].reshape(-1)
        s = {"kind": kind, "stepper": st, "rho": rho.reshape(-1).clone(), "p": p.reshape(-1).clone(),
             "target": target.clone(), "inside": (~_edge(prm, dev, 2)).reshape(-1).double(), "fn": hydro_function()}
        st.forward(s["rho"], s["p"], checkpoint=False)  # fixes the dt sequence
        return s
    planes, v, p = _planes(case, prm, seed, dev)
    if kind == "host":
        g = HydroGrid(prm, precision=nv.BX_PREC_MIXED if case["precision"] == "mixed" else nv.BX_PREC_FP64)
        host = {"cons": planes.reshape(5, -1).T.contiguous().cpu().numpy(),
                "u": v.reshape(3, -1).T.contiguous().cpu().numpy(), "p": p.reshape(-1).cpu().numpy()}
        return {"kind": kind, "grid": g, "host": host, "steps": case["steps"], "mode": MODES[case["mode"]]}
    g = HydroGrid(prm)
    if case["gravity"] != "none":
        flags = nv.BX_GRAV_POTENTIAL | (nv.BX_GRAV_EXTERNAL if case["gravity"] == "point" else 0)
        g.set_gravity(flags, _phi(prm, dev).reshape(-1).cpu().numpy(), initial=False, **POINT)
    return {"kind": kind, "grid": g, "planes": planes, "out": torch.empty_like(planes), "steps": case["steps"],
            "mode": case["mode"], "gravity": case["gravity"]}


# --------------------------------------------------------------------- run
def _restart(g):
    g.time, g.dt, g.dtold, g.step_count = g.prm.starttime, 0.0, 0.0, 0


def run(s):
    kind = s["kind"]
    if kind in ("tubes", "boxes"):
        b = s["batch"]
        b.run(graph=True)
        b.sync()
        res = b.result()
        out = {k: np.concatenate([r[k] for r in res]) for k in ("cons", "u", "p")}
        out["time"] = np.array([r["time"] for r in res])
        out["steps"] = np.array([r["steps"] for r in res])
        out["status"] = np.array([r["status"] for r in res], np.int64)
        return out
    if kind == "adjoint":
        rho, p = s["rho"].detach().requires_grad_(), s["p"].detach().requires_grad_()
        final = s["fn"].apply(rho, p, s["stepper"])
        loss = 0.5 * ((final - s["target"]).square() * s["inside"]).sum()
        loss.backward()
        return {"rho": final.detach(), "grad_rho": rho.grad, "grad_p": p.grad}
    g = s["grid"]
    _restart(g)
    if kind == "host":
        g.upload(s["host"])
        dts = g.run(s["steps"], mode=s["mode"])
        out = g.download()
        return {"cons": out["cons"], "u": out["u"], "p": out["p"], "dts": dts}
    lib = nv.lib()
    nv.check(lib.bx_cons_device(g._h, ctypes.c_void_p(s["planes"].data_ptr()), 1), "bx_cons_device")
    if s["gravity"] != "none":  # the calls before the main loop
        g.calc_gforce()
        if s["gravity"] == "point":
            g.external_grav()
    if s["mode"] == "calls":
        dts = np.array(step_sequence(g, s["steps"], g.prm.endtime)[0])
    else:
        dts = g.run(s["steps"], mode=MODES[s["mode"]])
    nv.check(lib.bx_cons_device(g._h, ctypes.c_void_p(s["out"].data_ptr()), 0), "bx_cons_device")
    return {"cons": s["out"], "dts": dts}


# -------------------------------------------------------------------- work
def work(case):
    """A step reads the state and writes it (5 FP64 fields each way, FP32 in the mixed form)."""
    kind = case["kind"]
    if kind == "tubes":
        # row cells: mean of a log-uniform length, and steps in proportion to it (about 4 per cell of a tube)
        lo, hi = case["lmin"], case["lmax"]
        cells = case["count"] * (hi - lo) / math.log(hi / lo)
        updates = case["count"] * 4.0 * (case["endtime"] / 0.1) * (hi * hi - lo * lo) / (2.0 * math.log(hi / lo))
        return {"bytes": 2 * 72.0 * cells, "flops": 500.0 * updates}
    if kind == "boxes":
        mean = (case["lmax"] - case["lmin"]) / math.log(case["lmax"] / case["lmin"])
        cells = case["count"] * mean**3
        return {"bytes": 2 * 72.0 * cells, "flops": FLOPS * cells * 10 * case["endtime"]}
    prm = _params(case)
    n, updates = prm.ngrid, float(prm.interior_cells) * case["steps"]
    if kind == "host":
        size = 4 if case["precision"] == "mixed" else 8
        return {"bytes": 10.0 * size * updates + 2 * 72.0 * n, "flops": FLOPS * updates}
    if kind == "adjoint":
        return {"bytes": 3 * 80.0 * updates, "flops": 3 * FLOPS * updates}
    return {"bytes": 80.0 * updates, "flops": FLOPS * updates * (0.7 if prm.nz < 6 else 1.0)}


# ------------------------------------------------------------------- exact
def _gas(prm):
    """Gas constant in code units (AU, year/2pi) and the mean molecular weight of the mixture."""
    unit_time = (3600.0 * 365.25 * 24.0) / (2.0 * math.pi)
    rgas = 8.254e7 / (1.496e13 / unit_time) ** 2
    return rgas, 1.0 / (prm.xabun * 0.5 + prm.yabun * 0.25 + prm.zabun / prm.mu_z)


def _floor(x, lo):
    return torch.where(x > lo, x, lo)


class _Plain:
    """The step of main.f90:211-555 in plain torch FP64, fixed gamma: whole-array operations, no kernels of the package."""

    def __init__(self, prm, dev):
        self.prm, self.dev = prm, dev
        self.flat = prm.nz < 6
        self.inside = ~_edge(prm, dev, 2)
        self.rgas, self.muc = _gas(prm)
        self.gm1 = prm.gammafix - 1.0
        self.vol = prm.dx * prm.dy * prm.dz
        # ghost cells: per axis the donor index (mirrored at a wall, else the nearest interior cell) and the sign
        self.donor, self.sign = [], []
        for axis, n in enumerate((prm.nx, prm.ny, prm.nz)):
            idx, sg = torch.arange(n, device=dev), torch.ones(n, dtype=torch.float64, device=dev)
            if axis < 2 or not self.flat:
                for lo, wall in ((True, prm.no_outflow[2 * axis]), (False, prm.no_outflow[2 * axis + 1])):
                    for k in (0, 1):
                        ghost, mirror, near = (k, 3 - k, 2) if lo else (n - 1 - k, n - 4 + k, n - 3)
                        idx[ghost] = mirror if wall else near
                        sg[ghost] = -1.0 if wall else 1.0
            self.donor.append(idx)
            self.sign.append(sg)
        self.x, self.y, self.z = _coords(prm, dev)
        self.gf = None

    def ghosts(self, c):
        f = c.index_select(3, self.donor[0]).index_select(2, self.donor[1]).index_select(1, self.donor[2])
        return torch.stack([f[0], f[1] * self.sign[0][None, None, :], f[2] * self.sign[1][None, :, None],
                            f[3] * self.sign[2][:, None, None], f[4]])

    def state(self, c, u, p):
        ek = c[0] * 0.5 * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2])
        pn = _floor(c[4] - ek, self.prm.small_eps) * self.gm1
        low = c[0] < 1e-4
        if not bool(low.any()):
            return c, pn
        pl = c[0] * torch.clamp(p / (c[0] * self.rgas) * self.muc, max=5e3) * self.rgas / self.muc
        c = torch.cat([c[:4], torch.where(low, pl / self.gm1 + ek, c[4])[None]])
        return c, torch.where(low, pl, pn)

    def velocity(self, c):
        u = c[1:4] / c[0]
        fast = (u.abs() > self.prm.vlimit).any(0)
        if not bool(fast.any()):
            return c, u
        uc = torch.where(fast, u * self.prm.vlimit / u.square().sum(0).sqrt(), u)
        m = uc * c[0]
        e = _floor(c[4] - 0.5 * c[1:4].square().sum(0) / c[0], self.prm.small_eps) + 0.5 * m.square().sum(0) / c[0]
        return torch.cat([c[:1], torch.where(fast, m, c[1:4]), torch.where(fast, e, c[4])[None]]), uc

    def rate(self, c, u, p):
        s = torch.sqrt(self.prm.gammafix * p / c[0])
        return (s + u[0].abs()) / self.prm.dx + (s + u[1].abs()) / self.prm.dy + (s + u[2].abs()) / self.prm.dz

    def source(self, c, u, dt):
        rho, m = c[0], c[1:4]
        work = 0.0
        if self.prm.fluxangmom:
            x, y = self.x, self.y
            w = x * u[1] - y * u[0]
            k = rho * (w * w) / (x * x + y * y) ** 2 * dt
            m = torch.stack([m[0] + k * x, m[1] + k * y, m[2]])
        if self.gf is not None:
            m = m + rho * self.gf * dt
            work = dt * rho * (u * self.gf).sum(0)
        ek = 0.5 * (m[0] * m[0] + m[1] * m[1] + m[2] * m[2]) / rho
        e = _floor(c[4] - ek + work, self.prm.small_eps) + ek
        return torch.where(self.inside, torch.cat([rho[None], m, e[None]]), c)

    def flux(self, c, old, u, p, dt):
        prm, g, ang = self.prm, self.prm.gammafix, self.prm.fluxangmom
        if ang:  # momenta about the z axis
            c, old = self._turn(c), None if old is None else self._turn(old)
        eps = _floor(c[4] - 0.5 * c[0] * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2]), prm.small_eps)
        snd = torch.sqrt(p * g / c[0])
        W = torch.cat([c[:1], u, p[None], eps[None]] + ([c[1:3]] if ang else []))
        total = 0.0
        for d, dim, ds, area in ((0, 3, prm.dx, prm.dy * prm.dz), (1, 2, prm.dy, prm.dx * prm.dz),
                                 (2, 1, prm.dz, prm.dx * prm.dy)):
            if d == 2 and self.flat:
                continue
            n = W.shape[dim]
            a, b, e = W.narrow(dim, 0, n - 2), W.narrow(dim, 1, n - 2), W.narrow(dim, 2, n - 2)
            x1, x2, x3 = 1.25 * (b - a), 0.5 * (e - a), 1.25 * (e - b)
            mn, mx = torch.minimum(x1, torch.minimum(x2, x3)), torch.maximum(x1, torch.maximum(x2, x3))
            s = torch.where(mn > 0, mn, torch.where(mx < 0, mx, 0.0))
            pad = [0, 0, 0, 0, 0, 0]
            pad[2 * (3 - dim)] = pad[2 * (3 - dim) + 1] = 1
            s = torch.where(self.inside, torch.nn.functional.pad(s, pad), 0.0)
            minus = W + 0.5 * (-1.0 - _neg(u[d] - snd) * dt / ds) * s
            plus = W + 0.5 * (1.0 - _floor(u[d] + snd, 0.0) * dt / ds) * s
            F, pf = self._hll(plus.narrow(dim, 0, n - 1), minus.narrow(dim, 1, n - 1), d)
            dF = torch.nn.functional.pad(F.narrow(dim, 1, n - 2) - F.narrow(dim, 0, n - 2), pad)
            if ang and d < 2:  # the pressure force projected with the cell's own position
                dp = torch.nn.functional.pad(pf.narrow(dim - 1, 1, n - 2) - pf.narrow(dim - 1, 0, n - 2), pad)
                r = torch.sqrt(self.x * self.x + self.y * self.y)
                along, turn = (self.x / r, -self.y) if d == 0 else (self.y / r, self.x)
                dF = torch.stack([dF[0], dF[1] + dp * along, dF[2] + dp * turn, dF[3], dF[4]])
            total = total + area * dF
        ft = torch.where(self.inside, -(total * dt / self.vol), 0.0)
        U = c + ft if old is None else 0.5 * (old + c + ft)
        if ang:
            U = self._turn_back(U)
        r = _floor(U[0], prm.small_rho)
        e = torch.where(U[4] < 0.0, 0.5 * U[1:4].square().sum(0) / r + prm.small_eps, U[4])
        return torch.cat([r[None], U[1:4], e[None]])

    def _hll(self, L, R, d):
        g, ang = self.prm.gammafix, self.prm.fluxangmom
        sides = []
        for S in (L, R):
            m = S[0] * S[1:4]
            if ang:
                m = torch.stack([S[6], S[7], m[2]])
            E = S[5] + 0.5 * S[0] * (S[1] * S[1] + S[2] * S[2] + S[3] * S[3])
            v = S[1 + d]
            f = torch.cat([(S[0] * v)[None], m * v, ((E + S[4]) * v)[None]])
            if not (ang and d < 2):
                f = torch.stack([f[k] + (S[4] if k == 1 + d else 0.0) for k in range(5)])
            sides.append((torch.cat([S[:1], m, E[None]]), f, v, torch.sqrt(g * S[4] / S[0]), S[4]))
        (sl, fl, vl, cl, pl), (sr, fr, vr, cr, pr) = sides
        ap = _larger(_floor(vr + cr, 0.0), vl + cl)
        am = _larger(_floor(cr - vr, 0.0), cl - vl)
        den = ap + am
        pf = (ap * pl + am * pr) / den if ang and d < 2 else None
        return (ap * fl + am * fr - ap * am * (sr - sl)) / den, pf

    def _turn(self, c):
        x, y = self.x, self.y + self.prm.yoffset
        r = torch.sqrt(x * x + y * y)
        return torch.stack([c[0], (c[1] * x + c[2] * y) / r, x * c[2] - y * c[1], c[3], c[4]])

    def _turn_back(self, c):
        x, y = self.x, self.y + self.prm.yoffset
        r = torch.sqrt(x * x + y * y)
        return torch.stack([c[0], (c[1] * x - c[2] * y / r) / r, (c[1] * y + c[2] * x / r) / r, c[3], c[4]])

    def force(self, phi, rho, point):
        """Centred differences of the potential, and a softened point mass at minus the grid's mass moment."""
        prm, gf = self.prm, []
        for dim, d in ((2, prm.dx), (1, prm.dy), (0, prm.dz)):
            gf.append(-(torch.roll(phi, -1, dim) - torch.roll(phi, 1, dim)) / (2.0 * d))
        self.gf = torch.stack(gf)
        if point:
            mass, radius = POINT["object_mass"], POINT["object_radius"]
            x = self.x + (self.x * rho).sum() * self.vol / mass
            y = self.y + (self.y * rho).sum() * self.vol / mass
            r = torch.sqrt(x * x + y * y)
            h = r / radius
            w = torch.where(h < 1, h * (1.5 * h - 0.75 * h * h), torch.where(h < 2, 1.0 - 0.25 * (2.0 - h) ** 3, 1.0))
            dw = torch.where(h < 1, h * (3.0 - 2.25 * h), torch.where(h < 2, 0.75 * (2.0 - h) ** 2, 0.0))
            k = -mass * w / r**3 + mass * dw / (r * r * radius)
            self.gf = torch.stack([self.gf[0] + k * x, self.gf[1] + k * y, self.gf[2]])

    def step(self, c, u, p, dt, refresh=None):
        """One step of full length dt from (c, u, p) after its first state call."""
        c = self.ghosts(self.source(c, u, 0.5 * dt))
        c, p = self.state(c, u, p)
        c, u = self.velocity(c)
        old = c
        c = self.ghosts(self.flux(c, None, u, p, dt))
        c, p = self.state(c, u, p)
        c, u = self.velocity(c)
        c = self.ghosts(self.flux(c, old, u, p, dt))
        c, p = self.state(c, u, p)
        c, u = self.velocity(c)
        if refresh is not None:
            refresh(c[0])
        c = self.ghosts(self.source(c, u, 0.5 * dt))
        c, p = self.state(c, u, p)
        c, u = self.velocity(c)
        return c, u, p

    def run(self, c, u, p, steps, refresh=None):
        dts, last = [], 0.0
        for k in range(steps):
            c, p = self.state(c, u, p)
            dt = self.prm.cfl / float(self.rate(c, u, p).max())
            if k > 0:
                dt = min(dt, last * 1.1)
            last = dt
            c, u, p = self.step(c, u, p, dt, refresh)
            dts.append(dt)
        return c, u, p, np.array(dts)


def _neg(x):
    return torch.where(x < 0.0, x, 0.0)


def _larger(x, y):
    return torch.where(x > y, x, y)


def exact(case, seed):
    kind = case["kind"]
    # the batches take thousands of steps each, a grid at a time; the equation of state has tables in place of a formula
    if kind in ("tubes", "boxes") or case.get("eos"):
        return None
    prm, dev = _params(case), _device()
    P = _Plain(prm, dev)
    if kind == "adjoint":
        return _exact_adjoint(case, prm, P, seed, dev)
    c, v, p = _planes(case, prm, seed, dev)
    refresh = None
    if kind != "host":  # the device planes carry neither velocity nor pressure
        v = c[1:4] / c[0]
        p = _floor(c[4] - c[0] * 0.5 * v.square().sum(0), prm.small_eps) * P.gm1
        if case["gravity"] != "none":
            phi, point = _phi(prm, dev), case["gravity"] == "point"
            refresh = lambda rho: P.force(phi, rho, point)  # noqa: E731
            refresh(c[0])
    c, u, p, dts = P.run(c, v, p, case["steps"], refresh)
    if kind == "host":
        return {"cons": c.reshape(5, -1).T, "u": u.reshape(3, -1).T, "p": p.reshape(-1), "dts": dts}
    return {"cons": c, "dts": dts}


def _exact_adjoint(case, prm, P, seed, dev):
    from torch.utils.checkpoint import checkpoint

    rho, v, p = _fields(case, prm, seed, dev)
    target = _fields(case, prm, seed + 7919, dev)[0]
    rho, p = rho.clone().requires_grad_(), p.clone().requires_grad_()
    c = P.ghosts(torch.cat([rho[None], rho * v, (p / P.gm1 + rho * 0.5 * v.square().sum(0))[None]]))

    def one(c, dt):
        u = c[1:4] / c[0]
        pr = _floor(c[4] - c[0] * 0.5 * u.square().sum(0), prm.small_eps) * P.gm1
        return P.step(c, u, pr, dt)[0]

    last = 0.0
    for k in range(case["steps"]):
        with torch.no_grad():
            u = c[1:4] / c[0]
            pr = _floor(c[4] - c[0] * 0.5 * u.square().sum(0), prm.small_eps) * P.gm1
            dt = prm.cfl / float(P.rate(c, u, pr).max())
            dt = min(dt, last * 1.1) if k else dt
            last = dt
        c = checkpoint(one, c, dt, use_reentrant=False)
    loss = 0.5 * ((c[0] - target).square() * P.inside).sum()
    loss.backward()
    return {"rho": c[0].detach().reshape(-1), "grad_rho": rho.grad.reshape(-1), "grad_p": p.grad.reshape(-1)}
