"""The flux subroutine where its route changes: gas without pressure, which
the tile takes on three axes and hands over on two, and grids thin in x, which
go cell by cell, against the oracle."""
from __future__ import annotations

import dataclasses
import os
import sys

import numpy as np
import pytest

import fakehip
from boxzyhydro_amd import ics
from boxzyhydro_amd.hydro import HydroGrid
from boxzyhydro_amd.params import box_params

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import pyoracle as po  # noqa: E402
from test_ang_tile import _check as check_ang  # noqa: E402  (the oracle has no flux_ang)


def _same(a, b):
    a, b = np.asarray(a), np.asarray(b)
    nan = np.isnan(a)
    return np.array_equal(nan, np.isnan(b)) and np.array_equal(a[~nan].view(np.uint64), b[~nan].view(np.uint64))


def _fluxes(prm, ic, dt=0.05):
    g, o = HydroGrid(prm, ic), po.OracleGrid(prm, ic)
    g.dt = dt
    for avg in (0, 1):
        g.copy_old()
        o.copy_old()
        g.flux(avg)
        o.flux(avg, dt)
        assert _same(g.download()["cons"], o.cons), avg
    g.close()


@pytest.mark.gpu
@pytest.mark.parametrize("ang", [False, True])
@pytest.mark.parametrize("still", [0.0, 0.2])  # two still cells side by side: 0/0
@pytest.mark.parametrize("share,zero", [(0.1, 0.0), (0.6, 0.0), (1.0, 0.0), (0.3, -0.0)])
@pytest.mark.parametrize("size", [(36, 20, 14), (69, 13, 9), (24, 14, 4)])
def test_gas_without_pressure(size, share, zero, still, ang):
    prm = dataclasses.replace(box_params(8), nx=size[0], ny=size[1], nz=size[2], dx=0.5, dy=0.3, dz=0.7,
                              small_eps=0.0, fluxangmom=ang, yoffset=0.1 if ang else 0.0)
    rng = np.random.default_rng(size[0])
    ic = {k: v.copy() for k, v in ics.box_ic(prm, seed=4, sigma_cells=1.0).items()}
    cold = rng.random(prm.ngrid) < share
    ic["p"][cold] = zero
    ic["cons"][cold, 4] = 0.5 * ic["cons"][cold, 0] * (ic["u"][cold] ** 2).sum(1)
    rest = rng.random(prm.ngrid) < still
    ic["u"][rest] = 0.0
    ic["cons"][rest, 1:4] = 0.0
    print("cold", size, share, zero, still, ang, flush=True)
    if ang:
        check_ang(prm, ic)
    else:
        _fluxes(prm, ic)


ROUTE = """
from boxzyhydro_amd.hydro import make_params
names = []
launch(lambda name, g, b, args: names.append(name))
for nx, ny, nz, ang in CASES:
    p = make_params(dataclasses.replace(box_params(8), nx=nx, ny=ny, nz=nz, fluxangmom=ang))
    h = ctypes.c_void_p()
    nv.check(nv.lib().bx_create(ctypes.byref(p), 0, ctypes.byref(h)), "create")
    names.clear()
    nv.check(nv.lib().bx_flux(h, 0, 1e-6), "flux")
    print(int(any("k_stage" in x for x in names)), end=" ")
    nv.lib().bx_destroy(h)
"""


def test_route_of_thin_grids(tmp_path):
    thin = [(5, 132, 132, False), (6, 32772, 1, False), (5, 132, 132, True)]
    tiled = [(5, 132, 131, False), (7, 260, 132, False), (6, 260, 132, True), (6, 32771, 1, False)]
    out = fakehip.run(tmp_path, ROUTE.replace("CASES", repr(thin + tiled)))
    assert out.split() == ["0"] * len(thin) + ["1"] * len(tiled)


@pytest.mark.gpu
@pytest.mark.parametrize("ang", [False, True])
@pytest.mark.parametrize("size", [(5, 132, 133), (6, 200, 173), (6, 16390, 2)])
def test_thin_grids(size, ang):
    prm = dataclasses.replace(box_params(8), nx=size[0], ny=size[1], nz=size[2], dx=0.5, dy=0.3, dz=0.7,
                              fluxangmom=ang, yoffset=0.1 if ang else 0.0)
    ic = {k: v.copy() for k, v in ics.box_ic(prm, seed=4, sigma_cells=1.0).items()}
    print("thin", size, ang, flush=True)
    if ang:
        check_ang(prm, ic)
    else:
        _fluxes(prm, ic)
