"""The tiled flux of the call-by-call path (bx_flux) against the oracle, one
call at a time: odd sizes at the edges of tiles and chunks, walls, a gamma
that varies from cell to cell, and values that the tile hands over to the
cell-by-cell kernel (NaN, infinities, zero and negative pressures, numbers
whose products overflow)."""
from __future__ import annotations

import dataclasses
import os
import sys

import numpy as np
import pytest

from boxzyhydro_amd import ics
from boxzyhydro_amd.hydro import HydroGrid
from boxzyhydro_amd.params import box_params

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import pyoracle as po  # noqa: E402


def _same(a, b):
    a, b = np.asarray(a), np.asarray(b)
    nan = np.isnan(a)
    return np.array_equal(nan, np.isnan(b)) and np.array_equal(a[~nan].view(np.uint64), b[~nan].view(np.uint64))


def _run(prm, ic, dt=0.05):
    g, o = HydroGrid(prm, ic), po.OracleGrid(prm, ic)
    g.dt = dt
    bad = []
    for name in ("copy_old", "flux0", "set_ghost_cells", "state", "velocity", "flux1", "set_ghost_cells", "state"):
        if name.startswith("flux"):
            g.flux(int(name[4]))
            o.flux(int(name[4]), dt)
        else:
            getattr(g, name)()
            getattr(o, name)()
        out = g.download()
        bad += [(name, k) for k in ("cons", "u", "p") if not _same(out[k], getattr(o, k))]
    g.close()
    assert not bad, bad[:6]


def _ic(prm, seed=4):
    ic = ics.box_ic(prm, seed=seed, sigma_cells=1.0)
    return {k: v.copy() for k, v in ic.items()}


@pytest.mark.gpu
@pytest.mark.parametrize("walls", [False, True])
@pytest.mark.parametrize("shape", [(5, 5, 6), (20, 13, 11), (69, 12, 9), (70, 21, 44), (133, 6, 3), (36, 36, 36)])
def test_flux_matches_oracle(shape, walls):
    no = {f"no_outflow_{a}{s}": walls for a in "xyz" for s in "lr"}
    prm = dataclasses.replace(box_params(8), nx=shape[0], ny=shape[1], nz=shape[2], dx=0.5, dy=0.3, dz=0.7, **no)
    _run(prm, _ic(prm))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(20, 13, 11), (70, 21, 14), (40, 9, 4)])
def test_flux_varying_gamma(shape):
    prm = dataclasses.replace(box_params(8), nx=shape[0], ny=shape[1], nz=shape[2])
    ic = _ic(prm)
    ic["adindx"] = 1.2 + 0.5 * np.random.default_rng(7).random(prm.ngrid)
    g, o = HydroGrid(prm, ic), po.OracleGrid(prm, ic)
    g.dt = 0.05
    for avg in (0, 1):  # no state() between: adindx stays the uploaded one
        g.flux(avg)
        o.flux(avg, 0.05)
        assert _same(g.download()["cons"], o.cons)
    g.close()


@pytest.mark.gpu
@pytest.mark.parametrize("nz", [4, 12])
@pytest.mark.parametrize("field,value", [("p", -1.0), ("p", 0.0), ("p", np.nan), ("E", np.inf), ("rho", -0.3),
                                         ("u", np.nan), ("u", 1e200), ("E", -np.inf)])
def test_flux_hands_over_values_outside_its_range(field, value, nz):
    prm = dataclasses.replace(box_params(8), nx=24, ny=14, nz=nz, vlimit=1e300)
    ic = _ic(prm)
    c = 9 + 7 * 24 + (nz // 2) * 24 * 14
    if field == "p":
        ic["p"][c] = value
    elif field == "u":
        ic["u"][c, 1] = value
    else:
        ic["cons"][c, 0 if field == "rho" else 4] = value
    _run(prm, ic)
