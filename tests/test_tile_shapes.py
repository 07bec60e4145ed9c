"""The tiles of 32 columns (two rows to a wave) of the stage and flux kernels:
at sizes where the rule takes them, and at their edges, the bits are those of
the 64-column tiles (which the other tests hold against the oracle)."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from boxzyhydro_amd import ics
from boxzyhydro_amd import native as nv
from boxzyhydro_amd.hydro import HydroGrid
from boxzyhydro_amd.params import box_params

# grids (with ghosts) that take 32 x 16 tiles: one, two and three tiles wide, full and
# one column short, ragged rows; then ones that take 32 x 8
SIZES = [(36, 100, 70), (35, 340, 24), (100, 60, 44), (99, 62, 44), (36, 36, 36), (36, 53, 6), (36, 70, 5), (67, 13, 9)]


def _params(size, walls=""):
    no = {f"no_outflow_{s.lower()}{'l' if s.islower() else 'r'}": s in walls for s in "xXyYzZ"}
    return dataclasses.replace(box_params(8), nx=size[0], ny=size[1], nz=size[2], dx=0.5, dy=0.3, dz=0.7, **no)


def _run(prm, ic, mode, variant, phi=None, precision=None, steps=6):
    g = HydroGrid(prm, ic, precision=precision) if precision is not None else HydroGrid(prm, ic)
    if phi is not None:
        g.set_gravity(nv.BX_GRAV_POTENTIAL, phi)
    if variant is not None:
        g.tune(8, 3, variant)
    d = g.run(steps, mode=mode)
    out = g.download()
    g.close()
    return np.asarray(d), out


def _equal(a, b):
    assert np.array_equal(a[0].view(np.uint64), b[0].view(np.uint64))
    for k in ("cons", "u", "p"):
        assert np.array_equal(a[1][k].view(np.uint64), b[1][k].view(np.uint64)), k


@pytest.mark.gpu
@pytest.mark.parametrize("walls", ["", "xYz", "xXyYzZ"])
@pytest.mark.parametrize("size", SIZES)
def test_fp64_steps(size, walls):
    prm = _params(size, walls)
    ic = ics.box_ic(prm, seed=3, sigma_cells=1.0)
    want = _run(prm, ic, nv.BX_STEP_GRAPH, 11)
    _equal(_run(prm, ic, nv.BX_STEP_GRAPH, None), want)
    _equal(_run(prm, ic, nv.BX_STEP_EXACT, None), want)


@pytest.mark.gpu
@pytest.mark.parametrize("size", SIZES[:4])
def test_steps_with_gravity(size):
    prm = _params(size)
    ic = ics.box_ic(prm, seed=3, sigma_cells=1.0)
    phi = 0.05 * np.random.default_rng(2).standard_normal(prm.ngrid)
    _equal(_run(prm, ic, nv.BX_STEP_FUSED, None, phi), _run(prm, ic, nv.BX_STEP_FUSED, 11, phi))


@pytest.mark.gpu
@pytest.mark.parametrize("walls", ["", "xXyYzZ"])
@pytest.mark.parametrize("size", SIZES)
def test_mixed_steps(size, walls):
    prm = _params(size, walls)
    ic = ics.box_ic(prm, seed=3, sigma_cells=1.0)
    a, b = (_run(prm, ic, nv.BX_STEP_FUSED, v, precision=nv.BX_PREC_MIXED) for v in (None, 10))
    _equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("size", SIZES[:5])
def test_flux_with_varying_gamma(size):
    import os
    import sys

    sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
    import pyoracle as po

    prm = _params(size)
    ic = {k: v.copy() for k, v in ics.box_ic(prm, seed=4, sigma_cells=1.0).items()}
    ic["adindx"] = 1.2 + 0.5 * np.random.default_rng(7).random(prm.ngrid)
    g, o = HydroGrid(prm, ic), po.OracleGrid(prm, ic)
    g.dt = 0.05
    for avg in (0, 1):
        g.flux(avg)
        o.flux(avg, 0.05)
        assert np.array_equal(g.download()["cons"].view(np.uint64), np.asarray(o.cons).view(np.uint64))
    g.close()
