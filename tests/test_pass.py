"""The fused pointwise passes of the exact step (BX_STEP_EXACT) against the
same calls one by one on a second grid, bit for bit: several steps (so that a
step's last pass starts the next one), interior-only and chained ghost tables,
low densities, the velocity limit, tables, uniform and per-cell forces."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from boxzyhydro_amd import ics
from boxzyhydro_amd import native as nv
from boxzyhydro_amd.hydro import HydroGrid, step_sequence
from boxzyhydro_amd.params import box_params


def _walls(sides):
    return {f"no_outflow_{s}": True for s in sides}


CASES = {
    "outflow": ({}, (21, 13, 9)),
    "flat_z": ({}, (37, 18, 4)),
    "one_wall": (_walls(["xl"]), (17, 12, 8)),
    "all_walls": (_walls(["xl", "xr", "yl", "yr", "zl", "zr"]), (12, 13, 14)),
    "clamped": (dict(vlimit=0.05), (16, 9, 10)),
    "tables": (dict(H2STAT=0, NEOS_RHO=200, dTk_eos=10.0, tk_bgrnd=3.0), (19, 12, 11)),
    "tables_walls": (dict(H2STAT=0, NEOS_RHO=200, dTk_eos=10.0, tk_bgrnd=3.0, **_walls(["xl", "yr"])), (12, 11, 10)),
    "angular": (dict(fluxangmom=True, yoffset=0.3), (20, 16, 9)),
    "largest_block": ({}, (68, 66, 7)),
}


@pytest.mark.gpu
@pytest.mark.parametrize("thin", [False, True])
@pytest.mark.parametrize("name", sorted(CASES))
def test_exact_steps_equal_the_calls(name, thin):
    over, (nx, ny, nz) = CASES[name]
    prm = dataclasses.replace(box_params(8), nx=nx, ny=ny, nz=nz, **over)
    ic = {k: v.copy() for k, v in ics.box_ic(prm, seed=3, sigma_cells=1.5).items()}
    if thin:  # cells on either side of the density below which state() sets the pressure
        low = np.random.default_rng(1).random(prm.ngrid) < 0.3
        ic["cons"][low] *= 5e-5 / ic["cons"][low, :1]
    a, b = HydroGrid(prm, ic), HydroGrid(prm, ic)
    print(f"passes {name} thin={thin}", flush=True)
    da = a.run(4, mode=nv.BX_STEP_EXACT)
    db, _ = step_sequence(b, 4, prm.endtime)
    assert [float(x) for x in da] == [float(x) for x in db]
    oa, ob = a.download(), b.download()
    oa["old"], ob["old"] = a.download_cons_old(), b.download_cons_old()
    if name.startswith("tables"):
        oa["muc"], ob["muc"] = a.download_muc(), b.download_muc()
    for k in oa:
        assert oa[k].tobytes() == ob[k].tobytes(), k
    a.close()
    b.close()
