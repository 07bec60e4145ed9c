"""The Courant rate that the fused step keeps in slots: wherever the fastest
cell lies, every step's dt is the exact sequence's."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from boxzyhydro_amd import ics
from boxzyhydro_amd import native as nv
from boxzyhydro_amd.hydro import HydroGrid
from boxzyhydro_amd.params import box_params


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [0, 10, 11])
@pytest.mark.parametrize("cell", [(2, 2, 2), (65, 2, 3), (66, 9, 11), (67, 18, 2), (30, 10, 7), (3, 17, 6)])
def test_dt_wherever_the_fastest_cell_lies(cell, variant):
    prm = dataclasses.replace(box_params(8), nx=70, ny=21, nz=14)
    ic = {k: v.copy() for k, v in ics.box_ic(prm, seed=6, sigma_cells=2.0).items()}
    c = cell[0] + 70 * (cell[1] + 21 * cell[2])
    ic["cons"][c, 4] *= 40.0
    ic["p"][c] = (ic["cons"][c, 4] - 0.5 * (ic["cons"][c, 1:4] ** 2).sum() / ic["cons"][c, 0]) * (prm.gammafix - 1.0)
    runs = []
    for mode in (nv.BX_STEP_EXACT, nv.BX_STEP_FUSED, nv.BX_STEP_GRAPH):
        g = HydroGrid(prm, ic)
        if mode != nv.BX_STEP_EXACT:
            g.tune(8, 3, variant)
        runs.append([float(x) for x in g.run(7, mode=mode)])
        if mode != nv.BX_STEP_EXACT:
            assert g.step_counts()[0] >= 5  # fused steps were taken
        g.close()
    assert len(runs[0]) == 7 and runs[0] == runs[1] == runs[2]
