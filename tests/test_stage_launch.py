"""Launch rules of the fused stage kernels: chunks of any length, 64 x 4 tiles
where 64 x 8 ones leave the chip idle, ghost cells read from their donors, dt
formed in stage 1.  Each mode against the exact call sequence, bit for bit, at
the sizes where a tile, a chunk or a wall can go wrong."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from boxzyhydro_amd import ics
from boxzyhydro_amd import native as nv
from boxzyhydro_amd.hydro import HydroGrid
from boxzyhydro_amd.params import box_params

SHAPES = [(1, 1, 2), (2, 3, 5), (16, 16, 16), (33, 9, 7), (64, 8, 4), (65, 17, 3), (130, 12, 40), (9, 70, -3)]
WALLS = ["", "xX", "yZ", "xXyYzZ"]


def _params(shape, walls):
    x, y, z = shape
    no = {f"no_outflow_{s.lower()}{'l' if s.islower() else 'r'}": s in walls for s in "xXyYzZ"}
    return dataclasses.replace(box_params(8), nx=x + 4, ny=y + 4, nz=-z if z < 0 else z + 4, dx=0.5, dy=0.3, dz=0.7, **no)


@pytest.mark.gpu
@pytest.mark.parametrize("walls", WALLS)
@pytest.mark.parametrize("shape", SHAPES)
def test_modes_match_exact(shape, walls):
    prm = _params(shape, walls)
    ic = ics.box_ic(prm, seed=3, sigma_cells=1.0)
    res = {}
    for mode in (nv.BX_STEP_EXACT, nv.BX_STEP_FUSED, nv.BX_STEP_GRAPH):
        g = HydroGrid(prm, ic)
        d = [g.run(k, mode=mode) for k in (1, 9, 1, 4)]  # runs of pairs, odd steps and single steps
        res[mode] = (np.concatenate(d), g.download(), g.time, g.dtold)
        g.close()
    want = res[nv.BX_STEP_EXACT]
    assert len(want[0]) == 15
    for mode in (nv.BX_STEP_FUSED, nv.BX_STEP_GRAPH):
        got = res[mode]
        assert np.array_equal(got[0].view(np.uint64), want[0].view(np.uint64))
        for k in ("cons", "u", "p"):
            assert np.array_equal(got[1][k].view(np.uint64), want[1][k].view(np.uint64)), (mode, k)
        assert got[2:] == want[2:]
