"""Batched tubes at the lengths where the work changes its form: one to
seventeen segments of 60 cells, partly filled last segments, tubes that a
workgroup holds in registers and longer ones that go through the rows, gangs
with members of few or no segments.  Every form against the oracle."""
from __future__ import annotations

import os
import sys

import numpy as np
import pytest

from boxzyhydro_amd import ics
from boxzyhydro_amd.batch import TubeBatch, grid_of_row

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import pyoracle as po  # noqa: E402

LENGTHS = [4, 5, 58, 59, 60, 61, 62, 63, 119, 121, 181, 239, 241, 479, 481, 482, 961]


@pytest.fixture(scope="module")
def problem():
    tubes, want = [], []
    for i, length in enumerate(LENGTHS):
        (prm, row), = ics.riemann_tubes(1, seed=i, lmin=length, lmax=length, endtime=min(0.1, 6.0 / length))
        tubes.append((prm, row))
        o = po.OracleGrid(prm, grid_of_row(prm, row))
        dts, _ = o.run(1_000_000)
        donor = np.clip(np.arange(prm.nx), 2, prm.nx - 3)
        want.append({"steps": len(dts), **{k: getattr(o, k).reshape(prm.shape + (-1,))[0, 2][donor]
                                           for k in ("cons", "u", "p")}})
    return tubes, want


@pytest.mark.gpu
@pytest.mark.parametrize("gang", [(0, 0), (2, 17), (3, 17), (6, 17), (15, 17)])
@pytest.mark.parametrize("waves", [0, 4, 8, 16])
def test_forms_match_oracle(problem, waves, gang):
    tubes, want = problem
    b = TubeBatch(tubes)
    if waves:
        b.tune(waves, 1)
    b.gang(*gang)
    for _ in range(2):
        b.run(graph=True)
        b.sync()
        for i, (r, w) in enumerate(zip(b.result(), want)):
            assert r["steps"] == w["steps"], (LENGTHS[i], r["steps"], w["steps"])
            for k in ("cons", "u", "p"):
                assert np.array_equal(np.asarray(r[k]).reshape(w[k].shape).view(np.uint64),
                                      np.ascontiguousarray(w[k]).view(np.uint64)), (LENGTHS[i], k)
    assert b.gang_fallbacks() == 0
