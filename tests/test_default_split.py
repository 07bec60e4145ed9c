"""The work split that the library's rule chooses can be named, given to
bx_tune and found by the autotuner, which must not leave a grid slower than an
untuned one."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

import fakehip
from boxzyhydro_amd import autotune, ics
from boxzyhydro_amd import native as nv
from boxzyhydro_amd.hydro import HydroGrid
from boxzyhydro_amd.params import box_params

HOST = """
from boxzyhydro_amd.hydro import HydroGrid
out = []
for precision in (nv.BX_PREC_FP64, nv.BX_PREC_MIXED):
    for size in ((36, 100, 70), (260, 260, 260), (100, 100, 100), (36, 36, 36), (404, 8, 4), (5, 5, 1), (67, 13, 9)):
        prm = dataclasses.replace(box_params(8), nx=size[0], ny=size[1], nz=size[2])
        g = HydroGrid(prm, precision=precision)
        split = g.default_split()
        assert split[0] >= 1 and 1 <= split[1] <= size[2] and 10 <= split[2] <= 13, (size, split)
        g.tune(*split)  # the rule's choice is accepted
        g.tune(8, 3, 0)
        assert g.default_split() == split
        out.append(split[2])
        for bad in (2, 3, 5, 9, 14) + ((13,) if precision else ()):
            try:
                g.tune(8, 3, bad)
                raise SystemExit(f"variant {bad} accepted")
            except nv.BoxzyError:
                pass
print(sorted(set(out)))
"""


def test_rule_is_a_valid_argument_of_tune(tmp_path):
    assert fakehip.run(tmp_path, HOST).strip() == "[10, 11, 12, 13]"


class _Grid:
    """A grid whose own split is the fastest."""

    def default_split(self):
        return (64, 7, 13)

    def tune(self, *split):
        self.split = split

    def run(self, steps, mode=None, endtime=None):
        self.clock += steps * (1.0 if self.split == (64, 7, 13) else 2.0)

    def sync(self):
        pass


def test_autotuner_times_the_default(monkeypatch):
    g = _Grid()
    g.clock, g.split = 0.0, None
    monkeypatch.setattr(autotune.time, "perf_counter", lambda: g.clock)
    best, results = autotune.tune_step(g)
    assert best == g.split == (64, 7, 13) and results[0][0] == best
    assert [c for c, _ in results[1:]] == autotune.DEFAULT_CANDIDATES
    best, results = autotune.tune_step(g, [(16, 16, 0), (16, 16, 1)])  # a caller's own list stays as it is
    assert [c for c, _ in results] == [(16, 16, 0), (16, 16, 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [12, 13])
@pytest.mark.parametrize("chunk", [1, 3, 64])
def test_tuned_narrow_tiles(variant, chunk):
    prm = dataclasses.replace(box_params(8), nx=67, ny=41, nz=14, dy=0.3, no_outflow_xl=True, no_outflow_yr=True)
    ic = ics.box_ic(prm, seed=5, sigma_cells=1.0)
    got = []
    for split in (None, (8, chunk, variant)):
        g = HydroGrid(prm, ic)
        if split:
            g.tune(*split)
        d = g.run(6, mode=nv.BX_STEP_GRAPH)
        got.append((np.asarray(d), g.download()))
        g.close()
    assert np.array_equal(got[0][0].view(np.uint64), got[1][0].view(np.uint64))
    for k in ("cons", "u", "p"):
        assert np.array_equal(got[0][1][k].view(np.uint64), got[1][1][k].view(np.uint64)), k
