"""How the cells of a tube are divided among a gang's workgroups: each cell of
the row belongs to one member and none lies past the row's end, also where the
last members have no segment.  A member reading past its row would take the
next tube's velocity into this tube's first dt, or read past the allocation."""
from __future__ import annotations

import ctypes
import subprocess

import numpy as np
import pytest

from boxzyhydro_amd import ics
from boxzyhydro_amd.batch import TubeBatch
from conftest import ROOT

SRC = """
#include "bx_gang.h"
extern "C" void gang_range(int nx, int member, int p, int *o)
{
    const bx::Range r = bx::tube_range(nx, member, p);
    const int v[7] = {r.nseg, r.s0, r.s1, r.c_lo, r.c_hi, r.left, r.right};
    for (int i = 0; i < 7; i++) o[i] = v[i];
}
"""


@pytest.fixture(scope="module")
def gang_range(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("gang") / "range.so")
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-D__host__=", "-D__device__=",
                    f"-I{ROOT}/boxzyhydro_amd/csrc", "-x", "c++", "-", "-o", so], input=SRC, text=True, check=True)
    f = ctypes.CDLL(so).gang_range

    def call(nx, member, p):
        o = (ctypes.c_int * 7)()
        f(nx, member, p, o)
        return tuple(o)
    return call


@pytest.mark.parametrize("p", [1, 2, 3, 4, 5, 6, 8, 15, 64])
def test_members_share_the_row(gang_range, p):
    for nx in list(range(8, 1300)) + [4099, 4100, 4159, 65536]:
        nseg = (nx - 4 + 59) // 60
        cell = seg = 0
        ranges = [gang_range(nx, m, p) for m in range(p)]
        for m, (ns, s0, s1, lo, hi, left, right) in enumerate(ranges):
            assert ns == nseg and s0 == seg and s0 <= s1 <= nseg, (nx, m)
            assert lo == cell and lo <= hi <= nx, (nx, m)
            if s0 < s1:
                assert lo == (0 if s0 == 0 else 2 + 60 * s0) and hi == (nx if s1 == nseg else 2 + 60 * s1), (nx, m)
            else:
                assert lo == hi, (nx, m)
            # a shared edge has a segment on either side
            assert bool(left) == (s0 < s1 and m > 0) and bool(right) == (s1 < nseg), (nx, m)
            assert not right or ranges[m + 1][1] < ranges[m + 1][2], (nx, m)
            cell, seg = hi, s1
        assert cell == nx and seg == nseg, nx


def _pair(length):
    (prm, row), = ics.riemann_tubes(1, seed=3, lmin=length, lmax=length, endtime=0.01)
    (fprm, frow), = ics.riemann_tubes(1, seed=4, lmin=64, lmax=64, endtime=0.01)
    frow = {k: v.copy() for k, v in frow.items()}
    frow["u"][:, 0] = 500.0  # the frame's rate takes u as it was set up
    return (prm, row), (fprm, frow)


@pytest.mark.gpu
@pytest.mark.parametrize("members,length", [(6, 721), (6, 837), (15, 961), (4, 541)])
def test_neighbour_does_not_change_dt(members, length):
    tubes = list(_pair(length))
    out = []
    for m, n in ((0, 0), (members, 2)):
        b = TubeBatch(tubes)
        b.gang(m, n)
        b.log_dt(64)
        b.run(maxsteps=20)
        b.sync()
        assert b.gang_fallbacks() == 0
        out.append((b.dts(), b.result()))
    for i in range(2):
        assert np.array_equal(out[0][0][i].view(np.uint64), out[1][0][i].view(np.uint64)), i
        for k in ("cons", "u", "p"):
            assert np.array_equal(out[0][1][i][k].view(np.uint64), out[1][1][i][k].view(np.uint64)), (i, k)


@pytest.mark.gpu
def test_no_step_leaves_the_set_up():
    slow, fast = _pair(721)
    for tubes in ([slow, fast], [fast, slow]):
        b = TubeBatch(tubes)
        b.gang(6, 2)
        b.run(maxsteps=0)
        b.sync()
        for (prm, row), r in zip(tubes, b.result()):
            assert r["steps"] == 0
            inner = slice(2, prm.nx - 2)
            for k in ("cons", "u", "p"):
                assert np.array_equal(np.asarray(r[k])[inner], np.asarray(row[k])[inner]), k
