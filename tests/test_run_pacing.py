"""Runs of fused steps (undone as a whole when a step meets an irregular
branch): whatever the steps at which that happens, the work undone stays a
small part of the steps taken."""
from __future__ import annotations

import ctypes
import random
import subprocess

import pytest

from conftest import ROOT

# fused_loop's use of RunPacing over n steps of which bad[] are irregular: steps undone, runs, steps in runs
SRC = """
#include "bx_runs.h"
extern "C" void flow(const unsigned char *bad, int n, long *o)
{
    bx::RunPacing r;
    o[0] = o[1] = o[2] = 0;
    for (int k = 0; k < n;) {
        const int K = (n - k < bx::kChunkSteps ? n - k : bx::kChunkSteps) & ~1;
        if (r.may_run() && K >= 2) {
            bool ok = true;
            for (int i = 0; i < K; i++) ok = ok && !bad[k + i];
            o[1]++;
            if (ok) {
                r.regular(K);
                k += K;
                o[2] += K;
                continue;
            }
            o[0] += K;
            r.undone();
        }
        if (bad[k]) r.irregular();
        else r.regular(1);
        k++;
    }
}
"""


@pytest.fixture(scope="module")
def flow(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("runs") / "runs.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{ROOT}/boxzyhydro_amd/csrc", "-x", "c++", "-",
                    "-o", so], input=SRC, text=True, check=True)
    f = ctypes.CDLL(so).flow

    def call(bad):
        o = (ctypes.c_long * 3)()
        f(bytes(bad), len(bad), o)
        return tuple(o)
    return call


def test_regular_flow_takes_full_runs(flow):
    assert flow([0] * 3200) == (0, 100, 3200)


@pytest.mark.parametrize("period", [1, 2, 5, 16, 17, 31, 33, 40, 64, 65, 100, 200, 256, 300, 1000])
def test_steady_irregular_steps(flow, period):
    n = 20000
    undone, _, _ = flow([int(i % period == period - 1) for i in range(n)])
    assert undone <= n / 8 + 160


@pytest.mark.parametrize("seed", range(8))
def test_irregular_steps_at_random(flow, seed):
    rng = random.Random(seed)
    rate = rng.choice([0.003, 0.01, 0.03, 0.1, 0.3])
    n = 20000
    undone, _, _ = flow([int(rng.random() < rate) for _ in range(n)])
    assert undone <= n / 8 + 160


def test_runs_come_back(flow):
    assert flow([1] + [0] * 2000)[::2] == (32, 2001 - 33)
    # irregular steps in a row, then none
    undone, _, inside = flow([1] * 500 + [0] * 2000)
    assert undone <= 32 and inside >= 1960
