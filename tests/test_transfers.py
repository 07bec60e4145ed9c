"""Host transfers at the sizes where they change their route: small arrays
copied directly, large ones in chunks by several workers, chunks that do not
divide the array."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from boxzyhydro_amd.hydro import HydroGrid
from boxzyhydro_amd.params import box_params


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(9, 8, 7), (61, 47, 73), (100, 100, 27), (101, 99, 107), (128, 128, 64)])
def test_upload_download_round_trip(shape):
    prm = dataclasses.replace(box_params(8), nx=shape[0], ny=shape[1], nz=shape[2])
    rng = np.random.default_rng(sum(shape))
    n = prm.ngrid
    want = {"cons": rng.standard_normal((n, 5)), "u": rng.standard_normal((n, 3)), "p": rng.standard_normal(n),
            "adindx": rng.standard_normal(n)}
    g = HydroGrid(prm)
    for _ in range(2):  # the second pass reuses the pinned slots
        g.upload(want)
        got = g.download()
        for k, v in want.items():
            assert np.array_equal(got[k].view(np.uint64), v.view(np.uint64)), k
        want = {k: v[::-1].copy() for k, v in want.items()}
    old = g.download_cons_old()
    assert np.array_equal(old, want["cons"][::-1])
    g.close()
