"""The reverse kernels at ragged sizes: the same problem with its axes
permuted gives the same gradient (each axis is reversed by another kernel:
x in whole-wave shifts, y and z in marches whose lanes run over rows), any
chunk length gives the same bits, and donors of many ghosts sum them all."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from boxzyhydro_amd import ics
from boxzyhydro_amd.hydro import HydroGrid
from boxzyhydro_amd.params import box_params


def _gradient(shape, rho, p, u, tgt, dts, chunk, walls):
    """shape (nx, ny, nz); rho, p, tgt (nz, ny, nx); u (3, nz, ny, nx)."""
    import torch

    from boxzyhydro_amd.adjoint import AdjointStepper

    prm = dataclasses.replace(box_params(8), nx=shape[0], ny=shape[1], nz=shape[2],
                              **{f"no_outflow_{a}{e}": a + e in walls for a in "xyz" for e in "lr"})
    # ghosts as the step leaves them (the adjoint's forward takes regular states only)
    rho, p, u = rho.reshape(-1), p.reshape(-1), u.reshape(3, -1)
    cons = np.stack([rho, *(rho * u), p / (prm.gammafix - 1.0) + 0.5 * rho * (u * u).sum(0)], axis=1)
    h = HydroGrid(prm, {"cons": cons, "u": u.T, "p": p})
    h.set_ghost_cells()
    h.set_ghost_cells()
    cons = h.download()["cons"]
    h.close()
    ghost = ics.boundary_flags(prm).reshape(-1) > 0
    rho = np.where(ghost, cons[:, 0], rho)
    u = np.where(ghost, cons[:, 1:4].T / cons[:, 0], u)
    pg = (cons[:, 4] - 0.5 * rho * (u * u).sum(0)) * (prm.gammafix - 1.0)
    p = np.where(ghost, pg, p)
    st = AdjointStepper(prm, np.ascontiguousarray(u.T), 4, 2)
    if chunk:
        st.tune(chunk, chunk)
    dev = torch.device("cuda", 0)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a).reshape(-1), device=dev)
    out = st.forward(t(rho), t(p), dts=dts)
    inside = torch.as_tensor(ics.boundary_flags(prm).reshape(-1) == 0, device=dev)
    lam = (out - t(tgt)) * inside
    g = st.backward(lam)
    used = np.array(st.dts) if dts is None else dts
    res = [np.asarray(a.cpu().numpy()).reshape(shape[::-1]) for a in g]
    return res, used


@pytest.mark.gpu
@pytest.mark.parametrize("wall", [False, True])
@pytest.mark.parametrize("shape", [(6, 70, 9), (7, 12, 69), (68, 8, 7), (69, 21, 13)])
def test_gradient_under_permuted_axes(shape, wall):
    nx, ny, nz = shape
    prm = dataclasses.replace(box_params(8), nx=nx, ny=ny, nz=nz)
    a, b = (ics.box_ic(prm, seed=s, sigma_cells=1.5) for s in (2, 5))
    cube = lambda q: np.ascontiguousarray(q).reshape(nz, ny, nx)
    rho, p, tgt = cube(a["cons"][:, 0]), cube(a["p"]), cube(b["cons"][:, 0])
    u = 0.3 * np.stack([cube(b["cons"][:, 0]) - 1.0, cube(b["p"]) - cube(b["p"]).mean(), cube(a["p"]) - cube(a["p"]).mean()])
    print(f"adjoint axes {shape} wall={wall}", flush=True)
    axes = "xyz"
    (gr, gp), dts = _gradient(shape, rho, p, u, tgt, None, 0, ["xl"] if wall else [])
    assert np.abs(gr).max() > 1e-3
    for chunk in (1, 5, 64):
        (cr, cp), _ = _gradient(shape, rho, p, u, tgt, dts, chunk, ["xl"] if wall else [])
        assert cr.tobytes() == gr.tobytes() and cp.tobytes() == gp.tobytes(), chunk
    for turn in (1, 2):  # axis k of the turned problem is axis (k + turn) % 3 of this one
        order = [(2 - (2 - q + turn) % 3) for q in range(3)]  # array axes are z, y, x
        f = lambda q: np.transpose(q, order)
        shp = tuple(shape[(k + turn) % 3] for k in range(3))
        uu = np.stack([f(u[(k + turn) % 3]) for k in range(3)])
        side = axes[(0 - turn) % 3] + "l"
        (tr, tp), _ = _gradient(shp, f(rho), f(p), uu, f(tgt), dts, 0, [side] if wall else [])
        # the sums over directions and ghosts run in another order: rounding only
        for got, want in ((tr, gr), (tp, gp)):
            np.testing.assert_allclose(got, f(want), rtol=0, atol=1e-11 * np.abs(want).max())
