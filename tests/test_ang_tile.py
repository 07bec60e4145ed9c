"""The tiled flux of the angular-momentum form (flux_ang.f90:6-618) against the
same formulas written out here over whole arrays, one call at a time and bit
for bit: sizes at the edges of tiles, a cell on the axis (where the projection
divides by r = 0), a gamma that varies, and values that the tile hands over to
the cell-by-cell kernel."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from boxzyhydro_amd import ics
from boxzyhydro_amd.hydro import HydroGrid
from boxzyhydro_amd.params import box_params


def _vmax(a, b):
    return np.where(a > b, a, b)


def _vmin(a, b):
    return np.where(a < b, a, b)


def _slope(c0, c1, c2):
    x1, x2, x3 = 1.25 * (c1 - c0), 0.5 * (c2 - c0), 1.25 * (c2 - c1)
    up, dn = (x1 > 0) & (x2 > 0) & (x3 > 0), (x1 < 0) & (x2 < 0) & (x3 < 0)
    return np.where(up, _vmin(x1, _vmin(x2, x3)), np.where(dn, _vmax(x1, _vmax(x2, x3)), 0.0))


@np.errstate(all="ignore")
def flux_ang(prm, cons, old, u, p, ad, avg, dt):
    """(cons, cons_old) after flux(avg), the ghosts before their fill."""
    nx, ny, nz = prm.nx, prm.ny, prm.nz
    flat = nz < 6
    cube = lambda q: np.ascontiguousarray(q).reshape(nz, ny, nx)
    q = [cube(cons[:, k]) for k in range(5)]
    o = [cube(old[:, k]) for k in range(5)]
    v = [cube(u[:, k]) for k in range(3)]
    p, ad = cube(p), cube(ad)
    ds = (prm.dx, prm.dy, prm.dz)
    x = (ds[0] * (np.arange(1, nx + 1) - (nx + 1.0) / 2.0))[None, None, :]
    y = (ds[1] * (np.arange(1, ny + 1) - (ny + 1.0) / 2.0))[None, :, None]
    yo = y + prm.yoffset
    r, ro = np.sqrt(x * x + y * y), np.sqrt(x * x + yo * yo)

    def to(m1, m2):
        return (m1 * x + m2 * yo) / ro, x * m2 - yo * m1

    def back(rm, am):
        return (rm * x - am * yo / ro) / ro, (rm * yo + am * x / ro) / ro

    q[1], q[2] = to(q[1], q[2])
    if avg:
        o[1], o[2] = to(o[1], o[2])
    edge = lambda n: np.isin(np.arange(n), [0, 1, n - 2, n - 1])
    ghost = ((edge(nz) & (not flat))[:, None, None] | edge(ny)[None, :, None] | edge(nx)[None, None, :])
    eps = _vmax(q[4] - 0.5 * q[0] * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]), prm.small_eps)
    snd = np.sqrt(p * ad / q[0])
    fields = [q[0], v[0], v[1], v[2], p, eps, ad, q[1], q[2]]
    tot = None
    for d, area in ((0, ds[1] * ds[2]), (1, ds[0] * ds[2]), (2, ds[1] * ds[0])):
        ax = 2 - d
        lower = (lambda a: a) if d == 2 and flat else (lambda a: np.roll(a, 1, ax))
        upper = (lambda a: a) if d == 2 and flat else (lambda a: np.roll(a, -1, ax))
        lp, lm = _vmax(v[d] + snd, 0.0) * dt / ds[d], _vmin(v[d] - snd, 0.0) * dt / ds[d]
        zc = 0.0 * (dt * 0.5 / ds[d])
        mi, pl = [], []
        for k, f in enumerate(fields):
            s = np.where(ghost, 0.0, _slope(lower(f), f, upper(f)))
            a, b = f + 0.5 * (-1.0 - lm) * s, f + 0.5 * (1.0 - lp) * s
            mi.append(a + zc if k < 7 else a)
            pl.append(b + zc if k < 7 else b)

        def hll(L, R):
            def side(S):
                dd, v0, v1, v2, pp, e, g, rm, am = S
                st = [dd, rm, am, dd * v2, e + 0.5 * dd * (v0 * v0 + v1 * v1 + v2 * v2)]
                vd = (v0, v1, v2)[d]
                if d == 0:
                    pr = (pp * x / r, -(pp * y), 0.0)
                elif d == 1:
                    pr = (pp * y / r, pp * x, 0.0)
                else:
                    pr = (0.0, 0.0, pp)
                fl = [st[0] * vd] + [pr[k] + st[1 + k] * vd for k in range(3)] + [(st[4] + pp) * vd]
                return st, fl, vd, np.sqrt(g * pp / dd)

            sl, fl, vl, cl = side(L)
            sr, fr, vr, cr = side(R)
            ap = _vmax(_vmax(0.0, vr + cr), vl + cl)
            am = _vmax(_vmax(0.0, -(vr - cr)), -(vl - cl))
            return [(ap * fl[i] + am * fr[i] - ap * am * (sr[i] - sl[i])) / (ap + am) for i in range(5)]

        f0 = hll([lower(a) for a in pl], mi)
        f1 = hll(pl, [upper(a) for a in mi])
        term = [area * (f1[i] - f0[i]) for i in range(5)]
        tot = term if tot is None else [tot[i] + term[i] for i in range(5)]
    ft = [np.where(ghost, 0.0, -(t * dt / (ds[0] * ds[1] * ds[2]))) for t in tot]
    U = [q[i] + ft[i] if avg == 0 else 0.5 * (o[i] + q[i] + ft[i]) for i in range(5)]
    U[1], U[2] = back(U[1], U[2])
    if avg:
        o[1], o[2] = back(o[1], o[2])
    U[0] = _vmax(U[0], prm.small_rho)
    U[4] = np.where(U[4] < 0.0, 0.5 * (U[1] * U[1] + U[2] * U[2] + U[3] * U[3]) / U[0] + prm.small_eps, U[4])
    flat_ = lambda w: np.stack([a.ravel() for a in w], axis=1)
    return flat_(U), flat_(o), ~ghost.ravel()


def _same(a, b):
    nan = np.isnan(a)
    return np.array_equal(nan, np.isnan(b)) and np.array_equal(a[~nan].view(np.uint64), b[~nan].view(np.uint64))


def _check(prm, ic, dt=0.03):
    g = HydroGrid(prm, ic)
    g.dt = dt
    g.copy_old()
    for avg in (0, 1):
        s, old = g.download(), g.download_cons_old()
        want, wold, inner = flux_ang(prm, s["cons"], old, s["u"], s["p"], s["adindx"], avg, dt)
        g.flux(avg)
        assert _same(g.download()["cons"][inner], want[inner]), avg
        if avg:
            assert _same(g.download_cons_old(), wold)
    g.close()


def _params(shape, **over):
    return dataclasses.replace(box_params(8), nx=shape[0], ny=shape[1], nz=shape[2], fluxangmom=True,
                               **{"dx": 0.5, "dy": 0.3, "dz": 0.7, **over})


def _ic(prm, gamma):
    ic = {k: v.copy() for k, v in ics.box_ic(prm, seed=4, sigma_cells=1.0).items()}
    if gamma:
        ic["adindx"] = 1.2 + 0.5 * np.random.default_rng(7).random(prm.ngrid)
    return ic


@pytest.mark.gpu
@pytest.mark.parametrize("gamma", [False, True])
@pytest.mark.parametrize("shape", [(6, 6, 6), (20, 14, 11), (68, 12, 9), (69, 9, 4), (133, 6, 14), (70, 21, 44)])
def test_flux_ang_matches_formulas(shape, gamma):
    for over in ({"yoffset": 0.25}, {"dx": 0.5, "dy": 0.5, "dz": 0.5}):
        prm = _params(shape, **over)
        _check(prm, _ic(prm, gamma))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(15, 11, 9), (67, 13, 4)])
def test_flux_ang_with_a_cell_on_the_axis(shape):
    prm = _params(shape)
    _check(prm, _ic(prm, False))
    prm = _params(shape, yoffset=0.25)
    _check(prm, _ic(prm, False))


@pytest.mark.gpu
@pytest.mark.parametrize("field,value", [("p", -1.0), ("p", np.nan), ("mx", np.inf), ("my", 1e200), ("mx", np.nan)])
def test_flux_ang_hands_over_values_outside_its_range(field, value):
    prm = _params((24, 14, 9), vlimit=1e300)
    ic = _ic(prm, False)
    c = 9 + 7 * 24 + 4 * 24 * 14
    if field == "p":
        ic["p"][c] = value
    else:
        ic["cons"][c, 1 if field == "mx" else 2] = value
    _check(prm, ic)
