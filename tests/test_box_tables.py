"""What a batch of grids hands its kernel, for every combination of walls: the
tables, scratch and regions lie within their allocations and within each
other, and the ghost table of the fused steps is a pair of set_ghost_cells
calls.  On the CPU, over the stand-in HIP runtime."""
from __future__ import annotations

import fakehip

PROGRAM = """
import itertools
from boxzyhydro_amd.boxes import GridBatch
SIZES = [(5, 5, 6), (6, 6, 6), (9, 8, 7), (12, 7, 4), (5, 6, 1), (7, 11, 10)]
class Box(ctypes.Structure):
    _fields_ = ([(k, ctypes.c_int64) for k in ("n", "ic_off", "reg_off", "g_off", "x_off", "ng", "ns", "d2_off", "d2_scratch")]
                + [(k, ctypes.c_int32) for k in ("nd2", "nx", "ny", "nz", "flatz", "maxsteps")]
                + [("real", ctypes.c_double * 18)]
                + [(k, ctypes.c_int32) for k in ("fusable", "zlo", "zhi", "ly", "lz", "vol_pow2")]
                + [("ds_pow2", ctypes.c_int32 * 3), ("inv", ctypes.c_double * 5)])
POINTERS = ("boxes order queue ic reg gdst gsrc gsign gxsrc fsrc fsign d2dst d2src d2sign t_out steps_out status dtlog").split()
class Args(ctypes.Structure):
    _fields_ = [("nbox", ctypes.c_int32), ("maxlog", ctypes.c_int32)] + [(k, ctypes.c_void_p) for k in POINTERS]
grids = []
for size in SIZES:
    for w in itertools.product((False, True), repeat=6):
        walls = dict(zip(("no_outflow_xl", "no_outflow_xr", "no_outflow_yl", "no_outflow_yr", "no_outflow_zl",
                          "no_outflow_zr"), w))
        prm = dataclasses.replace(box_params(8), nx=size[0], ny=size[1], nz=size[2], **walls)
        grids.append((prm, ics.box_ic(prm, seed=0)))

def pair(gd, gs, gg, gx, n):
    # two set_ghost_cells calls on (cell, sign) of every cell
    cell, sign = np.arange(n), np.zeros(n, int)
    for _ in range(2):
        c0, s0 = cell.copy(), sign.copy()
        for d, s, g in zip(gd, gs, gg):
            k = s if s >= 0 else gx[-s - 1]
            cell[d], sign[d] = (c0[k], s0[k] ^ g)
    return cell, sign

chained = 0
def check(args):
    global chained
    a = ctypes.cast(args[0], ctypes.POINTER(Args)).contents
    assert a.nbox == len(grids)
    assert fake.fake_room(a.boxes) == a.nbox * ctypes.sizeof(Box)
    boxes = ctypes.cast(a.boxes, ctypes.POINTER(Box * a.nbox)).contents
    def table(ptr, off, cnt):
        assert off >= 0 and fake.fake_room(ptr) >= 4 * (off + cnt)
        return np.ctypeslib.as_array(ctypes.cast(ptr + 4 * off, ctypes.POINTER(ctypes.c_int32)), (cnt,)).copy() if cnt else np.zeros(0, int)
    reg = ic = 0
    for (prm, _), b in zip(grids, boxes):
        assert (b.nx, b.ny, b.nz, b.n) == (prm.nx, prm.ny, prm.nz, prm.ngrid)
        assert b.flatz == (b.nz < 6) and (b.zlo, b.zhi) == ((0, b.nz) if b.flatz else (2, b.nz - 2))
        assert b.reg_off == reg and b.ic_off == ic
        assert b.d2_scratch == 30 * b.n + 5 * b.ns  # behind the donors' snapshot
        reg += 30 * b.n + 5 * b.ns + 6 * b.nd2
        ic += 9 * b.n
        gd, gs, gg = (table(p, b.g_off, b.ng) for p in (a.gdst, a.gsrc, a.gsign))
        fs, fg = (table(p, b.g_off, b.ng) for p in (a.fsrc, a.fsign))
        gx = table(a.gxsrc, b.x_off, b.ns)
        z, y, x = np.unravel_index(np.arange(b.n), (b.nz, b.ny, b.nx))
        ghost = (x < 2) | (x > b.nx - 3) | (y < 2) | (y > b.ny - 3)
        if not b.flatz:
            ghost |= (z < 2) | (z > b.nz - 3)
        assert sorted(gd) == list(np.flatnonzero(ghost)) and len(set(gd)) == b.ng
        assert ((gs >= -b.ns) & (gs < b.n)).all() and ((gx >= 0) & (gx < b.n)).all()
        assert ghost[gx].all() and not ghost[gs[gs >= 0]].any()
        assert ((gg >= 0) & (gg < 8)).all()
        assert b.nd2 == 0 or b.ns > 0
        if not b.fusable:
            assert b.nd2 == 0
            continue
        chained += b.ns > 0
        assert ((fs >= 0) & (fs < b.n)).all() and not ghost[fs].any() and ((fg >= 0) & (fg < 8)).all()
        dd, ds, dg = (table(p, b.d2_off, b.nd2) for p in (a.d2dst, a.d2src, a.d2sign))
        assert b.nd2 <= 64 and len(set(dd)) == b.nd2
        cell, sign = pair(gd, gs, gg, gx, b.n)
        deep = [k for k in range(b.ng) if ghost[cell[gd[k]]]]
        assert [gd[k] for k in deep] == list(dd)
        for k in range(b.ng):
            c, s = cell[gd[k]], sign[gd[k]]
            if ghost[c]:  # the pre-pair value of another ghost, which its own pair gave it
                c, s = cell[c], s ^ sign[c]
            assert (fs[k], fg[k]) == (c, s), (prm, k)
        assert list(ds) == [fs[k] for k in deep] and list(dg) == [fg[k] for k in deep]
    assert fake.fake_room(a.reg) == 8 * reg and fake.fake_room(a.ic) == 8 * ic
    assert sorted(table(a.order, 0, a.nbox)) == list(range(a.nbox))
    for p in (a.t_out, a.steps_out, a.status):
        assert fake.fake_room(p) >= 4 * a.nbox

seen = []
def on_launch(name, grid, block, args):
    if "k_boxesI" in name:
        try:
            check(args)
            seen.append(name)
        except AssertionError:
            import traceback
            traceback.print_exc()
            os._exit(1)
launch(on_launch)
b = GridBatch(grids)
b.run(graph=False)
for waves in (4, 8, 16):
    b.tune(waves, 1)
    b.run(graph=False)
assert len(seen) == 4 and fake.fake_bad() == 0
print(chained, [("Lb1" in s) for s in seen])
"""


def test_tables_of_every_wall_combination(tmp_path):
    chained, builds = fakehip.run(tmp_path, PROGRAM).split(" ", 1)
    assert int(chained) > 100
    # chained grids take fused steps in the 8-wave build alone
    assert builds.strip() == "[True, False, True, False]"
