"""Host transfers where no pinned memory is to be had: the chunks that the
device forms must fit the staging buffer.  On the CPU, over the stand-in HIP
runtime; the launches are carried out here."""
from __future__ import annotations

import pytest

import fakehip

# k_boxes_rows and the planes <-> rows kernels, as the library launches them
KERNELS = """
sizes = []
def rows_of(ptr, cnt):
    assert fake.fake_room(ptr) >= 8 * cnt, (fake.fake_room(ptr), 8 * cnt)
    sizes.append(8 * cnt)
    return np.ctypeslib.as_array(ctypes.cast(ptr, ctypes.POINTER(ctypes.c_double)), (cnt,))
failed = []
def on_launch(name, grid, block, args):
    try:
        go(name, args)
    except AssertionError as e:
        failed.append((name, e))
def planes_of(ptr, k, n):
    return np.ctypeslib.as_array(ctypes.cast(ptr, ctypes.POINTER(ctypes.c_double)), (k, n))
"""

BOXES = KERNELS + """
from boxzyhydro_amd.boxes import GridBatch
def go(name, args):
    if "k_boxes_rows" in name:
        first, k = arg(args, 4, ctypes.c_int), arg(args, 5, ctypes.c_int)
        e0, cnt = arg(args, 6, ctypes.c_int64), arg(args, 7, ctypes.c_int64)
        rows_of(arg(args, 8, ctypes.c_void_p), cnt)[:] = first * 1e9 + e0 + np.arange(cnt)
launch(on_launch, 1 << 20)
prm = dataclasses.replace(box_params(8), nx=EDGE, ny=EDGE, nz=EDGE)
ic = ics.box_ic(prm, seed=0)
b = GridBatch([(prm, ic), (prm, ic)])
r = b.result()
assert not failed, failed
got = np.concatenate([x["cons"].reshape(-1) for x in r])
assert np.array_equal(got, np.arange(got.size)), got[:9]
for key, first in (("u", 5), ("p", 8)):
    got = np.concatenate([x[key].reshape(-1) for x in r])
    assert np.array_equal(got, first * 1e9 + np.arange(got.size))
assert fake.fake_bad() == 0
print(max(sizes))
"""

GRID = KERNELS + """
from boxzyhydro_amd.hydro import HydroGrid
def go(name, args):
    if "k_rows_to_planes" in name or "k_planes_to_rows" in name:
        n0, cnt = arg(args, 0, ctypes.c_int64), arg(args, 1, ctypes.c_int64)
        k, n = arg(args, 2, ctypes.c_int), arg(args, 3, ctypes.c_int64)
        src, dst = arg(args, 4, ctypes.c_void_p), arg(args, 5, ctypes.c_void_p)
        m = cnt // k
        if "k_rows_to_planes" in name:
            planes_of(dst, k, n)[:, n0:n0 + m] = rows_of(src, cnt).reshape(m, k).T
        else:
            rows_of(dst, cnt)[:] = planes_of(src, k, n)[:, n0:n0 + m].T.reshape(-1)
launch(on_launch, 1 << 20)
prm = dataclasses.replace(box_params(8), nx=EDGE, ny=EDGE, nz=EDGE)
rng = np.random.default_rng(0)
want = {"cons": rng.standard_normal((prm.ngrid, 5)), "u": rng.standard_normal((prm.ngrid, 3)),
        "p": rng.standard_normal(prm.ngrid), "adindx": rng.standard_normal(prm.ngrid)}
g = HydroGrid(prm)
g.upload(want)
got = g.download()
assert not failed, failed
for k, v in want.items():
    assert np.array_equal(got[k], v), k
assert fake.fake_bad() == 0
print(max(sizes))
"""


@pytest.mark.parametrize("program", [BOXES, GRID], ids=["boxes", "grid"])
@pytest.mark.parametrize("edge", [8, 60, 96])  # below 8 MB, below and above the staging buffer's 24 MiB
def test_chunks_fit_the_staging_buffer(tmp_path, program, edge):
    out = fakehip.run(tmp_path, program.replace("EDGE", str(edge)))
    assert int(out) <= 24 << 20


THREADS = GRID.replace("launch(on_launch, 1 << 20)", "launch(on_launch)").replace("g.upload(want)", """
g.upload(want)  # makes the buffers and slots
want = {k: v[::-1].copy() for k, v in want.items()}
fake.fake_no_new(1)
g.upload(want)""").replace("assert not failed, failed", """fake.fake_no_new(0)
assert not failed, failed""", 1)


def test_transfers_without_memory_for_a_thread(tmp_path):
    """Large transfers whose workers cannot be made: an exception while some
    run would end the process."""
    fakehip.run(tmp_path, THREADS.replace("EDGE", "96"))
