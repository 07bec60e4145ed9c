"""Grids whose x-y plane the tiled kernels cannot address (32-bit byte offsets
within a plane; rows of tiles in the launch's y dimension): the flux subroutine
takes the cell-by-cell kernel, the fused modes the exact sequence.  On the CPU,
over the stand-in HIP runtime: which kernels are launched."""
from __future__ import annotations

import pytest

import fakehip

PROGRAM = """
names = set()
launch(lambda name, g, b, args: names.add(name))
L = nv.lib()
prm = nv.BxParams()
from boxzyhydro_amd.hydro import make_params
p = make_params(dataclasses.replace(box_params(8), nx=NX, ny=NY, nz=1, **OPTIONS), PRECISION)
h = ctypes.c_void_p()
nv.check(L.bx_create(ctypes.byref(p), 0, ctypes.byref(h)), "create")
for avg in (0, 1):
    nv.check(L.bx_flux(h, avg, 1e-6), "flux")
flux = set(names)
names.clear()
t, dto, st, k = ctypes.c_double(), ctypes.c_double(), ctypes.c_int32(), ctypes.c_int32()
for end in (1.0, 2.0):  # the first step is an exact one on every grid
    rc = L.bx_step(h, nv.BX_STEP_GRAPH, 1, end, ctypes.byref(t), ctypes.byref(dto), ctypes.byref(st), None, ctypes.byref(k))
print(int(any("k_stage" in x for x in flux)), int(any("k_flux_cells" in x for x in flux)),
      int(any("k_regular" in x for x in names)), rc)
L.bx_destroy(h)
"""


def _run(tmp_path, nx, ny, precision="nv.BX_PREC_FP64", options="{}"):
    src = PROGRAM.replace("NX", str(nx)).replace("NY", str(ny)).replace("PRECISION", precision).replace("OPTIONS", options)
    return [int(v) for v in fakehip.run(tmp_path, src).split()]


@pytest.mark.parametrize("options", ["{}", "dict(fluxangmom=True)"])
@pytest.mark.parametrize("nx,ny", [(1 << 15, 1 << 14), (404, 8), (7, 262144)])
def test_planes_within_reach_take_the_tile(tmp_path, nx, ny, options):
    assert _run(tmp_path, nx, ny, options=options) == [1, 1, int(options == "{}"), 0]


@pytest.mark.parametrize("options", ["{}", "dict(fluxangmom=True)"])
@pytest.mark.parametrize("nx,ny", [(23200, 23200), ((1 << 15) + 1, 1 << 14), (7, 262146)])
def test_planes_out_of_reach_go_cell_by_cell(tmp_path, nx, ny, options):
    assert _run(tmp_path, nx, ny, options=options) == [0, 1, 0, 0]


def test_mixed_form_refuses_them(tmp_path):
    assert _run(tmp_path, 1 << 15, 1 << 14, "nv.BX_PREC_MIXED")[3] == 0
    assert _run(tmp_path, 33000, 33000, "nv.BX_PREC_MIXED")[3] == -4
