"""The FP64 march with its rows prefetched into LDS steps the same bits as
without, at the edges of what it takes: one chunk a row (its own z neighbour),
the smallest x and y, faces that are not stepped, a last edge block of 1..4
planes, and a step with the diagnostics in it."""
import numpy as np
import pytest

import axions_amd as ax
from axions_amd.abi import AX_BC_ABSORBING, AX_BC_FIXED, AX_BC_NEUMANN, AX_BC_PERIODIC

pytestmark = pytest.mark.gpu

CASES = [(3, 3, 64, "periodic", 0), (4, 3, 128, "periodic", 1), (5, 4, 192, "fixed", 2), (9, 5, 64, "absorbing", 0),
         (7, 6, 128, "neumann", 3)]


@pytest.mark.parametrize("nx,ny,nz,faces,xseg", CASES)
def test_prefetched_rows_equal_direct_loads(nx, ny, nz, faces, xseg, monkeypatch):
    print(f"[row prefetch] {nx}x{ny}x{nz} {faces} xseg {xseg}", flush=True)
    b = {"periodic": AX_BC_PERIODIC, "fixed": AX_BC_FIXED, "absorbing": AX_BC_ABSORBING, "neumann": AX_BC_NEUMANN}[faces]
    p = ax.ah_params(nx, ny=ny, nz=nz, dt=0.1, boundary=b)
    got = []
    for direct in (False, True):
        if direct:
            monkeypatch.setenv("AX_NO_PREFETCH", "1")
        with ax.Lattice(p) as lat:
            lat.init_random_phase(5)
            lat.set_tile(xseg)
            lat.step(6)
            d = lat.step_diag(4, 2) if faces == "periodic" else []
            got.append((lat.get_state(), [x["wound_plaquettes"] for x in d]))
    assert np.array_equal(got[0][0].view(np.uint64), got[1][0].view(np.uint64))
    assert got[0][1] == got[1][1]
