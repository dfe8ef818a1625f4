"""The Moore march over chunks that cross rows (the neighbours' phi loaded
ahead of the plaquette sines, or with the band check not) steps the bits of
the site kernel: rows shorter and longer than a wave, one chunk a plane, a
last partial chunk, divisors that are and are not powers of two."""
import numpy as np
import pytest

import axions_amd as ax
from axions_amd.abi import AX_BC_FIXED, AX_BC_PERIODIC

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dx,boundary", [(0.5, AX_BC_PERIODIC), (0.7, AX_BC_PERIODIC), (0.7, AX_BC_FIXED)])
@pytest.mark.parametrize("shape", [(3, 3, 3), (4, 5, 13), (5, 7, 63), (4, 3, 65), (3, 6, 127)])
def test_moore_across_rows_equals_site_kernel(shape, dx, boundary, monkeypatch):
    print(f"[moore across rows] {shape} dx {dx} boundary {boundary}", flush=True)
    nx, ny, nz = shape
    p = ax.moore_params(nx, ny=ny, nz=nz, dx=dx, dt=0.1, boundary=boundary)
    got = []
    for site in (False, True):
        if site:
            monkeypatch.setenv("AX_FORCE_SITE_KERNEL", "1")
        with ax.Lattice(p) as lat:
            lat.init_random_phase(3)
            lat.step(7)
            got.append(lat.get_state())
    assert np.array_equal(got[0].view(np.uint64), got[1].view(np.uint64))
