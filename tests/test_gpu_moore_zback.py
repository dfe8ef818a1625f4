"""The band-checked Moore march over whole chunks (z-backward values from the
lane before, the chunk edge's from a pass over four planes) steps the bits of
the site kernel: one to three chunks a row, segments of 1..5 planes and whole,
the smallest x and y, and a state outside the band (plain divisions)."""
import numpy as np
import pytest

import axions_amd as ax

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1.0, 1e-200])
@pytest.mark.parametrize("nx,ny,nz,xseg", [(3, 3, 64, 1), (5, 4, 128, 3), (9, 3, 192, 5), (11, 5, 64, 0)])
def test_moore_whole_chunks_equal_site_kernel(nx, ny, nz, xseg, scale, monkeypatch):
    print(f"[moore z-back] {nx}x{ny}x{nz} xseg {xseg} scale {scale}", flush=True)
    p = ax.moore_params(nx, ny=ny, nz=nz, dx=0.7, dt=0.1)
    got = []
    for site in (False, True):
        if site:
            monkeypatch.setenv("AX_FORCE_SITE_KERNEL", "1")
        with ax.Lattice(p) as lat:
            lat.init_random_phase(6)
            if scale != 1.0:
                lat.set_state(lat.get_state() * scale)
            if not site:
                lat.set_tile(xseg)
            lat.step(6)
            got.append(lat.get_state())
    assert np.array_equal(got[0].view(np.uint64), got[1].view(np.uint64))
