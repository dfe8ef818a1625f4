"""The Abelian-Higgs step by 64-bit plane addresses (forced on small lattices):
whole chunks and chunks across rows, every boundary, both precisions, to the
bits of the step by buffer accesses."""
import numpy as np
import pytest

import axions_amd as ax
from axions_amd.abi import AX_BC_ABSORBING, AX_BC_FIXED, AX_BC_NEUMANN, AX_BC_PERIODIC

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("xy,z", [(AX_BC_PERIODIC, AX_BC_PERIODIC), (AX_BC_ABSORBING, AX_BC_PERIODIC),
                                  (AX_BC_NEUMANN, AX_BC_FIXED)])
@pytest.mark.parametrize("shape", [(5, 3, 64), (12, 9, 128), (9, 7, 65), (7, 5, 3), (40, 33, 192)])
def test_big_plane_step(shape, xy, z, precision, monkeypatch):
    nx, ny, nz = shape
    got = []
    for alpha in (0.0, 2.0):
        p = ax.ah_params(nx, ny=ny, nz=nz, dx=0.5 + alpha / 10, dt=0.05, alpha=alpha, boundary=xy, boundary_z=z,
                         precision=precision)
        for big in ("", "1"):
            print(f"[big planes] {shape} {xy}/{z} FP{precision} alpha={alpha} big={big}", flush=True)
            monkeypatch.setenv("AX_BIG_PLANES", "1") if big else monkeypatch.delenv("AX_BIG_PLANES", raising=False)
            with ax.Lattice(p) as lat:
                lat.init_random_phase(4)
                lat.step(6)
                got.append(lat.get_state())
    for a, b in zip(got[::2], got[1::2]):
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64))
