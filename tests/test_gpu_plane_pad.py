"""Planes an odd number of elements apart (AX_PLANE_PAD_BYTES): two sites a
thread are loaded only from aligned pairs, and states, energies and windings
are those of the default padding."""
import numpy as np
import pytest

import axions_amd as ax
from axions_amd.abi import AX_BC_PERIODIC

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("shape", [(6, 5, 130), (20, 30, 64)])
def test_odd_pitch_global(shape, precision, monkeypatch):
    nx, ny, nz = shape
    got = []
    for pad in (None, 4352 + precision // 8):
        print(f"[plane pad] {shape} FP{precision} pad {pad}", flush=True)
        if pad:
            monkeypatch.setenv("AX_PLANE_PAD_BYTES", str(pad))
        for boundary in (AX_BC_PERIODIC, ax.AX_BC_NEUMANN_XY):
            with ax.Lattice(ax.global_params(nx, ny=ny, nz=nz, boundary=boundary, precision=precision)) as lat:
                lat.init_random_phase(3)
                lat.step(5)
                got.append((lat.get_state(), lat.winding(), lat.diagnostics()))
    for (st, w, d), (st0, w0, d0) in zip(got[2:], got[:2]):
        assert np.array_equal(st.view(np.uint64), st0.view(np.uint64)) and np.array_equal(w, w0)
        assert d["wound_plaquettes"] == d0["wound_plaquettes"]
        # at most 4e4 nonnegative terms in another order
        assert abs(d["energy"] - d0["energy"]) <= 1e-11 * d0["energy"]
