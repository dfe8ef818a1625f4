"""The diagnostics and winding marches by their default x segments (one plane,
a few, uneven last ones) against the one-site kernels on the same state:
energy, Gauss law, finiteness, winding counts and fields, for every model and
precision -- also where the step's own segments play no part in them."""
import numpy as np
import pytest

import axions_amd as ax
from axions_amd.abi import AX_BC_FIXED, AX_BC_PERIODIC

pytestmark = pytest.mark.gpu

SHAPES = [(3, 3, 3), (33, 32, 32), (64, 48, 65), (37, 80, 130), (150, 40, 64), (101, 50, 51)]


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("model", ["ah", "moore"])
@pytest.mark.parametrize("boundary", [AX_BC_PERIODIC, AX_BC_FIXED])
@pytest.mark.parametrize("shape", SHAPES)
def test_diagnostics_by_segments(shape, boundary, model, precision, monkeypatch):
    print(f"[diag segments] {model} {shape} boundary={boundary} FP{precision}", flush=True)
    nx, ny, nz = shape
    build = ax.ah_params if model == "ah" else ax.moore_params
    p = build(nx, ny=ny, nz=nz, dt=0.1, boundary=boundary, precision=precision)
    with ax.Lattice(p) as lat:
        lat.init_random_phase(12)
        lat.step(5)
        w, d = lat.winding(), lat.diagnostics(winding=True)
        monkeypatch.setenv("AX_DIAG_SITE_KERNEL", "1")
        ws, ds = lat.winding(), lat.diagnostics(winding=True)
        monkeypatch.delenv("AX_DIAG_SITE_KERNEL")
    assert np.array_equal(w, ws) and d["wound_plaquettes"] == ds["wound_plaquettes"]
    assert d["finite"] == ds["finite"] == 1
    # at most 4e5 nonnegative terms, an ulp apart, in another order: 4e5 eps
    for key in ("energy", "gauss_mean"):
        assert abs(d[key] - ds[key]) <= 1e-10 * abs(ds[key]) + 1e-300, key
