"""Read-back of states, winding fields and crossings around the size where
downloads go through staged pieces: what set_state put in comes back."""
import numpy as np
import pytest

import axions_amd as ax

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("shape", [(5, 7, 9), (36, 38, 38), (37, 38, 38), (47, 47, 51), (64, 64, 64), (70, 81, 66)])
@pytest.mark.parametrize("model", ["ah", "moore", "global"])
def test_state_comes_back(model, shape, precision):
    print(f"[download] {model} {shape} FP{precision}", flush=True)
    nx, ny, nz = shape
    build = {"ah": ax.ah_params, "moore": ax.moore_params, "global": ax.global_params}[model]
    p = build(nx, ny=ny, nz=nz, precision=precision)
    st = np.random.default_rng(nx).standard_normal(ax.state_len(p))
    if precision == 32:
        st = st.astype(np.float32).astype(np.float64)
    with ax.Lattice(p) as lat:
        lat.set_state(st)
        for _ in range(2):
            assert np.array_equal(lat.get_state(), st)
        w = lat.winding().astype(np.int64)
        d = lat.diagnostics()
        assert int(np.abs(w).sum()) == d["wound_plaquettes"] > 0
        pts, n = lat.crossings()
        assert pts.shape == (n, 3) and n > 0
        part, _ = lat.crossings(cap=max(1, n // 3))
        assert np.array_equal(part, pts[:max(1, n // 3)])
