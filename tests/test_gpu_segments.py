"""The default x-segment length of the marching kernels: every rule outcome
(one plane, a few, the cap, uneven last segments) steps the same bits as one
segment over the whole x extent, and sums the same diagnostics."""
import numpy as np
import pytest

import axions_amd as ax

pytestmark = pytest.mark.gpu

SHAPES = [(3, 3, 3), (33, 32, 32), (64, 48, 65), (37, 80, 130), (150, 40, 64)]


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("model", ["ah", "moore"])
@pytest.mark.parametrize("shape", SHAPES)
def test_default_segments_equal_whole_x_segments(shape, model, precision):
    print(f"[segments] {model} {shape} FP{precision}", flush=True)
    nx, ny, nz = shape
    build = ax.ah_params if model == "ah" else ax.moore_params
    p = build(nx, ny=ny, nz=nz, dt=0.1, precision=precision)
    got = []
    for whole in (False, True):
        with ax.Lattice(p) as lat:
            lat.init_random_phase(11)
            if whole:
                lat.set_tile(0)
            else:
                assert 1 <= lat.tile()[0] <= 32
            d = lat.step_diag(7, 3)
            got.append((lat.get_state(), d))
    assert np.array_equal(got[0][0].view(np.uint64), got[1][0].view(np.uint64))
    for a, b in zip(got[0][1], got[1][1]):
        assert a["wound_plaquettes"] == b["wound_plaquettes"] and a["finite"] == b["finite"] == 1
        # sums of at most 4e5 nonnegative terms in another order: 4e5 eps
        assert abs(a["energy"] - b["energy"]) <= 1e-10 * abs(b["energy"])
        assert abs(a["gauss_mean"] - b["gauss_mean"]) <= 1e-10 * abs(b["gauss_mean"]) + 1e-300
