"""Crossings of fields where the face rejection and the compaction can go
wrong -- corners of zero, tiny, one-signed or non-finite values, few or no
roots, sizes around the 64-site chunk and the 512-site group -- against the
oracle, which solves every face: the same points in the same order, bit for
bit."""
import numpy as np
import pytest

import axions_amd as ax
from axions_amd.abi import AX_BC_FIXED, AX_BC_PERIODIC
from oracle import oracle_py as orc

pytestmark = pytest.mark.gpu

SHAPES = [(3, 3, 3), (4, 4, 4), (7, 5, 9), (8, 8, 8), (9, 8, 64), (5, 21, 130), (40, 33, 65),
          (3, 4, 3000), (3, 3, 9000)]
LEVELS = np.array([0.0, -0.0, 1e-300, -1e-300, 5e-324, 1e-12, -1e-12, 1.0, -1.0, 1e3, -1e-3])


def field(kind, shape, rng):
    if kind == "levels":          # corners from a few special values: ties, exact zeros, denormals
        return rng.choice(LEVELS, size=shape), rng.choice(LEVELS, size=shape)
    if kind == "network":         # a vortex line off the grid: almost every face has one sign
        x, y, _ = np.meshgrid(*[np.arange(n) - 0.37 * n for n in shape], indexing="ij")
        return np.tanh(0.3 * x), np.tanh(0.3 * y) + 1e-9 * rng.standard_normal(shape)
    re, im = rng.standard_normal(shape), rng.standard_normal(shape)
    if kind == "one_sign":        # Re phi barely of one sign: roots only through rounding
        return np.abs(re) * 1e-14 + 1e-15, im
    if kind == "nonfinite":
        for v in (re, im):
            v.reshape(-1)[rng.integers(0, v.size, max(1, v.size // 20))] = rng.choice([np.nan, np.inf, -np.inf])
    return re, im


@pytest.mark.parametrize("kind", ["random", "levels", "network", "one_sign", "nonfinite"])
@pytest.mark.parametrize("shape", SHAPES)
def test_crossings_match_the_oracle(shape, kind):
    nx, ny, nz = shape
    rng = np.random.default_rng(nx * 7919 + nz)
    for boundary, precision, spacing in ((AX_BC_PERIODIC, 64, 0.5), (AX_BC_FIXED, 64, 0.3), (AX_BC_PERIODIC, 32, 0.7)):
        print(f"[crossings] {shape} {kind} boundary={boundary} FP{precision}", flush=True)
        p = ax.ah_params(nx, ny=ny, nz=nz, dx=spacing, dy=1.3 * spacing, precision=precision, boundary=boundary)
        st = np.zeros((5, 2, nx, ny, nz))
        st[0], st[1] = field(kind, shape, rng)
        if precision == 32:
            with np.errstate(over="ignore"):
                st = st.astype(np.float32).astype(np.float64)
        st = st.reshape(-1)
        with ax.Lattice(p) as lat:
            lat.set_state(st)
            got, n = lat.crossings()
            part, n_part = lat.crossings(cap=n // 2)
            _, n_only = lat.crossings(cap=0)
        want, n_want = orc.crossings(p, st, 0)
        assert n == n_part == n_only == n_want
        assert np.array_equal(got.view(np.uint64), np.ascontiguousarray(want).view(np.uint64))
        assert np.array_equal(part.view(np.uint64), got[:n // 2].view(np.uint64))
