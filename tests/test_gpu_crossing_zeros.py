"""Crossings of fields with zeros, NaNs, infinities and values that FP32 takes
for zero, in patches and everywhere: the oracle's points."""
import numpy as np
import pytest

import axions_amd as ax
from oracle import oracle_py as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("value", [0.0, -0.0, np.nan, np.inf, 1e-60, 1e-45])
@pytest.mark.parametrize("where", ["everywhere", "re", "im", "patches", "plane"])
def test_odd_fields(where, value, precision):
    print(f"[crossing zeros] {where} {value} FP{precision}", flush=True)
    n = (12, 9, 70)
    p = ax.ah_params(n[0], ny=n[1], nz=n[2], precision=precision)
    rng = np.random.default_rng(6)
    st = rng.standard_normal(ax.state_len(p)).reshape(5, 2, *n)
    if where == "everywhere":
        st[:2] = value
    elif where in ("re", "im"):
        st[0 if where == "re" else 1] = value
    elif where == "patches":
        st[:2][np.broadcast_to(rng.random(n) < 0.4, (2, 2, *n))] = value
    else:
        st[0, :, 5:7] = value
    st = st.reshape(-1)
    if precision == 32:
        st = st.astype(np.float32).astype(np.float64)
    want, total = orc.crossings(p, st, 0)   # of FP64 fields
    with ax.Lattice(p) as lat:
        lat.set_state(st)
        got, count = lat.crossings()
    assert count == total
    assert np.array_equal(got.view(np.uint64), want.view(np.uint64))
