"""The energy of the global model where a block takes one to four runs of
sites, the last block partly or wholly past the lattice's end: the oracle's
one-thread sum."""
import numpy as np
import pytest

import axions_amd as ax
from axions_amd.abi import AX_BC_NEUMANN_XY, AX_BC_PERIODIC
from oracle import oracle_py as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("boundary", [AX_BC_PERIODIC, AX_BC_NEUMANN_XY])
@pytest.mark.parametrize("shape", [(16, 16, 16), (64, 64, 127), (64, 65, 128), (81, 81, 81), (101, 101, 101)])
def test_energy_by_runs(shape, boundary, precision):
    print(f"[global runs] {shape} boundary={boundary} FP{precision}", flush=True)
    nx, ny, nz = shape
    V = nx * ny * nz
    p = ax.global_params(nx, ny=ny, nz=nz, dx=0.25, dt=0.05, boundary=boundary, precision=precision)
    st = orc.init_random_phase(p, 6)
    st[2 * V:] = np.random.default_rng(4).uniform(-0.2, 0.2, 2 * V)
    if precision == 32:
        st = st.astype(np.float32)
    with ax.Lattice(p) as lat:
        lat.set_state(st.astype(np.float64))
        for n in range(2):
            lat.step(1)
            e = orc.global_step(p, st, 1)[0]
            d = lat.diagnostics(winding=False)
            # V nonnegative terms added one after another: V eps on either side
            assert d["finite"] == 1 and abs(d["energy"] - e) <= 2 * V * 2.0 ** -53 * e, (n, d["energy"], e)
