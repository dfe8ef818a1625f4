"""Windings of lattices with faces and of the global model by the marching
edge-value passes: the same integers as the site kernel, which evaluates
every plaquette's four edge phases in FP64, and the same counts in the
diagnostics."""
import numpy as np
import pytest

import axions_amd as ax
from axions_amd.abi import AX_BC_ABSORBING, AX_BC_FIXED, AX_BC_NEUMANN, AX_BC_PERIODIC

pytestmark = pytest.mark.gpu

CASES = {
    "absorbing": lambda n, pr: ax.ah_params(*n[:1], ny=n[1], nz=n[2], dt=0.05, boundary=AX_BC_ABSORBING, precision=pr),
    "absorbing_g0": lambda n, pr: ax.ah_params(*n[:1], ny=n[1], nz=n[2], dt=0.05, g=0.0, boundary=AX_BC_ABSORBING,
                                               boundary_z=AX_BC_FIXED, precision=pr),
    "neumann": lambda n, pr: ax.ah_params(*n[:1], ny=n[1], nz=n[2], dx=0.3, dt=0.05, boundary=AX_BC_NEUMANN,
                                          precision=pr),
    "z_fixed": lambda n, pr: ax.ah_params(*n[:1], ny=n[1], nz=n[2], boundary_z=AX_BC_FIXED, precision=pr),
    "moore_fixed": lambda n, pr: ax.moore_params(*n[:1], ny=n[1], nz=n[2], dt=0.1, boundary=AX_BC_FIXED, precision=pr),
    "moore_neumann": lambda n, pr: ax.moore_params(*n[:1], ny=n[1], nz=n[2], dt=0.1, boundary=AX_BC_NEUMANN,
                                                   precision=pr),
    "global": lambda n, pr: ax.global_params(*n[:1], ny=n[1], nz=n[2], precision=pr),
    "global_periodic": lambda n, pr: ax.global_params(*n[:1], ny=n[1], nz=n[2], boundary=AX_BC_PERIODIC, precision=pr),
}


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("shape", [(3, 3, 3), (5, 6, 64), (12, 9, 65), (33, 20, 130)])
@pytest.mark.parametrize("name", list(CASES))
def test_marching_windings_equal_the_site_kernel(name, shape, precision, monkeypatch):
    print(f"[winding faces] {name} {shape} FP{precision}", flush=True)
    p = CASES[name](shape, precision)
    with ax.Lattice(p) as lat:
        lat.init_random_phase(9)
        for steps in (0, 5):
            lat.step(steps)
            fields = (0, 1) if name.startswith("moore") else (0,)
            march = [lat.winding(f) for f in fields]
            d = lat.diagnostics()
            monkeypatch.setenv("AX_DIAG_SITE_KERNEL", "1")
            site = [lat.winding(f) for f in fields]
            ds = lat.diagnostics()
            monkeypatch.delenv("AX_DIAG_SITE_KERNEL")
            for m, s in zip(march, site):
                assert np.array_equal(m, s)
            assert d["wound_plaquettes"] == ds["wound_plaquettes"] == int(np.abs(site[0].astype(int)).sum())
            # the sums of at most 1e5 nonnegative terms in another order
            assert steps == 0 or abs(d["energy"] - ds["energy"]) <= 1e-11 * abs(ds["energy"])
