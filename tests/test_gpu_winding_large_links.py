"""Windings of lattices with faces where link angles are too large for FP32
edge values (2^23 and more): the integers of the site kernel, which sums the
plaquette in FP64, in the winding field and in the diagnostics' count."""
import numpy as np
import pytest

import axions_amd as ax
from axions_amd.abi import AX_BC_ABSORBING, AX_BC_FIXED, AX_BC_NEUMANN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("angle", [2.0 ** 22, 2.0 ** 23, 1e8, 1e9])
@pytest.mark.parametrize("shape", [(5, 6, 64), (33, 20, 65)])
@pytest.mark.parametrize("name", ["absorbing", "neumann", "z_fixed", "moore_fixed"])
def test_large_links(name, shape, angle, monkeypatch):
    print(f"[large links] {name} {shape} {angle:g}", flush=True)
    nx, ny, nz = shape
    if name == "moore_fixed":
        p = ax.moore_params(nx, ny=ny, nz=nz, boundary=AX_BC_FIXED)
    elif name == "z_fixed":
        p = ax.ah_params(nx, ny=ny, nz=nz, boundary_z=AX_BC_FIXED)
    else:
        p = ax.ah_params(nx, ny=ny, nz=nz, boundary=AX_BC_ABSORBING if name == "absorbing" else AX_BC_NEUMANN)
    rng = np.random.default_rng(8)
    nc = ax.ncomp(p)
    st = rng.standard_normal((nc, ax.state_len(p) // nc))
    st[-3:] = rng.uniform(-angle, angle, st[-3:].shape)
    fields = (0, 1) if name == "moore_fixed" else (0,)
    with ax.Lattice(p) as lat:
        lat.set_state(st.reshape(-1))
        march = [lat.winding(f) for f in fields]
        d = lat.diagnostics()
        monkeypatch.setenv("AX_DIAG_SITE_KERNEL", "1")
        site = [lat.winding(f) for f in fields]
        ds = lat.diagnostics()
        monkeypatch.delenv("AX_DIAG_SITE_KERNEL")
    for m, s in zip(march, site):
        assert np.array_equal(m, s)
    assert d["wound_plaquettes"] == ds["wound_plaquettes"] > 0
    assert d["string_length"] == ds["string_length"] and d["xi"] == ds["xi"]
