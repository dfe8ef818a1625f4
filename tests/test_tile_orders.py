"""The partial sums of the marching passes: their buffers hold a launch in
either work order, whichever AX_TILE_ORDER named when the lattice was made,
also where the chunks of a plane are no multiple of 8 and the XCD-aware order
has workgroups without work."""
import ctypes
import math

import numpy as np
import pytest

import axions_amd as ax
from axions_amd import abi
from axions_amd.lattice import lib

SHAPES = [(5, 13, 65), (3, 3, 3), (7, 9, 64), (40, 11, 100), (101, 101, 101), (64, 64, 64)]


def order(monkeypatch, name):
    monkeypatch.setenv("AX_TILE_ORDER", name) if name else monkeypatch.delenv("AX_TILE_ORDER", raising=False)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("model", ["ah", "moore"])
def test_partial_buffers_hold_either_order(shape, model, monkeypatch):
    """ax::diag_part_blocks at the creation's order against the workgroups of
    a march at the launch's (ax::fused_work_items of the same segments)."""
    blocks = lib._ZN2ax16diag_part_blocksERK9ax_params
    blocks.restype, blocks.argtypes = ctypes.c_size_t, [ctypes.POINTER(abi.AxParams)]
    items = lib._ZN2ax16fused_work_itemsEiiii
    nx, ny, nz = shape
    p = (ax.ah_params if model == "ah" else ax.moore_params)(nx, ny=ny, nz=nz)
    # the diagnostics' planes per wave: about sqrt(chunks x planes per SIMD), at most 32
    xs = min(32, max(1, int(math.sqrt(-(-ny * nz // 64) * nx / 1024) + 0.5)))
    xs = -(-nx // -(-nx // xs))
    for made in ("natural", ""):
        order(monkeypatch, made)
        room = blocks(ctypes.byref(p))
        for launched in ("natural", ""):
            order(monkeypatch, launched)
            assert items(nx, ny, nz, xs) <= room, (shape, made, launched)


@pytest.mark.parametrize("shape", [(4000, 3, 3), (1000, 10, 10), (200, 20, 20), (43, 28, 29), (600, 28, 29), (43, 43, 22)])
def test_narrow_planes_keep_the_xcds_busy(shape, monkeypatch):
    """No XCD gets more waves than its 128 SIMDs while others have far fewer,
    and below that the chunks of a plane stay together, eighths to an XCD."""
    order(monkeypatch, "")
    nx, ny, nz = shape
    chunks = -(-ny * nz // 64)
    for xs in (1, 2, 4, 32):
        segments = -(-nx // xs)
        work = lib._ZN2ax16fused_work_itemsEiiii(nx, ny, nz, xs)
        fullest = -(-work // 8)    # workgroup w goes to XCD w mod 8
        assert fullest <= max(128, 1.15 * chunks * segments / 8 + 1), (shape, xs)
        if -(-chunks // 8) * segments <= 128:
            assert work == 8 * -(-chunks // 8) * segments


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("shape", SHAPES[:4] + [(300, 3, 3), (100, 10, 10)])
def test_orders_of_creation_and_launch_may_differ(shape, precision, monkeypatch):
    """State, windings and sums: the same whichever order a lattice was
    created and whichever it is stepped and diagnosed in."""
    nx, ny, nz = shape
    p = ax.ah_params(nx, ny=ny, nz=nz, precision=precision)
    got = []
    for made, launched in (("", ""), ("natural", ""), ("", "natural"), ("natural", "natural")):
        print(f"[tile orders] {shape} FP{precision} {made or 'default'} -> {launched or 'default'}", flush=True)
        order(monkeypatch, made)
        with ax.Lattice(p) as lat:
            order(monkeypatch, launched)
            lat.init_random_phase(5)
            lat.step(4)
            d = lat.step_diag(5, 2)
            got.append((lat.get_state(), lat.winding(), d + [lat.diagnostics(winding=True)]))
    for st, w, d in got[1:]:
        assert np.array_equal(st.view(np.uint64), got[0][0].view(np.uint64))
        assert np.array_equal(w, got[0][1])
        for a, b in zip(d, got[0][2]):
            assert a["wound_plaquettes"] == b["wound_plaquettes"] and a["finite"] == b["finite"] == 1
            # at most 5e4 nonnegative terms summed in another order: 5e4 eps
            for key in ("energy", "gauss_mean"):
                assert abs(a[key] - b[key]) <= 1e-11 * abs(b[key]) + 1e-300
