"""The point pass of the crossings takes its faces from the count pass's
masks: after other lattices' calls left theirs in the shared scratch, with a
last chunk of 1..64 sites, more and fewer sites than a group, and room for no,
some and all points, it writes the rows that ax_crossings returns."""
import ctypes

import numpy as np
import pytest

import axions_amd as ax
from axions_amd.lattice import lib

pytestmark = pytest.mark.gpu

hip = ctypes.CDLL("libamdhip64.so")
hip.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
hip.hipFree.argtypes = [ctypes.c_void_p]
hip.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
hip.hipMemset.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t]
D2H = 2
UNTOUCHED = np.uint64(0xFFFFFFFFFFFFFFFF)


def noalloc(lat, cap):
    """The count, and the bits of cap + 1 rows, of which the call may write cap."""
    rows = np.empty((cap + 1, 3), dtype=np.uint64)
    count = np.empty(1, dtype=np.int64)
    buf = ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(buf), rows.nbytes + 8) == 0
    try:
        assert hip.hipMemset(buf, 0xFF, rows.nbytes + 8) == 0
        cnt = buf.value + rows.nbytes
        rc = lib.ax_crossings_noalloc(lat.handle, buf if cap else None, cap, cnt)
        assert rc == 0, lib.ax_last_error().decode()
        lat.sync()
        assert hip.hipMemcpy(rows.ctypes.data, buf, rows.nbytes, D2H) == 0
        assert hip.hipMemcpy(count.ctypes.data, cnt, 8, D2H) == 0
    finally:
        assert hip.hipFree(buf) == 0
    return int(count[0]), rows


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("shape", [(3, 3, 3), (4, 4, 4), (5, 13, 1 + 64), (33, 32, 64), (90, 80, 77)])
def test_masked_points(shape, precision):
    print(f"[crossing masks] {shape} FP{precision}", flush=True)
    nx, ny, nz = shape
    with ax.Lattice(ax.ah_params(96, precision=precision)) as other:
        other.init_random_phase(2)
        noalloc(other, 8)
    with ax.Lattice(ax.ah_params(nx, ny=ny, nz=nz, precision=precision)) as lat:
        for seed in (3, 4):   # the second state over the first one's masks
            lat.init_random_phase(seed)
            lat.step(2)
            want, total = lat.crossings()
            n, _ = noalloc(lat, 0)
            assert n == total == len(want) > 0
            for cap in (1, n // 2, n):
                got, rows = noalloc(lat, cap)
                assert got == n
                assert np.array_equal(rows[:cap], want[:cap].view(np.uint64))
                assert (rows[cap:] == UNTOUCHED).all()
