"""The point pass of the crossings takes its faces from the count pass's
masks: after other lattices' calls left theirs in the shared scratch, with a
last chunk of 1..64 sites, more and fewer sites than a group, and room for no,
some and all points, it writes the rows that ax_crossings returns."""
import numpy as np
import pytest
import torch

import axions_amd as ax
from axions_amd.lattice import lib

pytestmark = pytest.mark.gpu


def noalloc(lat, cap):
    pts = torch.full((max(cap, 1) + 1, 3), -7.0, dtype=torch.float64, device="cuda")
    cnt = torch.zeros(1, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    assert lib.ax_crossings_noalloc(lat.handle, pts.data_ptr() if cap else None, cap, cnt.data_ptr()) == 0
    lat.sync()
    return int(cnt), pts.cpu().numpy()


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
                got, pts = noalloc(lat, cap)
                assert got == n
                assert np.array_equal(pts[:cap].view(np.uint64), want[:cap].view(np.uint64))
                assert (pts[cap:] == -7.0).all()
