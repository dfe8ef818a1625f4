"""The step kernels keep their vector registers (read from the metadata of the
built library): none of the ensemble pool's, whose FP64 kernel took 1.25x the
time with 18 of them in scratch memory, and none of the Moore model's, which
took 1.5x on large planes with 30, and none of the Abelian-Higgs FP64 kernels
for whole chunks.  And the FP64 pool steps whole 64-site
chunks and chunks across rows side by side to the bits of single lattices."""
import os
import re

import numpy as np
import pytest

import axions_amd as ax
from axions_amd.abi import AX_REQ_DONE


def kernels():
    """Name -> metadata of the library's gfx950 kernels."""
    msgpack = pytest.importorskip("msgpack")
    with open(os.path.join(os.path.dirname(ax.__file__), "libaxions.so"), "rb") as f:
        blob = f.read()
    out, at = {}, -1
    while (at := blob.find(b"\xaeamdhsa.kernels", at + 1)) >= 0:
        u = msgpack.Unpacker(strict_map_key=False)
        u.feed(blob[at - 1:at + (1 << 20)])
        for k in u.unpack()["amdhsa.kernels"]:
            out[k[".name"]] = k
    return out


# ah_tiled_kernel<double, ..., FLAT = false>: powers of two or not, plain or
# not, by 64-bit planes, LDS prefetch or neither
AH_WHOLE = r"ah_tiled_kernelId(Lb[01]E){4}Lb0EE"


@pytest.mark.parametrize("kernel,variants", [("pool_step_kernel", 4), ("moore_tiled_kernel", 20), (AH_WHOLE, 12)])
def test_step_kernels_do_not_spill(kernel, variants):
    found = {n: k for n, k in kernels().items() if re.search(kernel, n)}
    assert len(found) == variants, sorted(found)
    for name, k in found.items():
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, name


@pytest.mark.gpu
def test_fp64_pool_both_chunk_forms():
    reqs = [(64, 31, 7), (100, 32, 5), (128, 33, 4), (65, 34, 9)]
    with ax.Pool(ax.ah_params(8, precision=64), hbm_budget=2 << 30, chunk_steps=4, autotune=0, ic_threads=2) as pool:
        ids = [pool.submit(seed, n, steps, keep_state=True) for n, seed, steps in reqs]
        assert pool.wait(timeout=100)
        for rid, (n, seed, steps) in zip(ids, reqs):
            print(f"[pool forms] {n}^3 {steps} steps", flush=True)
            assert pool.info(rid)["status"] == AX_REQ_DONE
            with ax.Lattice(ax.ah_params(n)) as lat:
                lat.init_random_phase(seed)
                lat.step(steps)
                want = lat.get_state()
            assert np.array_equal(pool.get_state(rid).view(np.uint64), want.view(np.uint64))
