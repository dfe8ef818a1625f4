"""The staged download on the CPU (axions_amd/csrc/ax_download.h over a
stand-in for the HIP runtime): what lies in the planes arrives, widened or as
it is, and the calling thread's current device is the one it had before, also
when a copy fails or there is no pinned memory."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
MiB = 1 << 20


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("ax_download") / "libdownload.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-pthread", "-D__HIP_PLATFORM_AMD__",
                           "-I", os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"), "-o", so,
                           os.path.join(HERE, "csrc", "download_harness.cpp"), "-Wl,-Bsymbolic"])
    L = ctypes.CDLL(so)
    L.run_download.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int,
                               ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.POINTER(ctypes.c_int)]
    return L


@pytest.mark.parametrize("device", [0, 1])
@pytest.mark.parametrize("widen", [0, 1])
@pytest.mark.parametrize("values,runs", [(5, 3), (MiB, 3), (MiB + 4, 4), (3 * MiB - 4, 10), (4 * MiB, 1)])
def test_runs_arrive_and_the_device_stays(lib, values, runs, widen, device):
    n = values // 4 if widen else values
    src = np.random.default_rng(n).integers(0, 1 << 16, n * runs).astype(np.float32 if widen else np.uint8)
    dst = np.zeros(src.size, dtype=np.float64 if widen else np.uint8)
    after = ctypes.c_int(-1)
    for no_pinned in (0, 1):
        dst[:] = 0
        assert lib.run_download(device, src.ctypes.data, dst.ctypes.data, n, runs, widen, -1, no_pinned, after) == 0
        assert np.array_equal(dst, src)
        assert after.value == device


@pytest.mark.parametrize("copy", [0, 3, 9])
def test_a_failed_copy_is_reported_and_the_device_stays(lib, copy):
    src = np.ones(16 * MiB, dtype=np.uint8)
    dst = np.zeros_like(src)
    after = ctypes.c_int(-1)
    assert lib.run_download(0, src.ctypes.data, dst.ctypes.data, src.size, 1, 0, copy, 0, after) != 0
    assert after.value == 0
