"""The default x-segment length (ax::default_xseg) follows the lattice without
a jump: two cubes of the same kind of rows that differ by a few sites an edge
get lengths within a quarter of each other, and two planes.  CPU only."""
import ctypes

import pytest

import axions_amd as ax
from axions_amd import abi
from axions_amd.lattice import lib


def length(model, n, precision):
    f = lib._ZN2ax12default_xsegERK9ax_params
    f.restype, f.argtypes = ctypes.c_int, [ctypes.POINTER(abi.AxParams)]
    p = (ax.ah_params if model == "ah" else ax.moore_params)(n, precision=precision)
    return f(ctypes.byref(p))


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("model", ["ah", "moore"])
@pytest.mark.parametrize("rows", ["whole chunks", "across rows"])
def test_no_jump(model, precision, rows, monkeypatch):
    monkeypatch.delenv("AX_TILED_XSEG", raising=False)
    edges = [n for n in range(16, 513) if (n % 64 == 0) == (rows == "whole chunks")]
    got = [length(model, n, precision) for n in edges]
    assert all(1 <= x <= n for x, n in zip(got, edges))
    if rows == "across rows":
        for (n0, a), (n1, b) in zip(zip(edges, got), list(zip(edges, got))[1:]):
            assert abs(a - b) <= 2 + max(a, b) // 4, (n0, a, n1, b)
    assert got == sorted(got) or max(abs(x - y) for x, y in zip(got, sorted(got))) <= 2
