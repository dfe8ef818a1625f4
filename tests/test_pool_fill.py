"""The pool's chunk fill counts the work items of its table -- 64-site chunks of
a plane, across rows, times x segments -- also for edges that are no multiple
of 64, where counting chunks row by row would stop at down to half the items
wanted.  CPU only."""
import ctypes

import numpy as np
import pytest

from test_sched_host import h  # noqa: F401  (the built harness)


def items_of(n, xseg):
    """The table's items (ax_pool.hip): nc = ceil(n n / 64) chunks, nseg segments."""
    return sum(-(-m * m // 64) * -(-m // x) for m, x in zip(n, xseg))


@pytest.mark.parametrize("seed", range(20))
def test_fill_counts_the_tables_items(h, seed):  # noqa: F811
    rng = np.random.default_rng(seed)
    arr = lambda v: (ctypes.c_int * len(v))(*v)
    count = int(rng.integers(1, 8))
    n = [int(rng.choice([3, 33, 64, 65, 72, 80, 96, 100, 129, 144, 200])) for _ in range(count)]
    xseg = [int(rng.choice([4, 8, 16, 32])) for _ in range(count)]
    want = int(rng.integers(1, 12000))
    xs = arr(xseg)
    work = h.fill_segments(count, arr(n), None, xs, want, 4)
    got = list(xs)
    assert work == items_of(n, got)
    assert all(g <= x and g >= min(x, 4) for g, x in zip(got, xseg))
    # full, or at the floor; and not shortened further than needed
    assert work >= want or all(g == 4 for g in got), (n, xseg, want, got)
    if got != xseg:
        longest = max(got)
        before = [min(x, 2 * longest) if g == longest else g for g, x in zip(got, xseg)]
        assert items_of(n, before) < want


def test_short_rows_are_not_counted_as_full_chunks(h):  # noqa: F811
    """One 65^3 lattice: a row of two chunks, of which the second holds one
    site, would count 130 items a plane; the table holds 67."""
    xs = (ctypes.c_int * 1)(32)
    assert h.fill_segments(1, (ctypes.c_int * 1)(65), None, xs, 1100, 4) == 67 * 17 and xs[0] == 4
