"""Candidate search where its kernel changes: 8 or 16 destination cells to a wave
(on both sides of the line between them), short and long leaf lists (by the ratio of
source to destination cells), lists that overflow (cells walked by a wave each), a
last wave with few cells, one destination cell, one source cell.

The pairs that make up A are every pair that overlaps: rows and columns of A add up
to the cells' areas (1e-12: FP64 sums of at most some thousand pairs) and a repeated
build gives the same arrays bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dst,src", [
    ((181, 181), (160, 150)),  # 32 761 destination cells: 8 to a wave
    ((182, 181), (160, 150)),  # 32 942: 16
    ((16, 9), (180, 90)),  # many source cells to a cell: long lists that overflow
    ((250, 200), (400, 500)),  # 4 to a cell: still short lists
    ((250, 200), (401, 500)),  # more than 4: long lists
    ((3, 2), (7, 3)),
    ((600, 400), (3, 2)),  # few source cells: lists of all of them
])
def test_search_finds_every_pair(cr, dst, src):
    print(f"[case] search {dst} <- {src}", flush=True)
    d, s = (cr.Grid.from_points(cr.lonlat_points(*n)) for n in (dst, src))
    R = cr.Regridder(d, s, radius=1.0)
    A = R.intersections
    np.testing.assert_allclose(np.asarray(A.sum(1)).ravel(), R.dst_areas, rtol=1e-12)
    np.testing.assert_allclose(np.asarray(A.sum(0)).ravel(), R.src_areas, rtol=1e-12)
    for transpose in (False, True):
        a, b = R._core.csr(transpose), cr.Regridder(d, s, radius=1.0)._core.csr(transpose)
        assert all(np.array_equal(x, y) for x, y in zip(a, b))
