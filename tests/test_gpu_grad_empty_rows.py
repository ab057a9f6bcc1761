"""The area term of destination cells without a source cell: 0 in ordinary use, NaN
for an upstream gradient that is not finite, and the formula's value for whatever y
holds there -- wherever the empty rows lie among the waves' 64 non-zeros."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("covered", ["north", "south", "band", "none"])
def test_area_term_of_uncovered_cells(cr, orc, covered):
    print(f"[case] empty rows {covered}", flush=True)
    p = cr.lonlat_points(24, 12)
    dst = cr.Grid.from_cells(cr.healpix_cells(8, "nested", 1), convex=True)
    q = {"north": p[:, 7:], "south": p[:, :5], "band": p[:, 5:8], "none": p[:2, 4:6] * 1.0}[covered]
    src = cr.Grid.from_points(np.ascontiguousarray(q))
    if covered == "none":  # a cell that meets no destination cell but its own few: drop those as well
        keep = np.asarray(abs(cr.Regridder(dst, src, radius=1.0).intersections).sum(1)).ravel() == 0.0
        dst = cr.Grid.from_cells(np.ascontiguousarray(cr.healpix_cells(8, "nested", 1)[keep]), convex=True)
    R = cr.Regridder(dst, src, radius=1.0)
    A = R.intersections
    empty = np.diff(A.indptr) == 0
    assert empty.any() and (A.nnz == 0) == (covered == "none")
    rng = np.random.default_rng(3)
    x, gy = (torch.tensor(rng.standard_normal(n), device=DEV) for n in (src.ncells, dst.ncells))
    y = cr.regrid(R, x)

    def g_dst(y, gy):
        return cr.regrid_backward(R, dst, src, x, y, gy, field_grad=False)[1].cpu().numpy().reshape(dst.ncells, -1)

    base = g_dst(y, gy)
    assert not base[empty].any() and np.isfinite(base).all()
    # values of the caller's there: dL/da_i = -gy_i y_i / a_i
    e = torch.tensor(empty, device=DEV)
    y2 = torch.where(e, torch.full_like(y, 0.5), y)
    got = g_dst(y2, gy)
    cells, a = dst.cells(), R.dst_areas
    for i in np.flatnonzero(empty):
        _, ga = orc.polygon_area_grad(cells[i])
        want = (-float(gy[i]) * 0.5 / a[i] * ga).ravel()
        assert np.abs(got[i] - want).max() <= 1e-10 * np.abs(want).max()
    scale = np.abs(base).max()
    assert covered == "none" or np.abs(got[~empty] - base[~empty]).max() <= 1e-12 * scale
    gy2 = torch.where(e, torch.full_like(gy, float("inf")), gy)  # inf * 0
    assert np.isnan(g_dst(y, gy2)[empty]).any(axis=1).all()
