"""Fields side by side in small matrices, where blocks take short runs of rows: FP64
equal to one single-field call per field bit for bit, FP32 the FP64 sums rounded once;
matrices with a pole's wide rows, where few FP64 fields go to the tile kernel, too."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _grids(cr, name):
    lonlat = lambda ni, nj: cr.Grid.from_points(cr.lonlat_points(ni, nj))  # noqa: E731
    cube = lambda ne: cr.Grid.from_points(cr.cubed_sphere_points(ne))  # noqa: E731
    return {"one source a row": lambda: (lonlat(36, 18), lonlat(72, 36)),
            "a pole's rows": lambda: (cube(24), lonlat(180, 90)),
            "a pole's rows, more of them": lambda: (cube(48), lonlat(360, 180)),
            "a few cells": lambda: (lonlat(3, 2), lonlat(5, 4))}[name]()


@pytest.mark.parametrize("name", ["one source a row", "a pole's rows", "a pole's rows, more of them", "a few cells"])
def test_small_levels(cr, name):
    R = cr.Regridder(*_grids(cr, name))
    for RR in (R, cr.transpose(R)):
        A, area = RR.intersections, RR.dst_areas
        n_out, n_in = A.shape
        for k in (6, 12, 13, 15, 16, 65, 129, 300):
            print(f"[case] small levels {name} {n_out} x {n_in} k={k}", flush=True)
            x = torch.tensor(np.random.default_rng(k).standard_normal((n_in, k)), device=DEV)
            y = cr.regrid(RR, x)
            for f in {0, k // 3, k - 2, k - 1}:
                assert torch.equal(cr.regrid(RR, x[:, f].contiguous()), y[:, f]), (k, f)
            if k < (6 if A.nnz // n_out <= 8 else 16):
                continue  # FP32 in the tile kernel, which rounds every segment of a row
            x32 = x.float()
            xin = x32.cpu().numpy().astype(np.float64)
            got = cr.regrid(RR, x32).cpu().numpy().astype(np.float64)
            ref, scale = (A @ xin) / area[:, None], (abs(A) @ abs(xin)) / area[:, None]
            # one rounding of the result, FP64 sums of at most n terms
            tol = 2.0**-24 * np.abs(ref) + np.diff(A.indptr).max() * 2.0**-52 * scale
            assert (np.abs(got - ref) <= 1.001 * tol).all(), k
