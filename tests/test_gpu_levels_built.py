"""Fields side by side with built regridders (rows in candidate order, polar rows of
every width), both directions: FP64 equal to one single-field call per field bit for
bit, FP32 the FP64 sums rounded once."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _grids(cr, name):
    lonlat = lambda ni, nj: cr.Grid.from_points(cr.lonlat_points(ni, nj))  # noqa: E731
    return {
        "lon-lat to HEALPix": lambda: (cr.Grid.healpix(32, "nested", step=2), lonlat(361, 181)),
        "lon-lat to a coarse lon-lat": lambda: (lonlat(36, 18), lonlat(720, 361)),  # rows of 400 and more
        "cubed sphere to lon-lat": lambda: (lonlat(180, 91), cr.Grid.from_points(cr.cubed_sphere_points(40))),
    }[name]()


@pytest.mark.parametrize("name", ["lon-lat to HEALPix", "lon-lat to a coarse lon-lat", "cubed sphere to lon-lat"])
def test_levels_of_built_regridders(cr, name):
    R = cr.Regridder(*_grids(cr, name))
    for RR in (R, cr.transpose(R)):
        A, area = RR.intersections, RR.dst_areas
        n_out, n_in = A.shape
        print(f"[case] built levels {name} rows up to {np.diff(A.indptr).max()}", flush=True)
        rng = np.random.default_rng(n_in)
        x = torch.tensor(rng.standard_normal((n_in, 37)), device=DEV)
        y = cr.regrid(RR, x)
        for f in range(0, 37, 4):
            assert torch.equal(cr.regrid(RR, x[:, f].contiguous()), y[:, f]), f
        x32 = x.float()
        y32 = cr.regrid(RR, x32).cpu().numpy().astype(np.float64)
        xin = x32.cpu().numpy().astype(np.float64)
        ref, scale = (A @ xin) / area[:, None], (abs(A) @ abs(xin)) / area[:, None]
        # one rounding of the result, FP64 sums of at most n terms
        tol = 2.0**-24 * np.abs(ref) + np.diff(A.indptr).max() * 2.0**-52 * scale
        assert (np.abs(y32 - ref) <= 1.001 * tol).all()
