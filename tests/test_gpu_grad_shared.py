"""Vertex gradients accumulated into one buffer by both grids of a call, or by calls
on two streams: nothing is lost (grids whose cells own their vertices, and grids that
share them; tables, re-oriented cells; both directions)."""
import threading

import numpy as np
import pytest
import torch

from polygrids import rotation

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _table(cr, cells):
    return cr.Grid.from_cells(np.ascontiguousarray(cells), convex=True)


def _grids(cr, name):
    a = cr.healpix_cells(32, "nested", 1)
    b = a @ rotation(4).T
    if name == "tables":
        return cr.Grid.healpix(32, "nested", step=1), _table(cr, b)
    if name == "re-oriented tables":  # every third cell clockwise
        for c in (a, b):
            c[::3] = c[::3, ::-1]
        return _table(cr, a), _table(cr, b)
    p = cr.lonlat_points(120, 60)
    return cr.Grid.from_points(p), cr.Grid.from_points(p @ rotation(5).T)


def _call(cr, R, dst, src, t, normalize, x, y, gy, gd, gs):
    cr._lib.check(cr._lib.lib.cr_regrid_backward(
        R._core.h, dst._h, src._h, t, normalize, 1, x.data_ptr(), 1, 1, y.data_ptr(), 1, 1, gy.data_ptr(), 1, 1, None, 1, 1,
        gd.data_ptr(), gs.data_ptr(), torch.cuda.current_stream().cuda_stream))


@pytest.mark.parametrize("transpose,normalize", [(0, 1), (0, 0), (1, 1)])
@pytest.mark.parametrize("name", ["tables", "re-oriented tables", "points"])
def test_one_buffer_for_both_grids(cr, name, transpose, normalize):
    print(f"[case] one buffer {name} {transpose} {normalize}", flush=True)
    dst, src = _grids(cr, name)
    assert dst.nverts == src.nverts
    R = cr.Regridder(dst, src, radius=1.0)
    RR = cr.transpose(R) if transpose else R
    x, gy = (torch.tensor(np.random.default_rng(i).random(dst.ncells), device=DEV) for i in (1, 2))
    y = cr.regrid(RR, x)
    ref = [torch.zeros(dst.nverts, 3, dtype=torch.float64, device=DEV) for _ in range(2)]
    _call(cr, R, dst, src, transpose, normalize, x, y, gy, *ref)
    want = ref[0] + ref[1]
    one = torch.zeros_like(want)
    for _ in range(3):
        _call(cr, R, dst, src, transpose, normalize, x, y, gy, one, one)
    tol = 1e-12 * float(want.abs().max())  # sums of a few dozen terms in any order
    assert float((one - 3 * want).abs().max()) <= 3 * tol


@pytest.mark.parametrize("transpose,normalize", [(0, 1), (0, 0), (1, 1)])
@pytest.mark.parametrize("name", ["tables", "re-oriented tables", "points"])
def test_one_buffer_on_two_streams(cr, name, transpose, normalize):
    print(f"[case] two streams {name} {transpose} {normalize}", flush=True)
    dst, src = _grids(cr, name)
    R = cr.Regridder(dst, src, radius=1.0)
    RR = cr.transpose(R) if transpose else R
    x, gy = (torch.tensor(np.random.default_rng(i).random(dst.ncells), device=DEV) for i in (1, 2))
    y = cr.regrid(RR, x)
    want, got = ([torch.zeros(dst.nverts, 3, dtype=torch.float64, device=DEV) for _ in range(2)] for _ in range(2))
    _call(cr, R, dst, src, transpose, normalize, x, y, gy, *want)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]

    def work(s):
        torch.cuda.set_device(0)
        with torch.cuda.stream(s):
            for _ in range(8):
                _call(cr, R, dst, src, transpose, normalize, x, y, gy, *got)


    threads = [threading.Thread(target=work, args=(s,)) for s in streams]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        assert float((g - 16 * w).abs().max()) <= 16 * 1e-12 * float(w.abs().max())
