"""Device memory between calls: two threads on hipStreamPerThread (one handle, two
streams)."""
import ctypes
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
PER_THREAD = 2  # hipStreamPerThread


def _grids(cr, n):
    return cr.Grid.from_points(cr.cubed_sphere_points(n)), cr.Grid.from_points(cr.lonlat_points(6 * n, 3 * n))


def _build(cr, dst, src, stream):
    L, h = cr._lib, ctypes.c_void_p()
    st = L.lib.cr_regridder_build(ctypes.byref(h), dst._h, src._h, None, stream)
    return st, h


def _backward(cr, h, dst, src, x, y, gy, g, stream):
    gx, gd, gs = g
    return cr._lib.lib.cr_regrid_backward(
        h, dst._h, src._h, 0, 1, 1, x.data_ptr(), 1, 1, y.data_ptr(), 1, 1, gy.data_ptr(), 1, 1, gx.data_ptr(), 1, 1,
        gd.data_ptr(), gs.data_ptr(), stream)


def test_threads_on_the_per_thread_stream(cr):
    L = cr._lib
    dst, src = _grids(cr, 40)
    R = cr.Regridder(dst, src)
    x, gy = (torch.tensor(np.random.default_rng(i).random(n), device=DEV) for i, n in ((1, src.ncells), (2, dst.ncells)))
    y = cr.regrid(R, x)

    def out():
        return [torch.zeros(n, dtype=torch.float64, device=DEV)
                for n in (src.ncells, 3 * dst.nverts, 3 * src.nverts)]

    ref = out()
    assert _backward(cr, R._core.h, dst, src, x, y, gy, ref, None) == L.CR_OK
    rp, col, val = R._core.csr(False)
    bad, start = [], threading.Barrier(2)
    got = [[out() for _ in range(6)] for _ in range(2)]
    torch.cuda.synchronize()

    def work(t):
        print(f"[case] per-thread stream, thread {t}", flush=True)
        torch.cuda.set_device(0)
        start.wait(timeout=60)
        for g in got[t]:
            st, h = _build(cr, dst, src, PER_THREAD)
            if st != L.CR_OK or _backward(cr, h, dst, src, x, y, gy, g, PER_THREAD) != L.CR_OK:
                bad.append(L.last_error())
                return
            rp2, col2, val2 = (np.empty_like(a) for a in (rp, col, val))
            L.lib.cr_regridder_copy_csr(h, 0, L.i64ptr(rp2), L.i32ptr(col2), L.dptr(val2))
            L.lib.cr_regridder_destroy(h)
            if not (np.array_equal(rp, rp2) and np.array_equal(col, col2) and np.array_equal(val, val2)):
                bad.append("another matrix")

    threads = [threading.Thread(target=work, args=(t,)) for t in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for g in got[0] + got[1]:
        assert torch.equal(g[0], ref[0])
        for a, b in zip(g[1:], ref[1:]):  # sums in any order of a few dozen terms
            assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())
