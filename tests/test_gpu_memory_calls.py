"""Device memory between calls: two threads on hipStreamPerThread (one handle, two
streams), calls on a stream that is being captured, and builds beside a capture on
another thread."""
import ctypes
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
PER_THREAD = 2  # hipStreamPerThread


def _hip():
    torch.ones(1, device=DEV)
    with open("/proc/self/maps") as f:
        return ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))


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


class _Capture:
    """A capture on a stream of its own: mode 1 is hipStreamCaptureModeThreadLocal."""

    def __init__(self, mode):
        self.hip, self.s, self.mode = _hip(), ctypes.c_void_p(), mode
        assert self.hip.hipStreamCreateWithFlags(ctypes.byref(self.s), 1) == 0

    def __enter__(self):
        torch.cuda.synchronize()
        assert self.hip.hipStreamBeginCapture(self.s, self.mode) == 0
        return self

    def active(self):
        st = ctypes.c_int()
        return self.hip.hipStreamIsCapturing(self.s, ctypes.byref(st)) == 0 and st.value == 1

    def __exit__(self, *exc):
        g = ctypes.c_void_p()
        self.ended = self.hip.hipStreamEndCapture(self.s, ctypes.byref(g))
        if g.value:
            self.hip.hipGraphDestroy(g)
        self.hip.hipStreamDestroy(self.s)


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_allocating_calls_are_refused_on_a_capturing_stream(cr, mode):
    print(f"[case] refused while capturing, mode {mode}", flush=True)
    L = cr._lib
    dst, src = _grids(cr, 12)
    R = cr.Regridder(dst, src)
    x, gy = torch.ones(src.ncells, dtype=torch.float64, device=DEV), torch.ones(dst.ncells, dtype=torch.float64, device=DEV)
    y = cr.regrid(R, x)
    g = [torch.zeros(n, dtype=torch.float64, device=DEV) for n in (src.ncells, 3 * dst.nverts, 3 * src.nverts)]
    pts = np.ascontiguousarray(cr.lonlat_points(12, 6).transpose(1, 0, 2))
    with _Capture(mode) as c:
        h = ctypes.c_void_p()
        got = [_build(cr, dst, src, c.s)[0],
               _backward(cr, R._core.h, dst, src, x, y, gy, g, c.s),
               L.lib.cr_regridder_normalize(R._core.h, c.s),
               L.lib.cr_regrid_prepare(R._core.h, 0, L.CR_F64, 1, 1, 1, c.s),
               L.lib.cr_grid_healpix(ctypes.byref(h), 4, 0, 2, c.s),
               L.lib.cr_grid_from_points(ctypes.byref(h), L.dptr(pts), 1, 12, 6, c.s)]
        active, message = c.active(), L.last_error()
    assert got == [L.CR_UNSUPPORTED] * len(got) and "captured" in message
    assert active and c.ended == 0  # the capture goes on without them
    assert _backward(cr, R._core.h, dst, src, x, y, gy, g, None) == L.CR_OK


@pytest.mark.parametrize("mode", [1, 2])
def test_builds_beside_a_capture_on_another_thread(cr, mode):
    print(f"[case] builds beside a capture, mode {mode}", flush=True)
    L = cr._lib
    dst, src = _grids(cr, 24)
    x = torch.ones(src.ncells, dtype=torch.float64, device=DEV)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    bad = []

    def work():
        torch.cuda.set_device(0)
        for _ in range(3):  # from the second on with blocks of a handle used on the side stream
            st, h = _build(cr, dst, src, side.cuda_stream)
            y = torch.empty(dst.ncells, dtype=torch.float64, device=DEV)
            if st != L.CR_OK or L.lib.cr_regrid(h, 0, L.CR_F64, 1, x.data_ptr(), 1, 1, y.data_ptr(), 1, 1, 1,
                                                side.cuda_stream) != L.CR_OK:
                bad.append(L.last_error())
            L.lib.cr_regridder_destroy(h)

    work()  # memory for y, and what is made once
    torch.cuda.synchronize()
    with _Capture(mode) as c:
        t = threading.Thread(target=work)
        t.start()
        t.join()
        active = c.active()
    assert active and c.ended == 0 and not bad
    torch.cuda.synchronize()
