"""Device memory handed on from released handles and temporaries: work still
pending on other streams when a handle is destroyed, and builds on several
threads and streams at once, give the results of undisturbed runs bit for bit."""
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _regridder(cr, nlon, nlat, ne):
    return cr.Regridder(cr.Grid.from_points(cr.cubed_sphere_points(ne)), cr.Grid.from_points(cr.lonlat_points(nlon, nlat)))


def _pass(cr, nlon, nlat, ne, x, stream):
    """Build on the stream, regrid there and back without a synchronisation, drop the handles."""
    with torch.cuda.stream(stream):
        R = _regridder(cr, nlon, nlat, ne)
        y = cr.regrid(R, x)
        return y, cr.regrid(cr.transpose(R), y)


def test_handle_destroyed_with_work_pending(cr):
    sizes = [(144, 72, 24), (360, 180, 48), (288, 144, 40)]
    xs = [torch.tensor(np.random.default_rng(i).random(a * b), device=DEV) for i, (a, b, _) in enumerate(sizes)]
    torch.cuda.synchronize()
    main = torch.cuda.current_stream()
    ref = []
    for s, x in zip(sizes, xs):
        y, z = _pass(cr, *s, x, main)
        torch.cuda.synchronize()
        ref.append((y.clone(), z.clone()))
    side = [torch.cuda.Stream(), torch.cuda.Stream()]
    for rep in range(3):
        print(f"[case] pending rep={rep}", flush=True)
        got = [_pass(cr, *s, x, side[(i + rep) % 2]) for i, (s, x) in enumerate(zip(sizes, xs))]
        torch.cuda.synchronize()
        for (y, z), (ry, rz) in zip(got, ref):
            assert torch.equal(y, ry) and torch.equal(z, rz)


def test_builds_on_several_threads(cr):
    print("[case] threads", flush=True)
    x = torch.tensor(np.random.default_rng(5).random(180 * 90), device=DEV)
    ref = _pass(cr, 180, 90, 30, x, torch.cuda.current_stream())
    torch.cuda.synchronize()
    bad = []

    def work(stream):
        for _ in range(4):
            y, z = _pass(cr, 180, 90, 30, x, stream)
            stream.synchronize()
            if not (torch.equal(y, ref[0]) and torch.equal(z, ref[1])):
                bad.append("differs")

    threads = [threading.Thread(target=work, args=(torch.cuda.Stream(),)) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
