"""Vertex gradients of cells that touch, each pair of cells by itself (far from the
others)."""
import numpy as np
import pytest
import torch

from test_arcs_host import EPS, around, around_and_cut, plane

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _polygons(rings):
    n = np.array([len(r) for r in rings])
    return np.concatenate(rings), np.concatenate(([0], np.cumsum(n))), np.arange(n.sum(), dtype=np.int32)


def _pair_grads(cr, dst_rings, src_rings, src_convex, **kw):
    """Gradients of sum(A_ii) for one destination and one source cell at each place."""
    dst = cr.Grid.from_polygons(*_polygons(dst_rings), convex=True)
    src = cr.Grid.from_polygons(*_polygons(src_rings), convex=src_convex)
    R = cr.Regridder(dst, src, radius=1.0, **kw)
    assert R.stats()["clip_with_dst"]
    x, gy = (torch.ones(n, dtype=torch.float64, device=DEV) for n in (src.ncells, dst.ncells))
    _, g_dst, g_src = cr.regrid_backward(R, dst, src, x, None, gy, normalize=False, field_grad=False)
    return R, g_dst.cpu().numpy(), g_src.cpu().numpy()


@pytest.mark.parametrize("shape", [around, around_and_cut])
def test_reflex_vertex_at_a_clip_edge(cr, orc, shape):
    print(f"[case] reflex vertex {shape.__name__}", flush=True)
    square, h = [(0.0, 0.0), (1.0, 0.0), (1.0, 1.0), (0.0, 1.0)], 0.01
    dst, src = [], []
    for i, eps in enumerate(EPS):
        dst.append(np.roll(plane(square, h, 100 + i), i % 4, axis=0))
        src.append(plane(shape(eps), h, 100 + i))
    R, g_dst, g_src = _pair_grads(cr, dst, src, False)
    A = R.intersections
    assert A.nnz == len(EPS)  # every cell meets its partner alone
    for i in range(len(EPS)):
        _, gs, gd = orc.clip_area_grad(src[i], dst[i])
        tol = 1e-9 * np.abs(gd).max()  # decisions within ~1e-10 edge lengths may go either way
        assert np.abs(g_dst[4 * i:4 * i + 4] - gd).max() <= tol, EPS[i]
        n = len(src[i])
        assert np.abs(g_src[n * i:n * i + n] - gs).max() <= tol, EPS[i]


def test_cells_that_only_touch(cr):
    """A vertex of the source quad on an edge of the destination quad, from outside:
    whether rounding makes that a pair (threshold_rel = 0 keeps every sliver) or not,
    the gradient is that of a sliver."""
    print("[case] touching cells", flush=True)
    rng = np.random.default_rng(7)
    h, square = 0.004, np.array([(0.0, 0.0), (1.0, 0.0), (1.0, 1.0), (0.0, 1.0)])
    dst, src = [], []
    for lat in np.linspace(-1.2, 1.2, 100):
        for lon in np.linspace(0.0, 2 * np.pi, 60, endpoint=False):
            c = np.array([np.cos(lat) * np.cos(lon), np.cos(lat) * np.sin(lon), np.sin(lat)])
            u = np.cross(c, rng.standard_normal(3))
            u /= np.linalg.norm(u)
            frame = np.stack([u, np.cross(c, u), c])
            place = lambda xy: (lambda p: p / np.linalg.norm(p, axis=1, keepdims=True))(  # noqa: E731
                np.concatenate([h * np.asarray(xy), np.ones((len(xy), 1))], 1) @ frame)
            d, turn, t = place(square), int(rng.integers(4)), rng.uniform(0.1, 0.9)
            tip = (1 - t) * d[0] + t * d[1]
            dst.append(np.roll(d, turn, axis=0))
            src.append(np.concatenate([(tip / np.linalg.norm(tip))[None],
                                       place([(t - 0.4, -0.6), (t + 0.1, -1.0), (t + 0.5, -0.5)])]))
    R, g_dst, g_src = _pair_grads(cr, dst, src, True, threshold_rel=0.0)
    assert R.intersections.nnz > 100
    # a sliver of depth d has a derivative of the order of d (1e-16 here); the whole cell's is h / 2
    assert max(np.abs(g_dst).max(), np.abs(g_src).max()) <= 1e-9 * h
