"""Vertex gradients by boundary arcs at the sizes where the kernel takes another
path, against the oracle's forward-mode dual numbers assembled pair by pair
(dL/dA_ij dA_ij/dV over the pairs plus the area term), on grids turned to
general position: 16-gons and 48-gons clipped by quads (masks of 32 and 64
bits), hexagons and padded pentagons clipping (8 clip lines, lines without a
length), a clipped source of more vertices than a pair keeps, rows of one or two
non-zeros (more rows in a wave than its window holds), a pole inside."""
import numpy as np
import pytest
import torch

from polygrids import geodesic_dual, rotation

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _table(cells):
    n, nv = cells.shape[:2]
    return cells.reshape(-1, 3), np.arange(0, n * nv + 1, nv), np.arange(n * nv, dtype=np.int32)


def _lonlat(cr, ni, nj, seed):
    P = cr.lonlat_points(ni, nj)
    if seed is not None:
        P = P @ rotation(seed).T
    v = np.ascontiguousarray(P.transpose(1, 0, 2)).reshape(-1, 3)
    i, j = np.meshgrid(np.arange(ni), np.arange(nj), indexing="xy")
    a = (i + j * (ni + 1)).reshape(-1)
    idx = np.stack([a, a + 1, a + ni + 2, a + ni + 1], 1).reshape(-1).astype(np.int32)
    return v, np.arange(0, 4 * ni * nj + 1, 4), idx


# name: (destination polygons, convex, source polygons, convex)
def _grids(cr, name):
    hp = lambda nside, step: _table(cr.healpix_cells(nside, "nested", step))  # noqa: E731
    return {
        "16-gons over quads": (hp(4, 4), False, _lonlat(cr, 24, 12, 1), True),
        "48-gons over quads": (hp(2, 12), False, _lonlat(cr, 18, 9, 2), True),
        "quads over 16-gons": (_lonlat(cr, 40, 20, 3), True, hp(2, 4), False),
        "short rows": (_lonlat(cr, 60, 30, 4), True, _lonlat(cr, 13, 6, 5), True),
        "hexagons over 16-gons": (geodesic_dual(2, rotation(6)), True, hp(4, 4), False),
        "quads over hexagons": (_lonlat(cr, 30, 15, None), True, geodesic_dual(2, rotation(7)), True),
    }[name]


@pytest.mark.parametrize("name", ["16-gons over quads", "48-gons over quads", "quads over 16-gons", "short rows",
                                  "hexagons over 16-gons", "quads over hexagons"])
def test_arcs_match_dual_numbers(cr, orc, name):
    print(f"[case] arcs {name}", flush=True)
    (dv, doff, didx), dconv, (sv, soff, sidx), sconv = _grids(cr, name)
    dst = cr.Grid.from_polygons(dv, doff, didx, convex=dconv)
    src = cr.Grid.from_polygons(sv, soff, sidx, convex=sconv)
    R = cr.Regridder(dst, src, radius=1.0)
    dcells, dvi = cr.polygons_to_cells(dv, doff, didx)
    scells, svi = cr.polygons_to_cells(sv, soff, sidx)
    rng = np.random.default_rng(9)
    s, w = rng.random((src.ncells, 2)), rng.standard_normal((dst.ncells, 2))
    x, gy = torch.tensor(s, device=DEV), torch.tensor(w, device=DEV)
    y = cr.regrid(R, x)
    _, g_dst, g_src = cr.regrid_backward(R, dst, src, x, y, gy, field_grad=False)

    clip_is_dst = bool(R.stats()["clip_with_dst"])
    ref = orc.build(dcells, scells, clip_is_dst=clip_is_dst)
    row, col = ref.row_index(), ref.col
    coef = (w[row] * s[col]).sum(1) / ref.a_dst[row]
    d = np.zeros((dst.ncells, 2))
    np.add.at(d, row, ref.val[:, None] * s[col])
    d /= ref.a_dst[:, None]
    want_dst, want_src = np.zeros((dst.nverts, 3)), np.zeros((src.nverts, 3))
    for k in range(row.size):
        i, j = row[k], col[k]
        if clip_is_dst:
            _, gs, gd = orc.clip_area_grad(scells[j], dcells[i])
        else:
            _, gd, gs = orc.clip_area_grad(dcells[i], scells[j])
        np.add.at(want_dst, dvi[i], coef[k] * gd)
        np.add.at(want_src, svi[j], coef[k] * gs)
    for i in range(dst.ncells):
        _, ga = orc.polygon_area_grad(dcells[i])
        np.add.at(want_dst, dvi[i], -(w[i] * d[i]).sum() / ref.a_dst[i] * ga)
    for got, want in ((g_dst, want_dst), (g_src, want_src)):
        scale = np.abs(want).max()
        np.testing.assert_allclose(got.cpu().numpy(), want, rtol=0, atol=1e-9 * scale)
