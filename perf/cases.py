"""Performance cases of the regridding library.

What a program does with it: build a regridder between two grids (online
coupling, moving grids, a new mesh), regrid fields with a regridder it keeps
(one field per call in a time loop, many fields per call in post-processing,
levels stored fastest or cells stored fastest, either direction), and take
gradients through a regrid (mesh optimisation, data assimilation).

Every case is a dict of plain values:

* ``kind``: ``"build"``, ``"regrid"`` or ``"grad"``;
* ``src``, ``dst``: ``"lonlat NI NJ"`` (point matrix), ``"cube NE"`` (six blocks
  of points), ``"healpix NSIDE STEP"`` (nested, STEP boundary points per side);
* ``jitter``: cubed-sphere points moved by N(0, jitter * cell width) and the
  whole sphere rotated, from the seed (0: the regular grid);
* ``dtype``, ``fields``, ``layout``: ``"cells"`` stores each field contiguously
  (``x[k, n]``, the spatial axis is dims=2), ``"levels"`` stores the fields of a
  cell side by side (``x[n, k]``, dims=1);
* ``transpose``: regrid with ``transpose(R)``; ``normalize``: ``Regridder(...;
  normalize)``.

``exact`` computes the same outputs from the same inputs in FP64 torch: the
spherical clip of every overlapping pair, vectorised over pairs, and autograd
through it for the vertex gradients.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import __graft_entry__

cr = __graft_entry__.load_package()


def _case(name, kind, src, dst, dtype="float64", fields=1, layout="cells", transpose=False, normalize=False, jitter=0.0):
    return {"name": name, "kind": kind, "src": src, "dst": dst, "dtype": dtype, "fields": fields, "layout": layout,
            "transpose": transpose, "normalize": normalize, "jitter": jitter}


def listed():
    return [
        # a regridder between two coarse analysis grids, then one field there and back: the smallest build
        _case("build 4deg-5deg", "build", "lonlat 90 45", "lonlat 72 36", normalize=True),
        # a coupler's start-up: a 1 degree atmosphere onto a cubed-sphere model grid
        _case("build 1deg-C48", "build", "lonlat 360 180", "cube 48"),
        # quarter-degree reanalysis onto HEALPix cells with curved edges: the benchmark's build
        _case("build quarter-H256", "build", "lonlat 1440 720", "healpix 256 4"),
        # one field per call between coarse grids, as in a time loop: latency
        _case("field 4deg-5deg", "regrid", "lonlat 90 45", "lonlat 72 36"),
        # one field per call at quarter degree
        _case("field quarter-H256", "regrid", "lonlat 1440 720", "healpix 256 4"),
        # 64 levels x 4 variables in one call, cells fastest: the benchmark's apply
        _case("batch quarter-H256", "regrid", "lonlat 1440 720", "healpix 256 4", "float32", 256),
        # the same fields carried back with the transposed regridder
        _case("batch quarter-H256 T", "regrid", "lonlat 1440 720", "healpix 256 4", "float32", 256, transpose=True),
        # the largest configuration: HEALPix 1024 model output onto a 0.1 degree grid
        _case("batch H1024-tenth", "regrid", "healpix 1024 1", "lonlat 3600 1800", "float32", 64),
        # columns of a model state with the levels fastest (the row-major order of x[n, k]), in FP64
        _case("levels f64 half-C90", "regrid", "lonlat 721 361", "cube 90", "float64", 37, "levels"),
        # the same layout in FP32 at quarter degree, as many levels as do not fill a wave
        _case("levels f32 quarter-H256", "regrid", "lonlat 1440 721", "healpix 256 1", "float32", 50, "levels"),
        # a step of mesh optimisation: a few fields forward, then gradients of fields and of both grids' points
        _case("grad C96-1deg", "grad", "cube 96", "lonlat 360 180", fields=4, layout="levels", jitter=0.05),
        # the benchmark's reverse mode: one field, gradients of all quarter-degree points and HEALPix vertices
        _case("grad quarter-H256", "grad", "lonlat 1440 720", "healpix 256 4"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid_near(rng, kinds, n):
    """A grid of about n cells, of one of the kinds."""
    kind = rng.choice(kinds)
    if kind == "lonlat":
        nj = max(9, int(round(math.sqrt(n / 2.0))))
        return "lonlat %d %d" % (2 * nj + rng.choice((0, 1, -1, 3)), nj)
    if kind == "cube":
        return "cube %d" % max(4, int(round(math.sqrt(n / 6.0))))
    nside = 1 << max(2, int(round(math.log2(max(1.0, math.sqrt(n / 12.0))))))
    return "healpix %d %d" % (nside, rng.choice((1, 2, 4)))


def draw(rng):
    kind = rng.choice(("build", "regrid", "regrid", "grad"))
    n = _log_int(rng, 2000, 700000)
    m = max(1500, min(700000, int(n * math.exp(rng.uniform(math.log(0.3), math.log(3.0))))))
    if kind == "grad":
        # sources whose points lie in general position, where the gradient is defined everywhere
        return {k: v for k, v in _case("", kind, _grid_near(rng, ("cube",), n), _grid_near(rng, ("lonlat",), m),
                                       fields=rng.choice((1, 1, 2, 3, 5)), layout=rng.choice(("cells", "levels")),
                                       jitter=rng.uniform(0.02, 0.08)).items() if k != "name"}
    src = _grid_near(rng, ("lonlat", "lonlat", "cube", "healpix"), n)
    dst = _grid_near(rng, ("lonlat", "cube") + (() if src.startswith("healpix") else ("healpix",)), m)
    c = _case("", kind, src, dst, transpose=kind == "regrid" and rng.random() < 0.4, normalize=rng.random() < 0.3,
              jitter=rng.choice((0.0, rng.uniform(0.02, 0.08))))
    if kind == "regrid":
        c["dtype"] = rng.choice(("float64", "float32", "float32"))
        cells = _cells(src) + _cells(dst)
        item = 8 if c["dtype"] == "float64" else 4
        most = min(300, int(2e9 / (cells * item)))  # the largest listed case moves 4.9 GB of fields
        c["fields"] = 1 if rng.random() < 0.25 else _log_int(rng, 2, max(3, most))
        c["layout"] = rng.choice(("cells", "levels"))
    del c["name"]
    return c


# ---------------------------------------------------------------- inputs --
def _spec(text):
    kind, *sizes = text.split()
    return kind, [int(s) for s in sizes]


def _cells(text):
    kind, s = _spec(text)
    return s[0] * s[1] if kind == "lonlat" else 6 * s[0] * s[0] if kind == "cube" else 12 * s[0] * s[0]


def _sincos_degrees(deg):
    q = np.rint(deg / 90.0)
    r = np.radians(deg - 90.0 * q)
    s, c, m = np.sin(r), np.cos(r), q.astype(np.int64) % 4
    return np.choose(m, (s, c, -s, -c)), np.choose(m, (c, -s, -c, s))


@functools.lru_cache(maxsize=8)
def _lonlat_points(ni, nj):
    """P[i, j] of the globe, south to north, west to east; exact at the poles and where the longitudes close."""
    sl, cl = _sincos_degrees(np.arange(ni + 1) * (360.0 / ni))
    sl[-1], cl[-1] = sl[0], cl[0]
    sp, cp = _sincos_degrees(-90.0 + np.arange(nj + 1) * (180.0 / nj))
    sp[-1], cp[-1] = 1.0, 0.0
    out = np.empty((nj + 1, ni + 1, 3))
    out[..., 0], out[..., 1], out[..., 2] = cp[:, None] * cl, cp[:, None] * sl, sp[:, None]
    return out.transpose(1, 0, 2)


def _cube_points(ne, jitter, seed):
    """Equiangular cubed sphere P[face, i, j]; with a jitter, its inner points moved and the whole rotated."""
    t = np.tan((np.arange(ne + 1) / ne - 0.5) * (math.pi / 2))
    t[0], t[-1] = -1.0, 1.0
    t = 0.5 * (t - t[::-1])
    normal = np.array([[1, 0, 0], [0, 1, 0], [-1, 0, 0], [0, -1, 0], [0, 0, 1], [0, 0, -1]], float)
    along_i = np.array([[0, 1, 0], [-1, 0, 0], [0, -1, 0], [1, 0, 0], [0, 1, 0], [0, 1, 0]], float)
    along_j = np.cross(normal, along_i)
    p = normal[:, None, None] + t[None, None, :, None] * along_i[:, None, None] + t[None, :, None, None] * along_j[:, None, None]
    p /= np.linalg.norm(p, axis=-1, keepdims=True)  # [face, j, i]
    if jitter:
        rng = np.random.default_rng(seed)
        inner = p[:, 1:-1, 1:-1]
        step = rng.normal(0.0, jitter * math.pi / 2 / ne, inner.shape)
        step -= (step * inner).sum(-1, keepdims=True) * inner
        p[:, 1:-1, 1:-1] = inner + step
        q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        p = p @ (q * np.linalg.det(q))
        # the blocks' shared edges come from the same sums only up to rounding: that is a model's own grid too
        p /= np.linalg.norm(p, axis=-1, keepdims=True)
    return p.transpose(0, 2, 1, 3)


def _points(text, jitter, seed):
    """The host point matrix of a grid, None for a HEALPix grid (made by the library from its nside)."""
    kind, s = _spec(text)
    return _lonlat_points(*s) if kind == "lonlat" else _cube_points(s[0], jitter, seed) if kind == "cube" else None


def _grid(text, points):
    if points is not None:
        return cr.Grid.from_points(points)
    _, (nside, step) = _spec(text)
    return cr.Grid.healpix(nside, "nested", step=step)


def _field(case, n, seed):
    """U[0, 1) fields, as the benchmark's single-field configurations have them."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    k = case["fields"]
    shape = (n,) if k == 1 else (k, n) if case["layout"] == "cells" else (n, k)
    return torch.rand(shape, generator=g, dtype=getattr(torch, case["dtype"]), device="cuda")


def _ends(case):
    """(source, destination) cells of the direction that is regridded."""
    ends = _cells(case["src"]), _cells(case["dst"])
    return ends[::-1] if case["transpose"] else ends


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case = case
    s.src_points = _points(case["src"], case["jitter"], 3 * seed)
    s.dst_points = _points(case["dst"], case["jitter"], 3 * seed + 1)
    n_from, n_to = _ends(case)
    s.x = _field(case, n_from, 2 * seed)
    if case["kind"] == "build":
        return s
    s.src, s.dst = _grid(case["src"], s.src_points), _grid(case["dst"], s.dst_points)
    s.R = cr.Regridder(s.dst, s.src, normalize=case["normalize"])
    if case["kind"] == "grad":
        g = torch.Generator(device="cuda").manual_seed(2 * seed + 1)
        if case["fields"] > 1 and case["layout"] == "cells":  # regrid_backward takes cells along the first axis
            s.x = s.x.t()
        s.gy = torch.randn((n_to,) + s.x.shape[1:], generator=g, dtype=torch.float64, device="cuda")
    else:
        if case["transpose"]:
            s.R = cr.transpose(s.R)
        s.dims = 2 if s.x.ndim == 2 and case["layout"] == "cells" else 1
        shape = list(s.x.shape)
        shape[s.dims - 1] = n_to
        s.y = torch.zeros(shape, dtype=s.x.dtype, device="cuda")
    return s


def run(s):
    kind = s.case["kind"]
    if kind == "regrid":
        return cr.regrid_(s.y, s.R, s.x, dims=s.dims)
    if kind == "build":
        dst, src = _grid(s.case["dst"], s.dst_points), _grid(s.case["src"], s.src_points)
        R = cr.Regridder(dst, src, normalize=s.case["normalize"])
        y = cr.regrid(R, s.x)
        return {"there": y, "back": cr.regrid(cr.transpose(R), y)}
    y = cr.regrid(s.R, s.x)
    gx, g_dst, g_src = cr.regrid_backward(s.R, s.dst, s.src, s.x, y, s.gy)
    return {"y": y, "gx": gx, "g_dst": g_dst, "g_src": g_src}


# ------------------------------------------------------------------ work --
def _edge_length(text):
    """Total length of a grid's edges on the unit sphere."""
    kind, s = _spec(text)
    return math.pi * s[0] + 4.0 * s[1] if kind == "lonlat" else 2.0 * math.sqrt(4.0 * math.pi * _cells(text))


def _overlaps(case):
    """About how many pairs of cells overlap: the faces of the two grids' overlay are the cells of both plus the
    crossings of their edges, of which lengths L1 and L2 in general position have 2/pi L1 L2 / area (Buffon)."""
    x = 2.0 / math.pi * _edge_length(case["src"]) * _edge_length(case["dst"]) / (4.0 * math.pi)
    return _cells(case["src"]) + _cells(case["dst"]) + x


def _vertices(text):
    kind, s = _spec(text)
    return (s[0] + 1) * (s[1] + 1) if kind == "lonlat" else 6 * (s[0] + 1) ** 2 if kind == "cube" else 48 * s[0] * s[0] * s[1]


def work(case):
    """Bytes and operations of one pass: every input and output once.  The matrix is 12 bytes a pair, a row pointer
    and an area 16 bytes a cell; a pair's clip and area take about 600 FP64 operations (their reverse mode twice
    that), a product and sum 2 per pair and field."""
    pairs, (n_from, n_to) = _overlaps(case), _ends(case)
    k, item = case["fields"], 8 if case["dtype"] == "float64" else 4
    matrix = 12.0 * pairs + 16.0 * n_to
    fields = float(k) * item * (n_from + n_to)
    if case["kind"] == "regrid":
        return {"bytes": matrix + fields, "flops": 2.0 * pairs * k}
    host = sum(24.0 * _vertices(t) for t in (case["src"], case["dst"]) if not t.startswith("healpix"))
    if case["kind"] == "build":  # CSR(A), CSR(A^T) and both areas come out, then a field goes there and back
        return {"bytes": host + 2 * 12.0 * pairs + 16.0 * (n_from + n_to) + 8.0 * (2 * n_to + n_from),
                "flops": (600.0 + 4.0) * pairs}
    verts = 24.0 * (_vertices(case["src"]) + _vertices(case["dst"]))
    return {"bytes": 2 * matrix + 2 * fields + 8.0 * k * (n_from + n_to) + 2 * verts, "flops": (1200.0 + 6.0 * k) * pairs}


# ----------------------------------------------------------------- exact --
def _healpix_vertices(nside, step):
    """Boundary points of the nested pixels, counter-clockwise from the north corner (Gorski et al. 2005)."""
    pix = torch.arange(12 * nside * nside, device="cuda")
    face, q = pix // (nside * nside), pix % (nside * nside)
    ix, iy = torch.zeros_like(q), torch.zeros_like(q)
    for b in range(nside.bit_length()):
        ix |= ((q >> (2 * b)) & 1) << b
        iy |= ((q >> (2 * b + 1)) & 1) << b
    M = nside * step
    row, colm = face // 4, face % 4
    jr, jp = 2 + row, torch.where(row == 1, 2 * colm, 2 * colm + 1)
    out = torch.empty(pix.numel(), 4 * step, 3, dtype=torch.float64, device="cuda")
    for v in range(4 * step):
        side, o = divmod(v, step)
        u, w = (((ix + 1) * step - o, (iy + 1) * step), (ix * step, (iy + 1) * step - o),
                (ix * step + o, iy * step), ((ix + 1) * step, iy * step + o))[side]
        K = jr * M - u - w
        cap = torch.minimum(K, 4 * M - K)
        polar = cap < M
        t = (cap * cap).double() / (3.0 * M * M)
        z = torch.where(polar, torch.where(K < M, 1.0 - t, t - 1.0), (2 * (2 * M - K)).double() / (3.0 * M))
        sth = torch.where(polar, (t * (2.0 - t)).sqrt(), ((1.0 - z) * (1.0 + z)).clamp_min(0).sqrt())
        phi = (math.pi / 4) * torch.where(polar, jp + (u - w).double() / cap.clamp_min(1), (jp * M + u - w).double() / M)
        out[:, v] = torch.stack((sth * torch.cos(phi), sth * torch.sin(phi), z), -1)
    return out.reshape(-1, 3)


def _mesh(text, points):
    """(vertices, rings): unit vectors (nv, 3) and the vertex numbers of every cell, counter-clockwise."""
    if points is None:
        _, (nside, step) = _spec(text)
        v = _healpix_vertices(nside, step)
        return v, torch.arange(v.shape[0], device="cuda").view(-1, 4 * step)
    p = points[None] if points.ndim == 3 else points
    v = torch.from_numpy(np.ascontiguousarray(p.transpose(0, 2, 1, 3))).cuda()  # [block, j, i]
    idx = torch.arange(v[..., 0].numel(), device="cuda").view(v.shape[:3])
    ring = torch.stack((idx[:, :-1, :-1], idx[:, :-1, 1:], idx[:, 1:, 1:], idx[:, 1:, :-1]), -1)
    return v.reshape(-1, 3), ring.reshape(-1, 4)


def _dot(a, b):
    return (a * b).sum(-1)


def _fan_area(ring, count=None):
    """Solid angle of each ring (N, V, 3), its first `count` vertices: triangles from its first vertex (Van Oosterom
    and Strackee 1983)."""
    a, b, c = ring[:, :1], ring[:, 1:-1], ring[:, 2:]
    num = _dot(a, torch.linalg.cross((b - a), (c - a)))
    tri = 2.0 * torch.atan2(num, 1.0 + _dot(a, b) + _dot(b, c) + _dot(c, a))
    if count is not None:
        k = torch.arange(2, ring.shape[1], device=ring.device)
        tri = torch.where(k < count[:, None], tri, torch.zeros_like(tri))
    return tri.sum(1)


def _clip_area(subject, clip):
    """Area of each subject ring (N, V, 3) inside its convex clip ring (N, C, 3), both counter-clockwise."""
    n = subject.shape[0]
    ring, count = subject, torch.full((n,), subject.shape[1], device=subject.device)
    for e in range(clip.shape[1]):
        a, b = clip[:, e], clip[:, (e + 1) % clip.shape[1]]
        normal = torch.linalg.cross(a, b - a)
        flat = _dot(normal, normal) < 1e-26  # two corners at a pole: no edge
        V = ring.shape[1]
        k = torch.arange(V, device=ring.device)
        live = k < count[:, None]
        nxt = torch.where(k + 1 < count[:, None], k + 1, torch.zeros_like(k))
        side = _dot(normal[:, None], ring - a[:, None])
        side = torch.where(flat[:, None], torch.ones_like(side), side)
        after, side_after = ring.gather(1, nxt[..., None].expand(-1, -1, 3)), side.gather(1, nxt)
        keep = live & (side >= 0)
        cross = live & ((side >= 0) != (side_after >= 0))
        p, q = torch.where(cross, side.abs(), torch.ones_like(side)), torch.where(cross, side_after.abs(), torch.ones_like(side))
        point = q[..., None] * ring + p[..., None] * after
        point = torch.where(cross[..., None], point, ring)
        point = point / _dot(point, point).sqrt()[..., None]
        both = torch.stack((ring, point), 2).reshape(n, 2 * V, 3)
        mask = torch.stack((keep, cross), 2).reshape(n, 2 * V)
        count = mask.sum(1)
        width = max(3, int(count.max())) if n else 3
        at = torch.where(mask, mask.cumsum(1) - 1, torch.full_like(mask, width, dtype=torch.long))
        ring = torch.zeros(n, width + 1, 3, dtype=both.dtype, device=both.device)
        ring = ring.scatter(1, at[..., None].expand(-1, -1, 3), both)[:, :width]
    # unused places hold zeros: their triangles are masked, but must not make a 0/0 gradient
    used = (torch.arange(ring.shape[1], device=ring.device) < count[:, None])[..., None]
    ring = torch.where(used, ring, torch.tensor([1.0, 0.0, 0.0], dtype=ring.dtype, device=ring.device))
    return _fan_area(ring, count)


def _pairs(cells1, cells2):
    """Yields (i, j) of the cells whose bounding balls meet, in blocks: i of the first table, j of the second."""
    def balls(cells):
        c = cells.mean(1)
        c = c / c.norm(dim=1, keepdim=True)
        return c, (cells - c[:, None]).norm(dim=2).max(1).values * (1 + 1e-9) + 1e-12

    (c1, r1), (c2, r2) = balls(cells1), balls(cells2)
    size = float(r1.max() + r2.max())
    W = int(2.0 / size) + 4
    vox = lambda c: ((c + 1.0) / size).long() + 1  # noqa: E731
    key = lambda v: (v[..., 0] * W + v[..., 1]) * W + v[..., 2]  # noqa: E731
    k2, order = key(vox(c2)).sort()
    d = torch.arange(-1, 2, device=c1.device)
    around = torch.cartesian_prod(d, d, d)
    q = key(vox(c1)[:, None] + around)  # (n1, 27)
    lo, hi = torch.searchsorted(k2, q), torch.searchsorted(k2, q, right=True)
    total = (hi - lo).sum(1).cumsum(0)
    block, at = 20_000_000, 0
    while at < c1.shape[0]:
        done = int(total[at - 1]) if at else 0
        end = max(at + 1, int(torch.searchsorted(total, torch.tensor(done + block, device=total.device))))
        l, m = lo[at:end].reshape(-1), (hi - lo)[at:end].reshape(-1)
        which = torch.repeat_interleave(torch.arange(l.numel(), device=l.device), m)
        j = order[l[which] + torch.arange(which.numel(), device=l.device) - (m.cumsum(0) - m)[which]]
        i = at + which // 27
        near = (c1[i] - c2[j]).norm(dim=1) <= r1[i] + r2[j]
        i, j = i[near], j[near]
        for k in range(0, i.numel(), 1_000_000):
            yield i[k:k + 1_000_000], j[k:k + 1_000_000]
        at = end


def exact(case, seed):
    points = _points(case["src"], case["jitter"], 3 * seed), _points(case["dst"], case["jitter"], 3 * seed + 1)
    (v_src, ring_src), (v_dst, ring_dst) = _mesh(case["src"], points[0]), _mesh(case["dst"], points[1])
    convex_dst = ring_dst.shape[1] == 4
    cells_src, cells_dst = v_src[ring_src], v_dst[ring_dst]
    x = _field(case, _ends(case)[0], 2 * seed).double()
    if case["fields"] > 1 and case["layout"] == "cells":
        x = x.t()
    x = x.reshape(x.shape[0], -1)
    area_src, area_dst = _fan_area(cells_src), _fan_area(cells_dst)

    def clip(i, j, src, dst):
        s, d = src[ring_src[j]], dst[ring_dst[i]]
        return _clip_area(s, d) if convex_dst else _clip_area(d, s)

    blocks = [(i, j, clip(i, j, v_src, v_dst)) for i, j in _pairs(cells_dst, cells_src)]
    if case["kind"] != "grad":  # a grad case clips them again
        blocks = [(i[a != 0], j[a != 0], a[a != 0]) for i, j, a in blocks]

    def product(x, back):
        n_to = (cells_src if back else cells_dst).shape[0]
        y = torch.zeros(n_to, x.shape[1], dtype=torch.float64, device="cuda")
        for f in range(0, x.shape[1], 16):
            xf = x[:, f:f + 16].contiguous()
            yf = torch.zeros(n_to, xf.shape[1], dtype=torch.float64, device="cuda")
            for i, j, a in blocks:
                yf.index_add_(0, j if back else i, a[:, None] * xf[i if back else j])
            y[:, f:f + 16] = yf
        return y

    def shaped(y, like_x=False):
        if case["fields"] == 1:
            return y[:, 0]
        return y.t().contiguous() if case["layout"] == "cells" and not like_x else y

    if case["kind"] == "regrid":
        area = area_src if case["transpose"] else area_dst
        return shaped(product(x, case["transpose"]) / area[:, None])
    y = product(x, False) / area_dst[:, None]
    if case["kind"] == "build":
        return {"there": shaped(y), "back": shaped(product(y, True) / area_src[:, None])}
    g = torch.Generator(device="cuda").manual_seed(2 * seed + 1)
    shape = (area_dst.shape[0],) + ((case["fields"],) if case["fields"] > 1 else ())
    gy = torch.randn(shape, generator=g, dtype=torch.float64, device="cuda").view(area_dst.shape[0], -1)
    gx = product(gy / area_dst[:, None], True)
    raw_src, raw_dst = v_src.clone().requires_grad_(), v_dst.clone().requires_grad_()
    for i, j, _ in blocks:
        src, dst = (v / v.norm(dim=1, keepdim=True) for v in (raw_src, raw_dst))
        weight = ((gy / area_dst[:, None])[i] * x[j]).sum(1)
        (weight * clip(i, j, src, dst)).sum().backward()
    dst = raw_dst / raw_dst.norm(dim=1, keepdim=True)
    (-((gy * y).sum(1) / area_dst) * _fan_area(dst[ring_dst])).sum().backward()
    # on the regular grids some vertices lie on the other grid's edges, where the area has only one-sided derivatives
    general = case["jitter"] > 0
    return {"y": shaped(y, True), "gx": shaped(gx, True), "g_dst": raw_dst.grad if general else None,
            "g_src": raw_src.grad if general else None}
