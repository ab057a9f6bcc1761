"""The reverse mode's boundary arcs at touching configurations, on the host: every
pair is either declined (the clip pipeline takes it) or has the gradient of the
oracle's dual numbers."""
import numpy as np
import pytest

import arcs_host
from polygrids import rotation


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    return arcs_host.load(tmp_path_factory.mktemp("arcs"))


def plane(xy, h, seed):
    """Points (x, y) of a plane, h wide, as unit vectors in general position."""
    xy = np.asarray(xy, dtype=np.float64)
    p = np.concatenate([h * xy, np.ones((len(xy), 1))], 1)
    p /= np.linalg.norm(p, axis=1, keepdims=True)
    return p @ rotation(seed).T


EPS = [0.0] + [s * e for e in (1e-15, 1e-14, 1e-13, 1e-12, 1e-11, 3e-11, 1e-10, 1e-9, 1e-6, 1e-3) for s in (1, -1)]


# the subject around the unit square, a reflex vertex `eps` inside the square's lower edge (or outside it)
def around(eps):
    return [(0.45, eps), (2.0, -1.0), (2.0, 2.0), (-1.0, 2.0), (-1.0, -1.0)]


# ... which also cuts the square's upper right corner off
def around_and_cut(eps):
    return [(0.45, eps), (2.0, -1.0), (2.0, 0.3), (0.3, 2.0), (-1.0, 2.0), (-1.0, -1.0)]


@pytest.mark.parametrize("shape", [around, around_and_cut])
@pytest.mark.parametrize("seed", range(4))
def test_reflex_vertex_at_a_clip_edge(host, orc, shape, seed):
    square = [(0.0, 0.0), (1.0, 0.0), (1.0, 1.0), (0.0, 1.0)]
    for h in (0.3, 0.01):
        clip = plane(square, h, seed)
        for eps in EPS:
            for turn in range(4):  # the edge's number among the clip edges
                c, subj = np.roll(clip, turn, axis=0), plane(shape(eps), h, seed)
                got = arcs_host.grad(host, subj, c)
                if got is None:
                    continue
                _, gs, gc = orc.clip_area_grad(subj, c)
                # decisions within ~1e-10 edge lengths may go either way
                for g, want in zip(got, (gs, gc)):
                    assert np.abs(g - want).max() <= 1e-9 * np.abs(gc).max(), (h, eps, turn)


def test_cells_that_only_touch(host):
    """A vertex of a quad on a clip edge from outside: rounding decides whether the
    intersection is empty or a sliver of ~1e-16 edge lengths; its gradient is small
    either way."""
    rng = np.random.default_rng(3)
    square, planned, slivers = np.array([(0.0, 0.0), (1.0, 0.0), (1.0, 1.0), (0.0, 1.0)]), 0, 0
    for it in range(60000):
        if it % 100 == 0:
            seed, turn = int(rng.integers(1 << 30)), int(rng.integers(4))
            clip = np.roll(plane(square, 0.01, seed), turn, axis=0)
        # the touching vertex: a point of the clip edge as the doubles have it
        t = rng.uniform(0.1, 0.9)
        k = (0 + turn) % 4
        tip = (1 - t) * clip[k] + t * clip[(k + 1) % 4]
        tip /= np.linalg.norm(tip)
        rest = plane([(t - 0.4, -0.6), (t + 0.1, -1.0), (t + 0.5, -0.5)], 0.01, seed)
        subj = np.concatenate([tip[None], rest])
        if arcs_host.area(host, subj, clip) <= 0.0:
            continue
        slivers += 1
        got = arcs_host.grad(host, subj, clip)
        if got is None:
            continue
        planned += 1
        # a sliver of depth d has a derivative of the order of d; the whole cell's is ~0.01
        assert max(np.abs(got[0]).max(), np.abs(got[1]).max()) <= 1e-11, it
    assert slivers > 1000
