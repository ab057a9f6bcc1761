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
