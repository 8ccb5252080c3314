"""Spheres that reach a face or a corner of the cell, lie within it or miss it: one pair's
values by the host code, against those of the pair mirrored in u and v, whose arcs are
found from the other pair of face lines.

Tolerance: both take the same points in the polar angle, so only rounding differs: far
spheres lose (distance / cell half width)^2 <= ~200 units in the last place of values up to
8 pi in a few terms, 200 x 2.2e-16 x 25 x ~10 = 1e-11; the tangent pair (distance 3 half widths)
100 times less."""
import numpy as np
import pytest

from dgv0d3v_direct_collision_amd.collision import agen_pair, grid_geometry

CASES = [(5, 3, 3.5), (3, 2, 1.5), (4, 3, 2.0), (7, 2, 1.7), (3, 1, 1.0)]


def _nodes(M, s, half):
    u, v, w, _, cc = grid_geometry(M, s, (-half, half))
    return np.stack([u, v, w], 1), (cc - 1) * s ** 3


def _index(x, p):
    return int(np.abs(x - np.asarray(p)).sum(1).argmin()) + 1


@pytest.mark.parametrize("case", CASES, ids=str)
def test_mirrored_in_u_and_v(case):
    M, s, half = case
    x, first = _nodes(M, s, half)
    rng = np.random.default_rng(3)
    D = s ** 3
    pairs = [tuple(p) for p in rng.integers(0, len(x), (150, 2)) if p[0] != p[1]]
    pairs += [(first + i, first + j) for i in range(D) for j in range(i + 1, D)][:40]   # within the canonical cell
    for axis in range(3):   # on lines along an axis: centres on faces, tangent lines
        for i in rng.integers(0, len(x), 25):
            p = x[i].copy()
            p[axis] = x[rng.integers(0, len(x)), axis]
            j = _index(x, p) - 1
            if j != i:
                pairs.append((int(i), j))
    worst = 0.0
    for i, j in pairs:
        a, _, _ = agen_pair(M, s, (-half, half), min(i, j) + 1, max(i, j) + 1)
        k, m = _index(x, x[i][[1, 0, 2]]), _index(x, x[j][[1, 0, 2]])
        b, _, _ = agen_pair(M, s, (-half, half), min(k, m), max(k, m))
        worst = max(worst, np.abs(a.reshape(s, s, s) - b.reshape(s, s, s).transpose(1, 0, 2)).max())
    assert worst <= 1e-11, worst


def test_tangent_to_a_face():
    """Radius equal to the distance of a face line, to rounding: (-1.4, 0, -1.4), (-1.4, 0, 2.8)
    on 15^3 nodes over [-3.5, 3.5]^3, and its mirror image in u and v."""
    x, _ = _nodes(5, 3, 3.5)
    a, _, _ = agen_pair(5, 3, (-3.5, 3.5), _index(x, (-1.4, 0, -1.4)), _index(x, (-1.4, 0, 2.8)))
    b, _, _ = agen_pair(5, 3, (-3.5, 3.5), _index(x, (0, -1.4, -1.4)), _index(x, (0, -1.4, 2.8)))
    assert np.abs(a.reshape(3, 3, 3) - b.reshape(3, 3, 3).transpose(1, 0, 2)).max() <= 1e-13
