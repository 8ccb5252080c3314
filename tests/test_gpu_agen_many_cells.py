"""Generated arrays of grids with more cell pairs than one launch has waves for: every record near the
canonical cell against the host's value of its pair, and no record elsewhere.

Tolerance: as for the other generated arrays, 1e-12 of the largest A."""
import numpy as np
import pytest

from dgv0d3v_direct_collision_amd.collision import agen_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,s,half,Trad,reach", [(9, 1, 4.5, 3.0, 5.0), (23, 1, 11.5, 2.5, 4.3), ((9, 8, 9), 2, 4.5, 1.3, 2.3)], ids=str)
def test_records_near_the_canonical_cell(M, s, half, Trad, reach):
    """reach: every pair at most Trad apart whose sphere meets the cell has both nodes within it of the cell's centre."""
    import dgv0d3v_direct_collision_amd as dgv
    g = dgv.DGV(M, s, (-half, half))
    print(f"\n[agen many cells] {M} s={s}", flush=True)
    try:
        g.generate_aarray(Trad=Trad, nquad=12)
        D = s ** 3
        counts, A, x, y = g.get_aarray_bases(range(D), index_base=1)
        l = np.repeat(np.arange(D), counts)
        have = {}
        for k in range(len(A)):
            have.setdefault((int(x[k]), int(y[k])), np.zeros(D))[l[k]] = A[k]
        X = np.stack([g.nodes_u, g.nodes_v, g.nodes_w], 1)
        cell = X[(g.ccell - 1) * D:g.ccell * D].mean(0)
        near = np.flatnonzero(np.linalg.norm(X - cell, axis=1) <= reach) + 1
        a, b = np.triu_indices(len(near), 1)
        i, j = near[a], near[b]
        close = np.linalg.norm(X[i - 1] - X[j - 1], axis=1) <= Trad * (1 + 1e-12)
        pairs = list(zip(i[close], j[close]))
        big, seen = np.abs(A).max(), 0
        for i, j in pairs:
            raw, a, _ = agen_pair(M, s, (-half, half), int(i), int(j), Trad=Trad, nquad=12)
            got = have.get((int(i), int(j)))
            if got is None:
                assert np.abs(raw).max() <= 1e-10, (i, j)
            else:
                seen += 1
                assert np.abs(got - a).max() <= 1e-12 * big, (i, j, np.abs(got - a).max() / big)
        assert seen == len(have) > 0
    finally:
        g.close()
