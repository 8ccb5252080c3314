"""Generated arrays on grids with many spheres that only touch the cell, lie within it
or reach a face or a corner exactly (integrated point by point), every record against the
host's value of its pair, and the pairs without a record against a host value of nothing.

Tolerance: host and device round differently (fused products, math functions), and far
spheres amplify it by (distance / half width)^2 <= ~100: 1e-12 of values up to 8 pi,
relative to the largest A; a pair without a record is one whose raw values are rounding."""
import numpy as np
import pytest

from dgv0d3v_direct_collision_amd.collision import agen_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,s,half,nquad", [(2, 3, 1.0, 16), (4, 2, 2.0, 24), ((2, 3, 4), 2, 1.5, 20), (5, 1, 2.5, 24), (1, 3, 1.0, 24)],
                         ids=lambda x: str(x).replace(" ", ""))
def test_against_host(M, s, half, nquad):
    import dgv0d3v_direct_collision_amd as dgv
    g = dgv.DGV(M, s, (-half, half))
    print(f"\n[agen marked] {M} s={s}", flush=True)
    try:
        g.generate_aarray(nquad=nquad)
        D, N = s ** 3, g.nnodes
        counts, A, x, y = g.get_aarray_bases(range(D), index_base=1)
        l = np.repeat(np.arange(D), counts)
        have = {}
        for k in range(len(A)):
            have.setdefault((int(x[k]), int(y[k])), np.zeros(D))[l[k]] = A[k]
        big = np.abs(A).max()
        rng = np.random.default_rng(5)
        pairs = [(i, j) for i in range(1, N + 1) for j in range(i + 1, N + 1)]
        if len(pairs) > 6000:
            pairs = [pairs[k] for k in rng.permutation(len(pairs))[:6000]]
        for i, j in pairs:
            raw, a, _ = agen_pair(M, s, (-half, half), i, j, nquad=nquad)
            got = have.get((i, j))
            if got is None:
                assert np.abs(raw).max() <= 1e-10, (i, j)
            else:
                assert np.abs(got - a).max() <= 1e-12 * big, (i, j, np.abs(got - a).max() / big)
    finally:
        g.close()
