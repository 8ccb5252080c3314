"""Batched items with fewer 64-instance chunks than their workgroup has waves
for: the blocks of an item are then cut into shares.  Any instance count must
give each instance the Q that a full item gives it.

Tolerances, from the arithmetic: the shares only regroup the FP64 sum of at most
~1000 block or round sums, whose absolute values add up to at most ~100 times Q,
so INT8_SPLIT and F64ACC differ by less than 1000 x 2^-53 x 100 ~ 1.1e-11; the
(hi, lo) FP32 pairs of COMP add ~1e4 round-offs of 2^-48, x 100: 4e-9."""
import numpy as np
import pytest

import oracle
from tests.helpers import bimodal, maxwellian, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("DGV_INT8_SPLIT", 1.1e-11), ("DGV_FP32_F64ACC", 1.1e-11), ("DGV_FP32_COMP", 4e-9)])
@pytest.mark.parametrize("grid", [(3, 3, (-1.5, 1.5)), ((5, 4, 3), 2, (-2.0, 2.0)), ((1, 2, 1), 3, (-1.0, 1.0))],
                         ids=lambda g: f"M{g[0]}s{g[1]}".replace(" ", ""))
def test_shares_match_full_items(grid, precision, tol):
    import dgv0d3v_direct_collision_amd as dgv
    M, s, box = grid
    G = oracle.Geometry(M, s, box)
    d = dgv.DGV(M, s, box)
    d.generate_aarray(nquad=12)
    full = 256   # four chunks: no item of any precision is divided
    f = np.stack([(1.0 + 0.01 * i) * bimodal(G.nodes_u, G.nodes_v, G.nodes_w, seed=i) if i % 3 < 2 else
                  maxwellian(G.nodes_u, G.nodes_v, G.nodes_w, 1.0 + 0.1 * (i % 7), (0.1, -0.2, 0.05), 0.6) for i in range(full)])

    def q_of(n, tile):
        b = dgv.DGVBatch([d], [0] * n, getattr(dgv, precision))
        try:
            if tile:
                b.set_tile(tile)
            for i in range(n):
                b.set_f(i, f[i])
            b.eval_q()
            return np.stack([b.get_q(i) for i in range(n)])
        finally:
            b.close()

    try:
        ref = q_of(full, 0)
        for n in (1, 63, 64, 65, 128, 129, 192):
            for tile in (0, 1, 300):
                print(f"[shares] {grid} {precision} n={n} tile={tile}", flush=True)
                q = q_of(n, tile)
                # the Maxwellians (i % 3 == 2) have Q ~ 0: nothing to measure against
                err = max(rel_l2(q[i], ref[i]) if np.any(ref[i]) else np.abs(q[i]).max() for i in range(n) if i % 3 < 2)
                assert err <= tol, (n, tile, err)
    finally:
        d.close()
