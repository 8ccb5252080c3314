"""EvalCollisionLinear of several vectors at the edges of its tiles (16 to 128
vectors, 128 columns, chunks of rows), with leading dimensions above N: against
2 f . fmA in numpy, and a vector's result whatever is passed with it.
Tolerance: relative L2 <= 1e-12 (FP64 in another order)."""
import numpy as np
import pytest

from tests.helpers import maxwellian, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", [((1, 3, 2), 3, (-1.0, 1.0)), ((4, 3, 3), 3, (-2.0, 2.0)), ((5, 6, 4), 2, (-2.0, 2.0)),
                                  ((1, 1, 1), 2, (-1.0, 1.0))], ids=lambda c: f"M{c[0]}s{c[1]}".replace(" ", ""))
def test_vectors_at_tile_edges(case):
    import dgv0d3v_direct_collision_amd as dgv
    M, s, box = case
    d = dgv.DGV(M, s, box)
    try:
        print(f"\n[linear] {case}", flush=True)
        d.generate_aarray(nquad=12)
        n = d.nnodes
        d.PrepareFMA_DGV(maxwellian(d.nodes_u, d.nodes_v, d.nodes_w, 1.0, (0.1, 0.0, -0.1), 0.5))
        fma = d.fmA
        nmax, ld, ldq = 260, n + 5, n + 3
        F = np.random.default_rng(n).standard_normal((nmax, ld))
        want = 2.0 * F[:, :n] @ fma
        d_f, d_q = d.device_alloc(F.nbytes), d.device_alloc(8 * nmax * ldq)
        d.htod(d_f, F)
        first = {}
        for nv in (1, 2, 15, 16, 17, 32, 33, 64, 65, 128, 129, 256, 257, 260):
            Q = np.full((nmax, ldq), 7.0)
            d.htod(d_q, Q)
            d.eval_linear_dev(d_f, d_q, nvec=nv, ldf=ld, ldq=ldq)
            d.synchronize()
            d.dtoh(Q, d_q)
            assert rel_l2(Q[:nv, :n], want[:nv]) <= 1e-12, nv
            assert np.all(Q[nv:] == 7.0) and np.all(Q[:, n:] == 7.0), nv
            for k in range(nv):
                assert np.array_equal(Q[k, :n], first.setdefault(k, Q[k, :n].copy())), (nv, k)
        d.device_free(d_f)
        d.device_free(d_q)
    finally:
        d.close()
