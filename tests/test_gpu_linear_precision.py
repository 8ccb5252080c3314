"""EvalCollisionLinear against the products with fmA summed in extended precision, on a grid whose chunks
of rows are long: no further from it than FP64 sums of 256 rows, one chain each, added in order.

Tolerance: those host sums round each product and each addition, the device's chains only the additions, and
the root mean square over 6 x 400 values scatters by a few per cent: a quarter above is room enough, and the
sums of whole chunks (about 1500 rows) in one chain are 1.5 times as far or more."""
import numpy as np
import pytest

from tests.helpers import maxwellian

pytestmark = pytest.mark.gpu


def test_long_chunks_at_27_cubed():
    import dgv0d3v_direct_collision_amd as dgv
    LD = np.longdouble
    d = dgv.DGV(9, 3, (-4.0, 4.0))
    try:
        print("\n[linear precision] 27^3 nodes", flush=True)
        d.generate_aarray(nquad=12)
        n = d.nnodes
        rng = np.random.default_rng(0)
        fm = maxwellian(d.nodes_u, d.nodes_v, d.nodes_w, 1.0, (0.1, -0.1, 0.2), 0.8)
        d.PrepareFMA_DGV(fm)
        cols = rng.choice(n, 400, replace=False)
        C = np.ascontiguousarray(d.fmA[:, cols])
        F = np.stack([maxwellian(d.nodes_u, d.nodes_v, d.nodes_w, 1.0, rng.uniform(-0.6, 0.6, 3), rng.uniform(0.4, 1.2)) *
                      (1 + 0.1 * rng.standard_normal(n)) for _ in range(6)])
        exact = np.stack([2 * (f.astype(LD)[:, None] * C).sum(0) for f in F])
        host = np.zeros((6, 400))
        for k, f in enumerate(F):
            for r in range(0, n, 256):
                host[k] += np.add.accumulate(f[r:r + 256, None] * C[r:r + 256], axis=0)[-1]

        def error(q):
            return float(np.sqrt(np.mean([np.sum((q[k] - exact[k]) ** 2) / np.sum(exact[k] ** 2) for k in range(6)])))

        bound = 1.25 * error(2 * host)
        d_f, d_q = d.device_alloc(F.nbytes), d.device_alloc(F.nbytes)
        Q = np.empty_like(F)
        d.htod(d_f, F)
        d.eval_linear_dev(d_f, d_q, nvec=6)
        d.synchronize()
        d.dtoh(Q, d_q)
        print(f"[linear precision] error {error(Q[:, cols]):.2e}, bound {bound:.2e}", flush=True)
        assert error(Q[:, cols]) <= bound
        one = np.empty(n)
        for k in range(6):                      # one at a time: the same to the last bit
            d.htod(d_f, F[k])
            d.eval_linear_dev(d_f, d_q, nvec=1)
            d.synchronize()
            d.dtoh(one, d_q)
            assert np.array_equal(one, Q[k])
        d.device_free(d_f)
        d.device_free(d_q)
    finally:
        d.close()
