"""An infinite entry in the operator's last row gives infinity where one vector and where several are
passed: the rows that fill up the last tile are no rows of it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_infinite_last_row():
    import dgv0d3v_direct_collision_amd as dgv
    d = dgv.DGV((1, 1, 1), 3, (-1.0, 1.0))
    try:
        print("\n[linear infinite] 27 nodes", flush=True)
        n = d.nnodes
        cap = np.zeros(n, np.int32)
        cap[0] = 1
        d.set_aarray(cap, np.ones(1), np.array([1], np.int32), np.array([n], np.int32))   # one record: nodes 1 and 27
        fm = np.ones(n)
        fm[0] = np.inf
        d.PrepareFMA_DGV(fm)
        fma = d.fmA
        assert fma[n - 1, 0] == np.inf and np.isfinite(fma[0, 0])
        F = np.ones((40, n))
        d_f, d_q = d.device_alloc(F.nbytes), d.device_alloc(F.nbytes)
        d.htod(d_f, F)
        for nv in (1, 2, 20, 40):
            Q = np.zeros((40, n))
            d.eval_linear_dev(d_f, d_q, nvec=nv)
            d.synchronize()
            d.dtoh(Q, d_q)
            assert np.all(Q[:nv, 0] == np.inf), nv
            assert np.array_equal(np.isnan(Q[:nv, 1:]), np.tile(np.isnan(fma[n - 1, 1:]), (nv, 1))), nv
        d.device_free(d_f)
        d.device_free(d_q)
    finally:
        d.close()
