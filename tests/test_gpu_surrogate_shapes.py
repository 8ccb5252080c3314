"""A training step and a prediction of the surrogate at the edges of its tiles:
one row, one hidden unit, K chunks of a single step, ragged batches, products on
64-wide tiles and (4096 hidden units, 1000 rows) on 128-wide ones, against the CPU
reference with BF16 rounding at the GPU's points; and a readback of padded and
unpadded layers.

Tolerance: relative L2 <= 2e-3 per tensor, as for the other surrogate tests (the GPU
accumulates in FP32 and its BF16 roundings may fall the other way)."""
import numpy as np
import pytest

from oracle import surrogate_ref as sr
from tests.helpers import rel_l2
from tests.test_gpu_surrogate import random_layers, vdf_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,batch,rows", [((1,), 1, 1), ((130,), 129, 129), ((300, 70, 512), 64, 63), ((), 40, 40),
                                               ((4096,), 1000, 900)], ids=lambda x: str(x).replace(" ", ""))
def test_step_and_predict(hidden, batch, rows):
    import dgv0d3v_direct_collision_amd as dgv
    g = dgv.DGV(3, 3, (-3.0, 3.0))
    rng = np.random.default_rng(17)
    widths = [g.nnodes, *hidden, g.nnodes]
    s = dgv.Surrogate(g, widths, batch=batch, seed=3)
    try:
        print(f"\n[surrogate shapes] {widths} batch {batch} rows {rows}", flush=True)
        Ws, bs = random_layers(widths, rng)
        for l in range(len(Ws)):
            s.set_layer(l, Ws[l], bs[l])
        s.set_scales(0.2, 0.05)
        f = vdf_rows(g, rng, rows)
        q = rng.standard_normal((rows, g.nnodes)) * 0.05
        loss = s.train_step_host(f, q, lr=0.0)
        rloss, dWs, dbs, y = sr.forward_backward([W.astype(np.float64) for W in Ws], [b.astype(np.float64) for b in bs],
                                                 f, q, 0.2, 0.05, bf16_path=True)
        assert abs(loss - rloss) <= 1e-4 * rloss
        assert rel_l2(s.predict_host(f, project=False), 0.05 * y) <= 2e-3
        for l in range(len(Ws)):
            gW, gb = s.get_grad(l)
            assert gW.shape == dWs[l].shape
            assert rel_l2(gW, dWs[l]) <= 2e-3 and rel_l2(gb, dbs[l]) <= 2e-3, l
            W, b = s.get_layer(l)                       # lr = 0: unchanged, and dense whatever the padding
            assert np.array_equal(W, Ws[l]) and np.array_equal(b, bs[l])
    finally:
        s.close()
        g.close()
