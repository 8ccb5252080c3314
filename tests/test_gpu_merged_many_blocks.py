"""Merged rows built from more blocks than their kernels have workgroups (2^16): Q and the mixed term
against the pair-block kernel.  Tolerance: relative L2 <= 1e-12, as for the other merged-layout tests."""
import numpy as np
import pytest

from tests.helpers import bimodal, maxwellian, rel_l2

pytestmark = pytest.mark.gpu


def test_ten_by_nine_by_ten_cells_of_eight():
    import dgv0d3v_direct_collision_amd as dgv
    d = dgv.DGV((10, 9, 10), 2, (-3.0, 3.0))
    try:
        print("\n[merged] 10 x 9 x 10 cells of eight nodes", flush=True)
        d.generate_aarray(nquad=12)
        f = bimodal(d.nodes_u, d.nodes_v, d.nodes_w, seed=2)
        fm = maxwellian(d.nodes_u, d.nodes_v, d.nodes_w, 1.0, (0.1, -0.2, 0.05), 0.7)
        q, m = d.EvalCollisionPeriodicAPlus_DGV(f), d.EvalCollisionPeriodicMixedTermsA_DGV(f, fm)
        d.set_kernel(dgv.DGV_KERNEL_PAIRBLOCK)
        assert rel_l2(q, d.EvalCollisionPeriodicAPlus_DGV(f)) <= 1e-12
        assert rel_l2(m, d.EvalCollisionPeriodicMixedTermsA_DGV(f, fm)) <= 1e-12
    finally:
        d.close()
