"""The merged (box) layout of the A-array: Q and the mixed term against the
oracle's record loop and against the pair-block kernel, on arrays whose box
diagonals all merge, merge in part, or are stored in either node order.

Tolerance: relative L2 <= 1e-12 (FP64 in another order, as for the other
kernels; a merged coefficient differs from its records' by at most 2^-48)."""
import numpy as np
import pytest

import oracle
from tests.helpers import bimodal, maxwellian, rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-12

GRIDS = [(3, 3, (-1.5, 1.5)), ((4, 3, 2), 3, (-2.0, 2.0)), ((6, 5, 4), 2, (-2.5, 2.5)), ((1, 3, 2), 2, (-1.0, 1.0))]


def _vdfs(G):
    f = bimodal(G.nodes_u, G.nodes_v, G.nodes_w, seed=7)
    return f, maxwellian(G.nodes_u, G.nodes_v, G.nodes_w, 1.0, (0.1, -0.2, 0.05), 0.7)


def _check(d, G, A, tag):
    import dgv0d3v_direct_collision_amd as dgv
    f, fm = _vdfs(G)
    ref = oracle.eval_aplus(G, *A, f, nthreads=16)
    refm = oracle.eval_mixed(G, *A, f, fm)
    for tile in (0, 1, 97, 1 << 20):
        d.set_tile(tile)
        q, m = d.EvalCollisionPeriodicAPlus_DGV(f), d.EvalCollisionPeriodicMixedTermsA_DGV(f, fm)
        assert rel_l2(q, ref) <= TOL, (tag, tile, rel_l2(q, ref))
        assert rel_l2(m, refm) <= TOL, (tag, tile, rel_l2(m, refm))
        assert np.array_equal(q, d.EvalCollisionPeriodicAPlus_DGV(f)), (tag, tile)
    d.set_kernel(dgv.DGV_KERNEL_PAIRBLOCK)
    assert rel_l2(d.EvalCollisionPeriodicAPlus_DGV(f), ref) <= TOL, tag
    d.set_kernel(dgv.DGV_KERNEL_AUTO)
    assert rel_l2(d.EvalCollisionPeriodicAPlus_DGV(f), ref) <= TOL, tag


@pytest.mark.parametrize("case", GRIDS, ids=lambda c: f"M{c[0]}s{c[1]}".replace(" ", ""))
def test_generated_and_changed_arrays(case):
    import dgv0d3v_direct_collision_amd as dgv
    M, s, box = case
    G = oracle.Geometry(M, s, box)
    d = dgv.DGV(M, s, box)
    try:
        print(f"\n[merged] {case} generated", flush=True)
        d.generate_aarray(nquad=16)
        A = d.get_aarray()
        _check(d, G, A, "generated")
        print("[merged] threshold", flush=True)
        d.TruncAarrsTrhls_DGV(float(np.median(np.abs(A[1]))))
        _check(d, G, d.get_aarray(), "threshold")
        print("[merged] absolute values", flush=True)
        d.aarray_abs()
        _check(d, G, d.get_aarray(), "abs")
        print("[merged] radius", flush=True)
        d.set_aarray(*A)
        d.TruncAarrsRadius_DGV(1.2)
        _check(d, G, d.get_aarray(), "radius")
    finally:
        d.close()


def test_either_node_order_partial_merges_and_self_pairs():
    """Half of the records with xi and xi1 exchanged, a tenth changed by a part in
    1e6 (their boxes merge in part), and records with xi = xi1."""
    import dgv0d3v_direct_collision_amd as dgv
    M, s, box = (4, 3, 3), 3, (-2.0, 2.0)
    G = oracle.Geometry(M, s, box)
    d = dgv.DGV(M, s, box)
    try:
        print("\n[merged] exchanged nodes", flush=True)
        d.generate_aarray(nquad=16)
        capphi, A, xi, xi1 = d.get_aarray()
        rng = np.random.default_rng(3)
        swap = rng.random(len(A)) < 0.5
        xi, xi1 = np.where(swap, xi1, xi).astype(np.int32), np.where(swap, xi, xi1).astype(np.int32)
        A = A * np.where(rng.random(len(A)) < 0.1, 1.0 + 1e-6, 1.0)
        at = rng.random(len(A)) < 0.01
        xi1 = np.where(at, xi, xi1).astype(np.int32)
        d.set_aarray(capphi, A, xi, xi1)
        _check(d, G, (capphi, A, xi, xi1), "exchanged")
    finally:
        d.close()


def test_other_node_counts_of_eight():
    """Eight nodes per cell as 4 x 2 x 1: a box that is flat in w has two diagonals."""
    import dgv0d3v_direct_collision_amd as dgv
    M, s, box = (3, 2, 4), (4, 2, 1), (-1.5, 1.5)
    G = oracle.Geometry(M, s, box)
    X = np.stack([G.nodes_u, G.nodes_v, G.nodes_w], 1)
    i, j = np.triu_indices(G.nnodes, 1)
    # a coefficient that depends on the box alone: equal on its diagonals
    mid, dist = X[i] + X[j], ((X[i] - X[j]) ** 2).sum(1)
    D = 8
    capphi = np.zeros(G.nnodes, np.int32)
    capphi[(G.ccell - 1) * D:G.ccell * D] = len(i)
    A = np.concatenate([1e-3 * np.cos(1.0 + l + np.round(mid, 9) @ [0.3, 0.5, 0.7] + np.round(dist, 9)) for l in range(D)])
    xi, xi1 = np.tile(i + 1, D).astype(np.int32), np.tile(j + 1, D).astype(np.int32)
    d = dgv.DGV(M, s, box)
    try:
        print("\n[merged] 4 x 2 x 1 nodes per cell", flush=True)
        d.set_aarray(capphi, A, xi, xi1)
        _check(d, G, (capphi, A, xi, xi1), "4x2x1")
    finally:
        d.close()


def test_infinite_and_nan_values_stay_where_they_were():
    """Nodes whose Q is not finite are the pair-block kernel's."""
    import dgv0d3v_direct_collision_amd as dgv
    d = dgv.DGV((4, 3, 2), 3, (-2.0, 2.0))
    try:
        print("\n[merged] infinite f", flush=True)
        d.generate_aarray(nquad=16)
        rng = np.random.default_rng(1)
        for bad in (np.inf, np.nan):
            f = rng.random(d.nnodes)
            f[d.nnodes - 5] = bad
            q = d.EvalCollisionPeriodicAPlus_DGV(f)
            d.set_kernel(dgv.DGV_KERNEL_PAIRBLOCK)
            p = d.EvalCollisionPeriodicAPlus_DGV(f)
            d.set_kernel(dgv.DGV_KERNEL_AUTO)
            assert np.array_equal(np.isfinite(q), np.isfinite(p))
    finally:
        d.close()


@pytest.mark.parametrize("counts", [(1, 0), (16, 1), (17, 33), (64, 15)], ids=str)
def test_batch_on_merged_layouts(counts):
    """FP64 batches of two grids (32-instance chunks, a chunk of at most 16 columns,
    a grid without instances), every tile, against the single-VDF evaluator; and
    the same with one grid whose array does not merge."""
    import dgv0d3v_direct_collision_amd as dgv
    from tests.helpers import synthetic_aarray
    G = oracle.Geometry((2, 3, 2), 3, (-1.2, 1.2))
    a, c = dgv.DGV((4, 3, 3), 3, (-2.0, 2.0)), dgv.DGV((2, 3, 2), 3, (-1.2, 1.2))
    try:
        a.generate_aarray(nquad=16)
        for merged in (True, False):
            print(f"\n[merged] batch {counts} both grids merge: {merged}", flush=True)
            if merged:
                c.generate_aarray(nquad=16)
            else:
                c.set_aarray(*synthetic_aarray(G, seed=4))
            which = np.repeat([0, 1], counts).astype(np.int32)
            rng = np.random.default_rng(sum(counts))
            fs = [rng.random([a, c][k].nnodes) for k in which]
            ref = [[a, c][k].EvalCollisionPeriodicAPlus_DGV(f) for k, f in zip(which, fs)]
            b = dgv.DGVBatch([a, c], which, dgv.DGV_FP64)
            for i, f in enumerate(fs):
                b.set_f(i, f)
            for tile in (0, 1, 5000, 1 << 24):
                b.set_tile(tile)
                b.eval_q()
                err = max(rel_l2(b.get_q(i), r) for i, r in enumerate(ref))
                assert err <= TOL, (counts, merged, tile, err)
            b.set_probe_cells([0, 5])
            b.eval_q_probe()
            assert rel_l2(b.get_q(0), ref[0]) <= TOL
            b.rk_run(1e-4, 2, rkmts=2)
            f = fs[0].copy()
            a.rkmts = 2
            for _ in range(2):
                (a if which[0] == 0 else c).TimeIntegratorORK_SH_DGV(f, 1e-4)
            assert rel_l2(b.get_f(0), f) <= TOL
            b.close()
    finally:
        a.close()
        c.close()
