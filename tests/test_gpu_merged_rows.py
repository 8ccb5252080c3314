"""Which evaluations read the merged layout, and how many rows it has: generated arrays merge to about one
row per box of nodes, changed pairs stay apart, arrays that do not merge keep none."""
import numpy as np
import pytest

import oracle
from tests.helpers import synthetic_aarray
from tests.test_gpu_merged import GRIDS, _check

pytestmark = pytest.mark.gpu


def boxes_of(d):
    """(distinct boxes of the array's pairs, pairs with a node in the canonical cell, pairs)."""
    counts, _, xi, xi1 = d.get_aarray_bases(range(d.D), index_base=0)
    i, j = np.unique(np.stack([xi, xi1]), axis=1)
    key = []
    for c in (d.nodes_u, d.nodes_v, d.nodes_w):
        level = np.unique(np.round(c, 9), return_inverse=True)[1].ravel()
        key += [np.minimum(level[i], level[j]), np.maximum(level[i], level[j])]
    cc = d.ccell - 1
    return np.unique(np.stack(key), axis=1).shape[1], int(((i // d.D == cc) | (j // d.D == cc)).sum()), len(i)


def _merges(d, tag):
    boxes, canonical, pairs = boxes_of(d)
    m = d.merged_rows()
    print(f"[merged rows] {tag}: {m}, {boxes} boxes, {canonical} pairs of the canonical cell", flush=True)
    if not m["used"]:   # kept only where it leaves at most nine rows for ten pairs
        assert tag == "radius" and boxes + canonical > 0.9 * pairs, tag
        return
    assert m["pairs"] == pairs, tag
    assert boxes <= m["rows"] <= boxes + canonical, tag


@pytest.mark.parametrize("case", GRIDS, ids=lambda c: f"M{c[0]}s{c[1]}".replace(" ", ""))
def test_generated_arrays_merge(case):
    import dgv0d3v_direct_collision_amd as dgv
    M, s, box = case
    d = dgv.DGV(M, s, box)
    try:
        print(f"\n[merged rows] {case}", flush=True)
        d.generate_aarray(nquad=16)
        _merges(d, "generated")
        d.set_kernel(dgv.DGV_KERNEL_PAIRBLOCK)
        assert not d.merged_rows()["used"] and d.merged_rows()["rows"] > 0
        d.set_kernel(dgv.DGV_KERNEL_AUTO)
        A = d.get_aarray()
        d.aarray_abs()
        _merges(d, "abs")
        d.set_aarray(*A)
        _merges(d, "set")
        d.TruncAarrsRadius_DGV(1.2)
        _merges(d, "radius")
    finally:
        d.close()


def test_a_tenth_of_the_pairs_changed():
    """Their boxes keep more than one row, the layout stays in use."""
    import dgv0d3v_direct_collision_amd as dgv
    M, s, box = (4, 3, 3), 3, (-2.0, 2.0)
    G = oracle.Geometry(M, s, box)
    d = dgv.DGV(M, s, box)
    try:
        print("\n[merged rows] a tenth of the pairs changed", flush=True)
        d.generate_aarray(nquad=16)
        whole = d.merged_rows()["rows"]
        capphi, A, xi, xi1 = d.get_aarray()
        pair = np.unique(np.stack([xi, xi1]), axis=1, return_inverse=True)[1].ravel()
        rng = np.random.default_rng(3)
        changed = rng.random(pair.max() + 1) < 0.1
        swap = (rng.random(pair.max() + 1) < 0.5)[pair]
        xi, xi1 = np.where(swap, xi1, xi).astype(np.int32), np.where(swap, xi, xi1).astype(np.int32)
        A = A * np.where(changed[pair], 1.0 + 1e-6, 1.0)
        d.set_aarray(capphi, A, xi, xi1)
        m = d.merged_rows()
        print(f"[merged rows] {whole} -> {m}", flush=True)
        # a changed pair leaves its box's row, at most to a row of its own
        assert m["used"] and whole < m["rows"] <= whole + changed.sum()
        _check(d, G, (capphi, A, xi, xi1), "changed pairs")
    finally:
        d.close()


def test_arrays_that_do_not_merge():
    import dgv0d3v_direct_collision_amd as dgv
    d = dgv.DGV((2, 3, 2), 3, (-1.2, 1.2))
    one = dgv.DGV(3, 1, (-1.5, 1.5))
    try:
        d.set_aarray(*synthetic_aarray(oracle.Geometry((2, 3, 2), 3, (-1.2, 1.2)), seed=4))
        assert d.merged_rows() == dict(rows=0, pairs=0, used=False)
        one.generate_aarray(nquad=16)
        assert one.merged_rows() == dict(rows=0, pairs=0, used=False)
        with pytest.raises(dgv.DGVError):
            dgv.DGV(3, 3, (-1.5, 1.5)).merged_rows()
    finally:
        d.close()
        one.close()


def test_batches():
    import dgv0d3v_direct_collision_amd as dgv
    a, c = dgv.DGV((4, 3, 3), 3, (-2.0, 2.0)), dgv.DGV((2, 3, 2), 3, (-1.2, 1.2))
    try:
        a.generate_aarray(nquad=16)
        c.generate_aarray(nquad=16)
        for grids, precision, want in (([a, c], dgv.DGV_FP64, True), ([a], dgv.DGV_INT8_SPLIT, False), ([a], dgv.DGV_FP32_COMP, False)):
            b = dgv.DGVBatch(grids, [0], precision)
            assert b.merged == want
            b.close()
        c.set_aarray(*synthetic_aarray(oracle.Geometry((2, 3, 2), 3, (-1.2, 1.2)), seed=4))
        b = dgv.DGVBatch([a, c], [0, 1], dgv.DGV_FP64)
        assert not b.merged
        b.close()
    finally:
        a.close()
        c.close()


def test_more_blocks_than_workgroups():
    import dgv0d3v_direct_collision_amd as dgv
    d = dgv.DGV((10, 9, 10), 2, (-3.0, 3.0))
    try:
        d.generate_aarray(nquad=12)
        m = d.merged_rows()
        print(f"\n[merged rows] 10 x 9 x 10 cells of eight: {m}", flush=True)
        assert m["used"] and m["rows"] < 0.5 * m["pairs"]
    finally:
        d.close()
