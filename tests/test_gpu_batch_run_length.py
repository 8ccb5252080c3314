"""The length of a batch's runs of blocks costs no precision: FP64 Q of runs that hold a cell's whole
array against runs of 16 K pairs, each against the records' sum in extended precision.

Tolerance: rounding errors of the two orders of summation are of one size, and the root mean square of
162 values scatters by 1/sqrt(2 x 162) = 6 %, so a ratio above 1.5 is more than five deviations off."""
import numpy as np
import pytest

from tests.helpers import bimodal, maxwellian

pytestmark = pytest.mark.gpu


def exact_cells(d, M, f, cells):
    """Q of f at the nodes of the cells, summed in extended precision."""
    D = d.D
    counts, A, xi, xi1 = d.get_aarray_bases(range(D), index_base=0)
    ends = np.cumsum(counts)
    cell = lambda c: np.array([c // (M[1] * M[2]), c // M[2] % M[1], c % M[2]])
    can = cell(d.ccell - 1)
    f = f.astype(np.longdouble)
    out = []
    for c in cells:
        shift = cell(c) - can
        ds = ((shift[0] * M[1] + shift[1]) * M[2] + shift[2]) * D
        for l in range(D):
            r = slice(ends[l] - counts[l], ends[l])
            x, y, a = xi[r].astype(np.int64), xi1[r].astype(np.int64), A[r]
            ok = np.ones(len(x), bool)
            for n in (x, y):
                k = cell(n // D)
                for i in range(3):
                    ok &= (k[i] + shift[i] >= 0) & (k[i] + shift[i] < M[i])
            s = np.sum(a[ok].astype(np.longdouble) * f[x[ok] + ds] * f[y[ok] + ds])
            out.append(2 * s / d.nodes_gwts[c * D + l].astype(np.longdouble))
    return np.array(out)


def test_long_runs():
    import dgv0d3v_direct_collision_amd as dgv
    M = (5, 5, 5)
    d = dgv.DGV(M, 3, (-3.5, 3.5))
    try:
        print("\n[batch run length] 15^3 nodes", flush=True)
        d.generate_aarray(nquad=12)
        f = [bimodal(d.nodes_u, d.nodes_v, d.nodes_w, seed=4), maxwellian(d.nodes_u, d.nodes_v, d.nodes_w, 1.0, (0.3, 0.2, -0.1), 0.8) +
             maxwellian(d.nodes_u, d.nodes_v, d.nodes_w, 0.5, (-0.8, 0.1, 0.5), 0.5)]
        cells = (62, 37, 86)
        nodes = np.concatenate([np.arange(c * d.D, (c + 1) * d.D) for c in cells])
        ref = [exact_cells(d, M, x, cells) for x in f]
        b = dgv.DGVBatch([d], [0, 0], dgv.DGV_FP64)
        err = {}
        for tile in (1 << 14, 1 << 24):
            b.set_tile(tile)
            for i in range(2):
                b.set_f(i, f[i])
            b.eval_q()
            e = np.concatenate([(b.get_q(i)[nodes] - ref[i]) / np.linalg.norm(ref[i].astype(float)) for i in range(2)])
            err[tile] = float(np.sqrt(np.sum(e ** 2)))
        b.close()
        print(f"[batch run length] error with runs of 16 K pairs {err[1 << 14]:.2e}, of the whole array {err[1 << 24]:.2e}", flush=True)
        assert err[1 << 24] <= 1.5 * err[1 << 14]
    finally:
        d.close()
