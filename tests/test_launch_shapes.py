"""Launches on grids of many cells keep to the work-item limit of a grid dimension (fewer
than 2^32).  On the stand-in runtime, which refuses a launch above it (no GPU needed)."""
import pytest

from tests import fake_device


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return fake_device.library(str(tmp_path_factory.mktemp("fake")))


def test_generator_above_2_26_cell_pairs(lib):
    """23^3 cells of one node: 74 M cell pairs."""
    fake_device.run(lib, """
g = dgv.DGV(23, 1, (-11.5, 11.5))
g.generate_aarray(Trad=4.0)
assert "k_count" in launched() and "k_list" in launched() and "k_kept" in launched()
assert L.fake_widest_launch() < 2 ** 32
""")


@pytest.mark.slow
def test_merged_rows_above_2_24_blocks(lib):
    """18^3 cells of eight nodes, the canonical cell at the corner, a record per cell pair: 17 M blocks."""
    fake_device.run(lib, """
M = 18
g = dgv.DGV(M, 2, (-0.5, M - 0.5))
D, n = 8, g.nnodes
x, y = np.triu_indices(M ** 3)
xi, xi1 = (x * D + 1).astype(np.int32), (y * D + 2).astype(np.int32)
del x, y
cap = np.zeros(n, np.int32)
cap[(g.ccell - 1) * D] = len(xi)
g.set_aarray(cap, np.ones(len(xi)), xi, xi1)
assert "k_pair_index" in launched() and "k_quad_assign" in launched() and "k_quad_write" in launched()
assert L.fake_widest_launch() < 2 ** 32
""")


@pytest.mark.slow
def test_evaluations_of_many_items(lib):
    """16^3 cells of eight nodes, a record per cell pair: about 14 M work items, evaluated in several launches."""
    fake_device.run(lib, """
M = 16
g = dgv.DGV(M, 2, (-0.5 * M, 0.5 * M))
D, n = 8, g.nnodes
x, y = np.triu_indices(M ** 3)
xi, xi1 = (x * D + 1).astype(np.int32), (y * D + 2).astype(np.int32)
del x, y
cap = np.zeros(n, np.int32)
cap[(g.ccell - 1) * D] = len(xi)
g.set_aarray(cap, np.ones(len(xi)), xi, xi1)
p = C.c_void_p(8)
for call, a in ((L.dgv_eval_q_dev, (p, p)), (L.dgv_eval_mixed_dev, (p, p, p))):
    L.fake_reset()
    assert call(g.ctx, *a, C.c_int64(n)) == 0, L.dgv_last_error(g.ctx)
    assert launched().count("k_quad_eval") > 1
    assert 2 ** 22 <= L.fake_widest_launch() < 2 ** 32
""")
