"""Memory of a merged FP64 batch's partial sums, on the stand-in runtime (no GPU needed): the default run
length keeps them within a quarter of the coefficients' bytes or 1 GB, falls back to the fewest where that
much is not there, and a batch whose plan could not be built refuses to evaluate."""
import pytest

from tests import fake_device

BATCH = """
g = dgv.DGV(5, 2, (-2.5, 2.5))
n, D = g.nnodes, 8
i, j = np.triu_indices(n, 1)
cap = np.zeros(n, np.int32)
cap[(g.ccell - 1) * D:g.ccell * D] = len(i)
g.set_aarray(cap, np.ones(len(i) * D), np.tile(i + 1, D).astype(np.int32), np.tile(j + 1, D).astype(np.int32))
n = 16384
def make(): return dgv.DGVBatch([g], np.zeros(n, np.int32), dgv.DGV_FP64)
def code(call, *a):
    try:
        call(*a)
    except dgv.DGVError as e:
        return e.code
    return 0
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return fake_device.library(str(tmp_path_factory.mktemp("fake")))


def test_default_runs_fit_a_gigabyte(lib):
    fake_device.run(lib, BATCH + """
L.fake_reset()
b = make()
assert "k_quad_batch" not in launched()
assert L.fake_largest_malloc() <= 1e9, L.fake_largest_malloc()
b.eval_q()
assert "k_quad_batch" in launched() and "k_quad_batch_reduce" in launched()
L.fake_reset()
b.set_tile(512)                        # as asked
assert L.fake_largest_malloc() > 1e9
""")


def test_fewest_rows_where_memory_is_short(lib):
    fake_device.run(lib, BATCH + """
L.fake_fail_malloc_above(300_000_000)   # f and q of the batch take 131 MB each
b = make()
L.fake_reset()
b.eval_q()
assert "k_quad_batch" in launched()
""")


def test_no_plan_no_evaluation(lib):
    fake_device.run(lib, BATCH + """
b = make()
L.fake_fail_malloc_above(100_000_000)
assert code(b.set_tile, 0) == -4
L.fake_fail_malloc_above(1 << 40)
L.fake_reset()
assert code(b.eval_q) == -6 and not launched()
b.set_tile(0)
b.eval_q()
assert "k_quad_batch" in launched()
""")
