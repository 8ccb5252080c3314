"""Memory of the linearised operator's partial products, on the stand-in runtime (no GPU needed): as much as
the vectors of a call need, and more passes over the operator where that much is not there."""
import pytest

from tests import fake_device

LINEAR = """
g = dgv.DGV(5, 3, (-2.5, 2.5))
n, D = g.nnodes, 27
i, j = np.triu_indices(n, 1)
i, j = i[::29], j[::29]
cap = np.zeros(n, np.int32)
cap[(g.ccell - 1) * D:g.ccell * D] = len(i)
g.set_aarray(cap, np.ones(len(i) * D), np.tile(i + 1, D).astype(np.int32), np.tile(j + 1, D).astype(np.int32))
g.PrepareFMA_DGV(np.ones(n))
def passes(nvec):
    L.fake_reset()
    g.eval_linear_dev(8, 8, nvec=nvec)
    return launched().count("k_fma_rows") + launched().count("k_fma_gemv"), L.fake_largest_malloc()
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return fake_device.library(str(tmp_path_factory.mktemp("fake")))


def test_one_vector_takes_little(lib):
    """8 vectors' sums of 256-row chunks at most, as one pass over 8 vectors took before."""
    fake_device.run(lib, LINEAR + """
few = 8 * ((n + 255) // 256) * n * 8
p, m = passes(1)
assert p == 1 and 0 < m <= few, (p, m, few)
p, m = passes(8)
assert p == 1 and m == 0
p, m = passes(200)
assert p == 1 and m <= 200 * ((n + 255) // 256) * n * 8
assert passes(60) == (1, 0)
assert passes(300)[0] == 2
""")


def test_more_passes_without_memory_or_under_capture(lib):
    fake_device.run(lib, LINEAR + """
L.fake_fail_malloc_above(8 * ((n + 255) // 256) * n * 8)
assert passes(200)[0] == 25            # the first call of all
assert passes(1)[0] == 1
L.fake_fail_malloc_above(1 << 40)
L.fake_capturing(1)
assert passes(200) == (25, 0)
L.fake_capturing(0)
assert passes(200)[0] == 1
""")


@pytest.mark.parametrize("how", ['fail_kernel("k_fma_lists")', "L.fake_fail_malloc_above(300_000)"], ids=["launch", "memory"])
def test_a_plan_that_fails_keeps_nothing(lib, how):
    """However often PrepareFMA fails on the way to its plan, the next success finds the memory there."""
    fake_device.run(lib, LINEAR.replace("g.PrepareFMA_DGV(np.ones(n))", "") + f"""
def prepare():
    try:
        g.PrepareFMA_DGV(np.ones(n))
    except dgv.DGVError:
        return False
    return True
before = L.fake_live_bytes()
{how}
assert not prepare() and not prepare()
assert L.fake_live_bytes() - before < 10 * 8 * n, L.fake_live_bytes() - before   # the regime's vectors at most
fail_kernel("")
L.fake_fail_malloc_above(1 << 40)
assert prepare()
""")
