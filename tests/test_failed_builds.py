"""After a call that fails while it changes an A-array or its work plan, no evaluation reads what that
call dropped: it is refused with DGV_ERR_STATE until a call succeeds again.  On a stand-in for the HIP
runtime, where launches and allocations fail on demand (no GPU needed)."""
import pytest

from tests import fake_device

STATE = -6
GRID = """
g = dgv.DGV((3, 2, 2), 3, (-1.0, 1.0))
n, D = g.nnodes, 27
i, j = np.triu_indices(n, 1)
i, j = i[::7], j[::7]
cap = np.zeros(n, np.int32)
cc = (g.ccell - 1) * D
cap[cc:cc + D] = len(i)
A = np.tile(np.linspace(1.0, 2.0, len(i)), D)
rec = (cap, A, np.tile(i + 1, D).astype(np.int32), np.tile(j + 1, D).astype(np.int32))
def code(call, *a):
    try:
        call(*a)
    except dgv.DGVError as e:
        return e.code
    return 0
f = np.ones(n)
def evaluate():
    L.fake_reset()
    rc = code(g.EvalCollisionPeriodicAPlus_DGV, f)
    return rc, launched()
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return fake_device.library(str(tmp_path_factory.mktemp("fake")))


def test_pair_index_launch_fails(lib):
    """The merged rows are not built from tables that were never written."""
    out = fake_device.run(lib, GRID + """
fail_kernel("k_pair_index")
L.fake_reset()
print(code(g.set_aarray, *rec))
assert "k_pair_index" in launched()
assert "k_quad_assign" not in launched() and "k_quad_write" not in launched(), launched()
fail_kernel("")
rc, l = evaluate()
assert rc == -6 and not l, (rc, l)
assert code(g.set_aarray, *rec) == 0
rc, l = evaluate()
assert rc == 0 and "k_quad_eval" in l and "k_pb_reduce" in l, (rc, l)
""")
    assert int(out.split()[0]) < 0


@pytest.mark.parametrize("change,kernel", [("g.aarray_abs()", k) for k in ("k_abs_coeff", "k_pair_index", "k_quad_assign")] +
                         [("g.TruncAarrsTrhls_DGV(1.5)", k) for k in ("k_truncate", "k_gather_pairs")] +
                         [("g.TruncAarrsRadius_DGV(0.5)", "k_truncate")])
def test_changed_array_whose_merged_rows_fail(lib, change, kernel):
    """The merged rows of the array before the change are not read."""
    fake_device.run(lib, GRID + f"""
assert code(g.set_aarray, *rec) == 0
rc, l = evaluate()
assert rc == 0 and "k_quad_eval" in l
fail_kernel("{kernel}")
assert code(lambda: {change}) < 0
fail_kernel("")
rc, l = evaluate()
assert rc == {STATE} and not l, (rc, l)
assert code(g.set_aarray, *rec) == 0
assert evaluate()[0] == 0
""")


def test_truncation_refused_before_it_starts(lib):
    """No memory for its flags: the array is as it was and stays in use."""
    fake_device.run(lib, GRID + """
assert code(g.set_aarray, *rec) == 0
L.fake_fail_malloc_above(0)
assert code(lambda: g.TruncAarrsTrhls_DGV(1.5)) < 0
rc, l = evaluate()
assert rc == 0 and "k_quad_eval" in l, (rc, l)
""")


@pytest.mark.parametrize("change", ["g.set_tile(300)", "g.set_kernel(dgv.DGV_KERNEL_PAIRBLOCK)"])
def test_plan_without_memory(lib, change):
    fake_device.run(lib, GRID + f"""
assert code(g.set_aarray, *rec) == 0
L.fake_fail_malloc_above(4000)   # the partial sums are more
assert code(lambda: {change}) < 0
L.fake_fail_malloc_above(1 << 40)
rc, l = evaluate()
assert rc == {STATE} and not l, (rc, l)
assert code(lambda: g.set_tile(400)) == 0
assert evaluate()[0] == 0
""")
