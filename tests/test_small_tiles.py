"""The smallest work items that a caller can ask for: the merged plan takes no more partial sums for them than
the pair-block plan does, on the stand-in runtime (no GPU needed)."""
import pytest

from tests import fake_device


@pytest.mark.parametrize("grid,part", [("(6, 5, 5), 3, (-2.0, 2.0)", 5), ("(7, 6, 6), 2, (-2.0, 2.0)", 1)])
@pytest.mark.parametrize("tile", [1, 100])
def test_partial_sums(tmp_path_factory, grid, part, tile):
    lib = fake_device.library(str(tmp_path_factory.mktemp("fake")))
    fake_device.run(lib, f"""
g = dgv.DGV({grid})
n, D = g.nnodes, g.D
i, j = np.triu_indices(n, 1)
i, j = i[::{part}], j[::{part}]
cap = np.zeros(n, np.int32)
cap[(g.ccell - 1) * D:g.ccell * D] = len(i)
g.set_aarray(cap, np.ones(len(i) * D), np.tile(i + 1, D).astype(np.int32), np.tile(j + 1, D).astype(np.int32))
assert g.merged_rows()["used"]
L.fake_reset()
g.set_tile({tile})
merged = L.fake_largest_malloc()
g.set_kernel(dgv.DGV_KERNEL_PAIRBLOCK)
L.fake_reset()
g.set_tile({tile})
assert merged <= L.fake_largest_malloc(), (merged, L.fake_largest_malloc())
""")
