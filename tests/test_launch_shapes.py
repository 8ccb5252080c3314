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
