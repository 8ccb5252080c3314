"""dgv_ctx_autotune on the merged layout times the plan of a context that was never tuned beside the fixed
sizes and goes back to it where it is the fastest.  On the stand-in runtime, which says which candidate was
(no GPU needed)."""
import pytest

from tests import fake_device

GRID = """
g = dgv.DGV((5, 4, 4), 3, (-2.0, 2.0))
n, D = g.nnodes, 27
i, j = np.triu_indices(n, 1)
i, j = i[::6], j[::6]
cap = np.zeros(n, np.int32)
cap[(g.ccell - 1) * D:g.ccell * D] = len(i)
rec = (cap, np.ones(len(i) * D), np.tile(i + 1, D).astype(np.int32), np.tile(j + 1, D).astype(np.int32))
def items():
    L.fake_reset()
    g.eval_q_dev(8, 8)
    assert "k_quad_eval" in launched()
    return L.fake_widest_launch()
g.set_aarray(*rec)
own = items()
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return fake_device.library(str(tmp_path_factory.mktemp("fake")))


@pytest.mark.parametrize("set_before", [False, True])
def test_own_plan_wins(lib, set_before):
    fake_device.run(lib, GRID + f"""
if {set_before}:
    g.set_tile(512)
    assert items() != own
won = []
for k in range(8):
    L.fake_fastest(k)
    best, ms = g.autotune()
    assert best > 0
    if items() == own:
        won.append(k)
        g.set_aarray(*rec)               # kept for the next array
        assert items() == own
        g.set_tile(best)                 # the pairs named are the plan's
        assert items() == own
assert won, "no candidate is the context's own plan"
""")


def test_a_fixed_size_wins(lib):
    fake_device.run(lib, GRID + """
sizes = set()
for k in range(8):
    L.fake_fastest(k)
    best, _ = g.autotune()
    sizes.add(best)
    now = items()
    g.set_aarray(*rec)
    assert items() == now
assert {512, 1024, 2048, 4096, 8192, 16384} <= sizes and max(sizes) > 16384
""")
